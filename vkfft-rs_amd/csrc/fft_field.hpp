// fft_field.hpp -- small 2-D and 3-D complex fields in one kernel.
//
// A block holds whole fields in LDS and runs every stage of every axis there,
// last axis first; the first stage reads HBM and the last one writes it, so a
// field passes through memory once instead of once per axis, and one small
// field costs one launch. The Stockham stages ping-pong between two LDS
// buffers (one barrier a stage). The work items of a stage are the butterflies
// of all lines of all fields of the block, numbered (outer, butterfly,
// column): an item's first element is at o * n * inner + b * inner + c of the
// block's elements, so that adjacent lanes touch adjacent elements on every
// axis.
//
// Bound by the latency of the chain of stages (a table load, an LDS round trip and a
// barrier each) at 8 to 16 waves a CU: waves wait 63 to 70% of their cycles and issue
// VALU work in 12 to 14% (f32 64 x 64 x 244, f64 16^3 x 244); 8M f32 points of 64 x 64,
// 128 MB, take 45 us, 2.8 TB/s. Measured, us a pass, axis passes -> one kernel: f32 64 x 64 8.8 ->
// 7.7, x 244 15.4 -> 9.8, x 1953 52.1 -> 45.0; 16 x 16 x 31250 69 -> 44; 63 x 65 15.9 -> 9.0;
// 16^3 x 244 26.4 -> 10.2; 2 x 2000 x 250 35 -> 12; f64 30 x 14 x 2380 27.4 -> 15.7,
// 4 x 1000 x 250 92.7 -> 14.1. Nontemporal accesses measured the same.
//
// Twiddles by table_powers: error against 64 bits, f32, products of one root -> these
// loads, with the axis passes: 1000 x 2 x 2 2.19e-7 -> 1.29e-7 (1.57e-7), 80 x 60 1.65e-7
// -> 1.28e-7 (1.50e-7), 3087 x 2 2.02e-7 -> 1.38e-7 (1.86e-7), at the same times (all
// R - 1 roots from the table: 12 x 720 x 347 27.9 us against 26.6).
#pragma once
#include "fft_device.hpp"
#include "kernels.hpp"

namespace vkfx {

constexpr int kFieldPad = 3;  // one pad slot every 8 elements: stores R = 8 and 16 slots apart spread over the banks

enum FieldMode : int {
    FM_LDS = 0,    // LDS -> LDS
    FM_FIRST = 1,  // HBM -> LDS
    FM_LAST = 2,   // LDS -> HBM, scaled
};

// Quotient of x < 2^16 by a uniform d: one multiplication.
struct FieldDiv {
    unsigned m, d;
    __device__ __forceinline__ explicit FieldDiv(unsigned v) : m(v > 1 ? 0xffffffffu / v + 1 : 0), d(v) {}
    __device__ __forceinline__ int operator()(int x) const { return d > 1 ? (int)__umulhi((unsigned)x, m) : x; }
};

// A pointer that is the same in every lane, in scalar registers (the out-of-line
// stages get it in vector registers). f64 radices up to 10 take 120 registers forward
// this way, 152 without: fields of half a CU's LDS ran alone, 18 x 125 x 466 21.4 us
// against 15.1.
template <typename P>
__device__ __forceinline__ P* uniform(P* p) {
    const unsigned long long v = (unsigned long long)p;
    const unsigned lo = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)v);
    const unsigned hi = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)(v >> 32));
    return (P*)((unsigned long long)lo | (unsigned long long)hi << 32);
}

// One radix-R stage of the axis of n points and stride `inner`, `elems`
// elements in all, P the product of the axis's earlier radices.
template <typename T, int S, int R, int MODE>
__device__ __noinline__ void field_stage(const cpx<T>* src, cpx<T>* dst, int elems, int n, int inner, int P, const void* tw,
                                         const cpx<T>* gin, cpx<T>* gout, const T sc) {
#if defined(__HIP_DEVICE_COMPILE__)
    if constexpr (MODE != FM_FIRST) __builtin_assume(__builtin_amdgcn_is_shared((const void*)src));
    if constexpr (MODE != FM_LAST) __builtin_assume(__builtin_amdgcn_is_shared((const void*)dst));
#endif
    typedef T v2 __attribute__((ext_vector_type(2)));
    typedef const __attribute__((address_space(1))) v2* gin_t;
    typedef __attribute__((address_space(1))) v2* gout_t;
    elems = __builtin_amdgcn_readfirstlane(elems);
    n = __builtin_amdgcn_readfirstlane(n);
    inner = __builtin_amdgcn_readfirstlane(inner);
    P = __builtin_amdgcn_readfirstlane(P);
    tw = uniform(tw);
    gin = uniform(gin);
    gout = uniform(gout);
    const int NB = n / R, NBI = NB * inner, items = elems / R, step = NB / P, PI = P * inner;
    const FieldDiv by_line(NBI), by_col(inner), by_p(P);
    for (int w = threadIdx.x; w < items; w += blockDim.x) {
        const int o = by_line(w), r = w - o * NBI, b = by_col(r), c = r - b * inner;
        const int at = o * NBI * R + r;
        cpx<T> v[R];
#pragma unroll
        for (int i = 0; i < R; ++i) {
            if constexpr (MODE == FM_FIRST) {
                const v2 x = ((gin_t)gin)[at + i * NBI];
                v[i] = mk(x.x, x.y);
            } else {
                v[i] = src[lpad(at + i * NBI, kFieldPad)];
            }
        }
        const int k = b - by_p(b) * P;
        if (P > 1) {
            cpx<T> wp[R];
            table_powers<R>(tw, k * step, wp);
#pragma unroll
            for (int i = 1; i < R; ++i) v[i] = twmul<S>(v[i], wp[i]);
        }
        dft<R, S>(v);
        const int to = o * NBI * R + ((b - k) * R + k) * inner + c;
#pragma unroll
        for (int q = 0; q < R; ++q) {
            if constexpr (MODE == FM_LAST) {
                const cpx<T> y = scale(v[q], sc);
                v2 x;
                x.x = y.re;
                x.y = y.im;
                ((gout_t)gout)[to + q * PI] = x;
            } else {
                dst[lpad(to + q * PI, kFieldPad)] = v[q];
            }
        }
    }
    if constexpr (MODE != FM_LAST) __syncthreads();
}

template <typename T, int S, int TOP, int MODE>
__device__ __forceinline__ void field_stage_radix(int R, const cpx<T>* src, cpx<T>* dst, int elems, int n, int inner, int P,
                                                  const void* tw, const cpx<T>* gin, cpx<T>* gout, const T sc) {
    switch (R) {
#define VKFX_FIELD_CASE(RR) \
    case RR:                \
        if constexpr (RR <= TOP) field_stage<T, S, RR, MODE>(src, dst, elems, n, inner, P, tw, gin, gout, sc); \
        break;
        VKFX_FIELD_CASE(2)
        VKFX_FIELD_CASE(3)
        VKFX_FIELD_CASE(4)
        VKFX_FIELD_CASE(5)
        VKFX_FIELD_CASE(6)
        VKFX_FIELD_CASE(7)
        VKFX_FIELD_CASE(8)
        VKFX_FIELD_CASE(9)
        VKFX_FIELD_CASE(10)
        VKFX_FIELD_CASE(11)
        VKFX_FIELD_CASE(12)
        VKFX_FIELD_CASE(13)
        VKFX_FIELD_CASE(16)
#undef VKFX_FIELD_CASE
        default: break;
    }
}

// a.N points a field, a.nlines fields, field_pack(a) fields a block; field_dim, field_roots,
// field_stages: length, roots and number of stages of each axis, last axis first;
// a.radix: all stages in order. KF_FIELD_COPY: the fields are copied to LDS
// before the first stage.
template <typename T, int S, int TOP>
__global__ __launch_bounds__(512) void k_field(const KArgs a) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    cpx<T>* src = reinterpret_cast<cpx<T>*>(smem_raw);
    cpx<T>* dst = src + a.LS / 2;
    const long long first = (long long)blockIdx.x * field_pack(a), left = a.nlines - first;
    const int elems = (int)(left < field_pack(a) ? left : field_pack(a)) * a.N;
    const cpx<T>* in = (const cpx<T>*)a.in + first * a.N;
    cpx<T>* out = (cpx<T>*)a.out + first * a.N;
    const bool copy = (a.flags & KF_FIELD_COPY) != 0;
    if (copy) {
        for (int e = threadIdx.x; e < elems; e += blockDim.x) src[lpad(e, kFieldPad)] = in[e];
        __syncthreads();
    }
    int inner = 1, s = 0;
    for (int ax = 0; ax < 3; ++ax) {
        const int n = field_dim(a, ax);
        for (int j = 0, P = 1; j < field_stages(a, ax); ++j, ++s) {
            const int R = a.radix[s];
            if (s + 1 == a.nstages)
                field_stage_radix<T, S, TOP, FM_LAST>(R, src, dst, elems, n, inner, P, field_roots(a, ax), in, out, (T)a.scale);
            else if (s == 0 && !copy)
                field_stage_radix<T, S, TOP, FM_FIRST>(R, src, dst, elems, n, inner, P, field_roots(a, ax), in, out, (T)1);
            else
                field_stage_radix<T, S, TOP, FM_LDS>(R, src, dst, elems, n, inner, P, field_roots(a, ax), in, out, (T)1);
            P *= R;
            cpx<T>* x = src;
            src = dst;
            dst = x;
        }
        inner *= n;
    }
}

}  // namespace vkfx
