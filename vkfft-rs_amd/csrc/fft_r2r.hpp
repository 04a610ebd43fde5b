// fft_r2r.hpp -- DCT / DST lines in one kernel (policies of
// fft_kernels_impl.hpp, which includes this file after IoPlain).
//
// The line's n = a.nvalid reals are gathered into LDS as the complex line of
// the type's FFT, transformed there, and the outputs formed from LDS (both
// ends staged: a stage's elements are not adjacent reals). The even types pack
// two reals of the reordered line into one complex element, as an even R2C
// does, so the FFT has half the length of a complex FFT over reals with zero
// imaginary parts; every line stays on its own (two lines packed into one
// complex line would share rounding errors, infinities and NaNs). The phases
// and the half-size pre- and postprocess run in f64 in both precisions.
//
// Bound by HBM: 8 bytes of traffic a real (f32) in one pass, against a pre
// pass, a full-length complex FFT and a post pass (40 bytes a real, with the
// phases from sincospi and strided gathers). f32 DCT-II and its normalized
// inverse over 16 x 720 x 1280: 1020 us in 12 launches before, 131 us in 4 (32-36
// us a pass over 118 MB, 3.3-3.5 TB/s), with the error against 64 bits at 2.2e-7
// from 3.9e-7. The first version, with block-wide copies whose loads wait one at a
// time and a table lookup per phase, ran 276 us.
#pragma once

namespace vkfx {

// exp(-2 pi i k / L) of the launch's f64 phase table (one level for short lines)
__device__ __forceinline__ cpx<double> r2r_root(const KArgs& a, long long k) {
    return tw2<double>(a.rlo, a.rhi, a.rshift, k);
}
template <typename T>
__device__ __forceinline__ cpx<double> r2r_wide(cpx<T> v) {
    return mk((double)v.re, (double)v.im);
}
template <typename T>
__device__ __forceinline__ cpx<T> r2r_narrow(cpx<double> v) {
    return mk((T)v.re, (T)v.im);
}
// exp(i pi / 4) w
__device__ __forceinline__ cpx<double> r2r_eighth(cpx<double> w) {
    constexpr double h = 0.707106781186547524400844362104849039;
    return mk(h * (w.re - w.im), h * (w.re + w.im));
}
// Two adjacent reals of a contiguous line; the caller's buffer is aligned to
// one real only.
template <bool NT, typename T>
__device__ __forceinline__ cpx<T> r2r_ld2(const T* p) {
    typedef T v2 __attribute__((ext_vector_type(2), aligned(sizeof(T))));
    v2 v;
    if constexpr (NT)
        v = __builtin_nontemporal_load((const v2*)p);
    else
        v = *(const v2*)p;
    return mk(v.x, v.y);
}
template <bool NT, typename T>
__device__ __forceinline__ void r2r_st2(T* p, T x, T y) {
    typedef T v2 __attribute__((ext_vector_type(2), aligned(sizeof(T))));
    v2 v;
    v.x = x;
    v.y = y;
    if constexpr (NT)
        __builtin_nontemporal_store(v, (v2*)p);
    else
        *(v2*)p = v;
}
// Component m & 1 of complex element m / 2 of a packed line.
template <typename T>
__device__ __forceinline__ T& r2r_slot(cpx<T>* line, int m, int ps) {
    T* s = (T*)(line + lpad(m >> 1, ps));
    return s[m & 1];
}
// Makhoul's order: v[m] = x[2m] for m < ceil(n/2), else x[2(n-1-m)+1].
__device__ __forceinline__ int r2r_makhoul_pos(int j, int n) { return (j & 1) ? n - 1 - (j >> 1) : (j >> 1); }

// exp(-2 pi i k / L) for the k a thread visits. f32 lines of own-line shapes
// advance it by one f64 multiplication a visit (k grows by TT; the error of the
// at most 64 steps stays below 2^-45); f64 lines and the other shapes read
// the table at every k.
template <typename T, class D>
struct R2rPhase {
    static constexpr bool kStep = own_line<D>() && sizeof(T) == 4;
    cpx<double> w, step;
    __device__ __forceinline__ R2rPhase(const KArgs& a) {
        if constexpr (kStep) {
            const int tid = (int)threadIdx.x;
            w = r2r_root(a, D::COL ? tid / D::G(a) : tid % D::kTT);
            step = r2r_root(a, D::kTT);
        }
    }
    // the phase w_k and w_k^4
    __device__ __forceinline__ void next(const KArgs& a, int k, cpx<double>& wk, cpx<double>& w4) {
        if constexpr (kStep) {
            wk = w;
            const cpx<double> w2 = cmul(w, w);
            w4 = cmul(w2, w2);
            w = cmul(w, step);
        } else {
            wk = r2r_root(a, k);
            w4 = r2r_root(a, 4 * (long long)k);
        }
    }
};

// Type II over an even length n = 2M: v = Makhoul's reordering of x packed as
// z[i] = v[2i] + i v[2i+1], Z = FFT_M(z), V[k] = E + O and V[M-k] = conj(E - O)
// with E = (Z[k] + conj Z[M-k]) / 2, O = -i W (Z[k] - conj Z[M-k]) / 2,
// W = exp(-2 pi i k / n); then X[k] = 2 Re(w V[k]), X[n-k] = -2 Im(w V[k]) with
// w = exp(-i pi k / 2n). DST-II: x[j] (-1)^j on input, X taken at n-1-k.
struct IoR2rII : IoPlain {
    static constexpr bool kPtrLoad = false, kPtrStore = false;
    static constexpr int kLoad = LAY_STAGED;
    static constexpr int kStore = LAY_STAGED;
    template <typename T, class D>
    static __device__ __forceinline__ void prologue(const KArgs& a, cpx<T>* lds, const LineInfo* li) {
        const bool row = D::kFixed ? !D::COL : (a.flags & KF_IN_ROWMAJOR) != 0;
        const int n = (int)a.nvalid, PS = D::PS(a);
        const bool flip = a.rflip != 0;
        const T* in = (const T*)a.in;
        const long long es = a.in_es;
        // reals 2i and 2i+1 of the line are v[i] and v[n-1-i]
        visit_lines<D, D::kN, 8>(
            a, li, D::N(a), row,
            [&](const LineInfo& L, int i) {
                const T* p = in + L.ib + 2 * (long long)i * es;
                return row ? r2r_ld2<D::NTI>(p) : mk(ldg_s<D::NTI>(p), ldg_s<D::NTI>(p + es));
            },
            [&](const LineInfo&, int g, int i, cpx<T> u) {
                cpx<T>* line = lds + g * D::LS(a);
                r2r_slot(line, i, PS) = u.re;
                r2r_slot(line, n - 1 - i, PS) = flip ? -u.im : u.im;
            });
    }
    template <typename T, int S, class D>
    static __device__ __forceinline__ void epilogue(const KArgs& a, const cpx<T>* lds, const LineInfo* li) {
        const bool row = D::kFixed ? !D::COL : (a.flags & KF_OUT_ROWMAJOR) != 0;
        const int M = D::N(a), n = 2 * M, PS = D::PS(a);
        const bool flip = a.rflip != 0;
        T* out = (T*)a.out;
        const long long es = a.out_es;
        const double sc = a.scale;
        R2rPhase<T, D> phase(a);
        visit_lines<D, D::kN / 2 + 1, 1>(
            a, li, M / 2 + 1, row, [&](const LineInfo&, int) { return 0; },
            [&](const LineInfo& L, int g, int k, int) {
                cpx<double> w, W;
                phase.next(a, k, w, W);
                if (!L.valid) return;
                const cpx<T>* line = lds + g * D::LS(a);
                const cpx<double> A = r2r_wide(line[lpad(k, PS)]), B = conj(r2r_wide(line[lpad(k ? M - k : 0, PS)]));
                const cpx<double> E = A + B, O = muli<-1>(cmul(A - B, W));
                const cpx<double> u = E + O, v = E - O;  // 2 V[k], 2 conj V[M-k]
                T* y = out + L.ob;
                auto put = [&](int j, double x) {
                    stg_s<D::NTO>(y + (long long)(flip ? n - 1 - j : j) * es, (T)(sc * x));
                };
                put(k, w.re * u.re - w.im * u.im);
                if (k) put(n - k, -(w.re * u.im + w.im * u.re));
                if (2 * k != M) {
                    const cpx<double> wm = r2r_eighth(w);  // conj(w_(M-k))
                    put(M - k, wm.re * v.re - wm.im * v.im);
                    if (k) put(M + k, wm.re * v.im + wm.im * v.re);
                }
            });
    }
};

// Type III over an even length n = 2M: V[k] = conj(w)(x[k] - i x[n-k]) (x[n] = 0)
// and V[M-k] give Z[k] = P + Q, Z[M-k] = conj(P - Q) with P = V[k] + conj V[M-k],
// Q = i conj(W)(V[k] - conj V[M-k]); the inverse FFT_M is v packed, and
// x[2i] = v[i], x[2i+1] = v[n-1-i]. DST-III: x reversed on input, X[k] (-1)^k.
struct IoR2rIII : IoPlain {
    static constexpr bool kPtrLoad = false, kPtrStore = false;
    static constexpr int kLoad = LAY_STAGED;
    static constexpr int kStore = LAY_STAGED;
    template <typename T>
    struct Quad {
        T xk, xnk, xm, xp;  // x[k], x[n-k], x[M-k], x[M+k]
    };
    template <typename T, class D>
    static __device__ __forceinline__ void prologue(const KArgs& a, cpx<T>* lds, const LineInfo* li) {
        const bool row = D::kFixed ? !D::COL : (a.flags & KF_IN_ROWMAJOR) != 0;
        const int M = D::N(a), n = 2 * M, PS = D::PS(a);
        const bool flip = a.rflip != 0;
        const T* in = (const T*)a.in;
        const long long es = a.in_es;
        R2rPhase<T, D> phase(a);
        visit_lines<D, D::kN / 2 + 1, 4>(
            a, li, M / 2 + 1, row,
            [&](const LineInfo& L, int k) {
                const T* p = in + L.ib;
                auto at = [&](int j) { return ldg_s<D::NTI>(p + (long long)(flip ? n - 1 - j : j) * es); };
                // k = 0: x[n] does not exist (zero), x[M+k] = x[M-k]
                return Quad<T>{at(k), at(k ? n - k : M), at(M - k), at(M + k)};
            },
            [&](const LineInfo&, int g, int k, const Quad<T>& q) {
                cpx<double> w, W;
                phase.next(a, k, w, W);
                const double xk = q.xk, xnk = k ? (double)q.xnk : 0.0, xm = q.xm, xp = q.xp;
                const cpx<double> wm = r2r_eighth(w);  // conj(w_(M-k))
                const cpx<double> V = mk(xk * w.re - xnk * w.im, -xk * w.im - xnk * w.re);
                const cpx<double> Vm = mk(xm * wm.re + xp * wm.im, xm * wm.im - xp * wm.re);
                const cpx<double> P = V + conj(Vm), Q = muli<1>(cmulc(V - conj(Vm), W));
                cpx<T>* line = lds + g * D::LS(a);
                line[lpad(k, PS)] = r2r_narrow<T>(P + Q);
                if (k && 2 * k != M) line[lpad(M - k, PS)] = r2r_narrow<T>(conj(P - Q));
            });
    }
    template <typename T, int S, class D>
    static __device__ __forceinline__ void epilogue(const KArgs& a, const cpx<T>* lds, const LineInfo* li) {
        const bool row = D::kFixed ? !D::COL : (a.flags & KF_OUT_ROWMAJOR) != 0;
        const int n = (int)a.nvalid, PS = D::PS(a);
        const bool flip = a.rflip != 0;
        T* out = (T*)a.out;
        const long long es = a.out_es;
        const double sc = a.scale;
        visit_lines<D, D::kN, 1>(
            a, li, D::N(a), row, [&](const LineInfo&, int) { return 0; },
            [&](const LineInfo& L, int g, int i, int) {
                if (!L.valid) return;
                cpx<T>* line = const_cast<cpx<T>*>(lds) + g * D::LS(a);
                const T x = (T)(sc * (double)r2r_slot(line, i, PS));
                const T v = (T)(sc * (double)r2r_slot(line, n - 1 - i, PS));
                const T y = flip ? -v : v;
                T* p = out + L.ob + 2 * (long long)i * es;
                if (row) {
                    r2r_st2<D::NTO>(p, x, y);
                } else {
                    stg_s<D::NTO>(p, x);
                    stg_s<D::NTO>(p + es, y);
                }
            });
    }
};

// The other forms, on the runtime-shape kernels, chosen by a.rop:
// R2R_F_HALF (even type IV): z[j] = (x[2j] + i x[n-1-2j]) exp(-i pi (4j+1)/4n),
//   u = exp(-i pi j/n) FFT_M(z)[j], X[2j] = 2 Re u, X[n-1-2j] = -2 Im u; DST-IV: x
//   reversed, X[k] (-1)^k.
// R2R_F_SYM (type I): the even extension a[m] = x[m] (DCT-I, M = n - 1) or the odd
//   one a[m] = x[m-1], a[0] = a[M] = 0 (DST-I, M = n + 1), a[2M-m] = +-a[m], packed
//   as an even R2C of 2M reals; X[k] = A[k], or X[k-1] = -Im A[k].
// R2R_F_REORDER_FULL / R2R_F_SPECTRUM_FULL (odd types II / III): as the even
//   forms, with a full-length FFT over reals with zero imaginary parts.
struct IoR2rMisc : IoPlain {
    static constexpr bool kPtrLoad = false, kPtrStore = false;
    static constexpr int kLoad = LAY_STAGED;
    static constexpr int kStore = LAY_STAGED;
    template <typename T, class D>
    static __device__ void prologue(const KArgs& a, cpx<T>* lds, const LineInfo* li) {
        const bool row = (a.flags & KF_IN_ROWMAJOR) != 0;
        const int n = (int)a.nvalid, M = D::N(a), PS = D::PS(a);
        const bool flip = a.rflip != 0;
        const T* in = (const T*)a.in;
        const long long es = a.in_es;
        if (a.rop == R2R_F_HALF) {
            coop_for(D::G(a), M, row, [&](int g, int j) {
                const T* p = in + li[g].ib;
                auto at = [&](int i) { return (double)ldg_s<D::NTI>(p + (long long)(flip ? n - 1 - i : i) * es); };
                lds[g * D::LS(a) + lpad(j, PS)] =
                    r2r_narrow<T>(cmul(mk(at(2 * j), at(n - 1 - 2 * j)), r2r_root(a, 4 * (long long)j + 1)));
            });
        } else if (a.rop == R2R_F_SYM) {
            coop_for(D::G(a), M, row, [&](int g, int i) {
                const T* p = in + li[g].ib;
                auto at = [&](int m) -> T {
                    const int q = m <= M ? m : 2 * M - m;
                    if (!flip) return ldg_s<D::NTI>(p + (long long)q * es);
                    if (q == 0 || q == M) return (T)0;
                    const T v = ldg_s<D::NTI>(p + (long long)(q - 1) * es);
                    return m <= M ? v : -v;
                };
                lds[g * D::LS(a) + lpad(i, PS)] = mk(at(2 * i), at(2 * i + 1));
            });
        } else if (a.rop == R2R_F_REORDER_FULL) {
            coop_for(D::G(a), n, row, [&](int g, int j) {
                const T u = ldg_s<D::NTI>(in + li[g].ib + (long long)j * es);
                lds[g * D::LS(a) + lpad(r2r_makhoul_pos(j, n), PS)] = mk(flip && (j & 1) ? -u : u, (T)0);
            });
        } else {
            coop_for(D::G(a), n, row, [&](int g, int j) {
                const T* p = in + li[g].ib;
                auto at = [&](int i) { return (double)ldg_s<D::NTI>(p + (long long)(flip ? n - 1 - i : i) * es); };
                lds[g * D::LS(a) + lpad(j, PS)] = r2r_narrow<T>(cmulc(mk(at(j), j ? -at(n - j) : 0.0), r2r_root(a, j)));
            });
        }
    }
    template <typename T, int S, class D>
    static __device__ void epilogue(const KArgs& a, const cpx<T>* lds, const LineInfo* li) {
        const bool row = (a.flags & KF_OUT_ROWMAJOR) != 0;
        const int n = (int)a.nvalid, M = D::N(a), PS = D::PS(a);
        const bool flip = a.rflip != 0;
        T* out = (T*)a.out;
        const long long es = a.out_es;
        const double sc = a.scale;
        if (a.rop == R2R_F_HALF) {
            coop_for(D::G(a), M, row, [&](int g, int j) {
                if (!li[g].valid) return;
                const cpx<double> u = cmul(r2r_wide(lds[g * D::LS(a) + lpad(j, PS)]), r2r_root(a, 4 * (long long)j));
                T* y = out + li[g].ob;
                const double odd = flip ? 2.0 : -2.0;  // n - 1 - 2j is odd
                stg_s<D::NTO>(y + 2 * (long long)j * es, (T)(sc * (2.0 * u.re)));
                stg_s<D::NTO>(y + (long long)(n - 1 - 2 * j) * es, (T)(sc * (odd * u.im)));
            });
        } else if (a.rop == R2R_F_SYM) {
            coop_for(D::G(a), M / 2 + 1, row, [&](int g, int k) {
                if (!li[g].valid) return;
                const cpx<T>* line = lds + g * D::LS(a);
                const cpx<double> A = r2r_wide(line[lpad(k, PS)]), B = conj(r2r_wide(line[lpad(k ? M - k : 0, PS)]));
                const cpx<double> E = A + B, O = muli<-1>(cmul(A - B, r2r_root(a, k)));
                const cpx<double> u = E + O, v = E - O;  // 2 A[k], 2 conj A[M-k]
                T* y = out + li[g].ob;
                auto put = [&](int j, double x) { stg_s<D::NTO>(y + (long long)j * es, (T)(sc * (0.5 * x))); };
                if (!flip) {
                    put(k, u.re);
                    if (2 * k != M) put(M - k, v.re);
                } else if (k) {
                    put(k - 1, -u.im);
                    if (2 * k != M) put(M - k - 1, v.im);
                }
            });
        } else if (a.rop == R2R_F_REORDER_FULL) {
            coop_for(D::G(a), n, row, [&](int g, int k) {
                if (!li[g].valid) return;
                const cpx<double> z = r2r_wide(lds[g * D::LS(a) + lpad(k, PS)]), w = r2r_root(a, k);
                const int j = flip ? n - 1 - k : k;
                stg_s<D::NTO>(out + li[g].ob + (long long)j * es, (T)(sc * (2.0 * (z.re * w.re - z.im * w.im))));
            });
        } else {
            coop_for(D::G(a), n, row, [&](int g, int k) {
                if (!li[g].valid) return;
                const double v = (double)lds[g * D::LS(a) + lpad(r2r_makhoul_pos(k, n), PS)].re;
                stg_s<D::NTO>(out + li[g].ob + (long long)k * es, (T)(sc * (flip && (k & 1) ? -v : v)));
            });
        }
    }
};

}  // namespace vkfx
