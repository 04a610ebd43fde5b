// Host-side checks of the launch validation (csrc/launch_check.cpp) of the one-kernel
// DCT / DST lines and of the small fields: accepted launches of every form and rank,
// and each rule broken once. Prints "ok <cases>" and exits 0 when all agree.
#include <cstdio>
#include <cstring>

#include "kernels.hpp"

using namespace vkfx;

static int fails = 0, cases = 0;

static void expect(const char* name, hipError_t got, hipError_t want) {
    ++cases;
    if (got != want) {
        ++fails;
        std::printf("FAIL %s: got %d, want %d\n", name, (int)got, (int)want);
    }
}

static const double kTable = 0;
static const size_t kLimit = 160 * 1024;

static KArgs line_args(int N, long long n, int form, bool flip) {
    KArgs a;
    std::memset(&a, 0, sizeof a);
    a.N = N;
    a.TT = 4;
    a.G = 8;
    a.LS = N + 3;
    a.PS = 4;
    a.nstages = 1;
    a.radix[0] = N;
    a.in_es = a.out_es = 1;
    a.nvalid = n;
    a.rop = form;
    a.rflip = flip;
    a.rlo = a.rhi = &kTable;
    return a;
}
static hipError_t line(KernelKind kind, int dir, const KArgs& a) {
    return check_launch(kind, 0, dir, a, (unsigned)(a.G * a.TT), (size_t)a.G * a.LS * 8, kLimit, nullptr);
}

// axes: last one first, two stages each at most
static KArgs field_args(int rank, const int (*radix)[2]) {
    KArgs a;
    std::memset(&a, 0, sizeof a);
    a.N = 1;
    a.G = 1;
    a.TT = 64;
    for (int ax = 0; ax < 3; ++ax) {
        field_dim(a, ax) = 1;
        if (ax >= rank) continue;
        for (int j = 0; j < 2; ++j)
            if (radix[ax][j] > 1) {
                a.radix[a.nstages++] = radix[ax][j];
                field_dim(a, ax) *= radix[ax][j];
                ++field_stages(a, ax);
            }
        field_roots(a, ax) = &kTable;
        a.N *= field_dim(a, ax);
    }
    field_pack(a) = 1;
    a.LS = 2 * ((a.N + (a.N >> 3) + 2) / 2 * 2);
    return a;
}
static hipError_t field(int prec, const KArgs& a) {
    return check_launch(KK_FIELD, prec, -1, a, (unsigned)a.TT, (size_t)a.LS * (prec ? 16 : 8), kLimit, nullptr);
}

int main() {
    const hipError_t ok = hipSuccess, bad = hipErrorInvalidConfiguration;
    struct Form {
        const char* name;
        KernelKind kind;
        int dir, form, N;
        long long n;
        bool flip;
    };
    const Form forms[] = {{"type II", KK_R2R_II, -1, R2R_F_REORDER, 12, 24, false},
                          {"DST-II", KK_R2R_II, -1, R2R_F_REORDER, 12, 24, true},
                          {"type III", KK_R2R_III, 1, R2R_F_SPECTRUM, 12, 24, false},
                          {"type IV", KK_R2R_MISC, -1, R2R_F_HALF, 12, 24, false},
                          {"DCT-I", KK_R2R_MISC, -1, R2R_F_SYM, 12, 13, false},
                          {"DST-I", KK_R2R_MISC, -1, R2R_F_SYM, 12, 11, true},
                          {"odd type II", KK_R2R_MISC, -1, R2R_F_REORDER_FULL, 9, 9, false},
                          {"odd type III", KK_R2R_MISC, 1, R2R_F_SPECTRUM_FULL, 9, 9, false}};
    for (const Form& f : forms) {
        const KArgs a = line_args(f.N, f.n, f.form, f.flip);
        expect(f.name, line(f.kind, f.dir, a), ok);
        expect(f.name, line(f.kind, -f.dir, a), bad);  // the other direction
        KArgs b = a;
        b.nvalid += 1;  // no form of this N has that length
        expect(f.name, line(f.kind, f.dir, b), bad);
        b = a;
        b.rhi = nullptr;
        expect(f.name, line(f.kind, f.dir, b), bad);
        b = a;
        b.rop = 17;
        expect(f.name, line(f.kind, f.dir, b), bad);
        expect(f.name, line(f.kind == KK_R2R_MISC ? KK_R2R_II : KK_R2R_MISC, f.dir, a), bad);  // another kernel's form
        b = a;
        b.TT *= 32;  // more than 512 threads
        expect(f.name, line(f.kind, f.dir, b), bad);
    }
    const int r2[3][2] = {{8, 6}, {10, 0}, {0, 0}}, r3[3][2] = {{5, 0}, {4, 3}, {13, 2}}, big[3][2] = {{16, 0}, {12, 0}, {0, 0}};
    expect("field, rank 2", field(0, field_args(2, r2)), ok);
    expect("field, rank 2 f64", field(1, field_args(2, r2)), ok);
    KArgs f3 = field_args(3, r3);
    expect("field of radix 13 without its kernel", field(0, f3), bad);
    f3.flags = KF_FIELD_LARGE;
    expect("field, rank 3", field(0, f3), ok);
    expect("field, rank 3 f64", field(1, f3), ok);
    KArgs f = f3;
    field_roots(f, 2) = nullptr;
    expect("third axis without its roots", field(0, f), bad);
    f = f3;
    field_stages(f, 2) = 1;
    expect("third axis without its last stage", field(0, f), bad);
    f = f3;
    field_dim(f, 1) = 24;
    expect("axis length that is not the product of its radices", field(0, f), bad);
    f = f3;
    f.N += 1;
    expect("points that are not the product of the axes", field(0, f), bad);
    f = f3;
    f.LS -= 2 * ((f.N >> 3) + 2);
    expect("buffers without their pads", field(0, f), bad);
    f = f3;
    field_pack(f) = 2;
    expect("two fields in the LDS of one", field(0, f), bad);
    f = f3;
    field_pack(f) = 0;
    expect("no field a block", field(0, f), bad);
    f = f3;
    field_pack(f) = 65535 / f.N + 1;
    f.LS = 2 * (2 * f.N * field_pack(f));
    expect("indices beyond 16 bits", check_launch(KK_FIELD, 0, -1, f, 64, kLimit, kLimit, nullptr), bad);
    KArgs w = field_args(2, big);
    w.flags = KF_FIELD_LARGE;
    expect("field of radices 16 and 12", field(0, w), ok);
    expect("radix 12 in f64", field(1, w), bad);
    w.radix[0] = 14;
    expect("radix 14", field(0, w), bad);
    if (fails) return 1;
    std::printf("ok %d\n", cases);
    return 0;
}
