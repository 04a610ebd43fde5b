// Host-side checks of csrc/roots.hpp: every root of every length up to 700 and of
// some longer ones against the direct evaluation. Prints "ok <roots>" and exits 0.
#include <cstdio>

#include "roots.hpp"

int main() {
    std::vector<size_t> lengths;
    for (size_t n = 1; n <= 700; ++n) lengths.push_back(n);
    for (size_t n : {1000, 1001, 1024, 1080, 2187, 3087, 4096, 8190, 8192}) lengths.push_back(n);
    size_t total = 0;
    for (size_t n : lengths) {
        std::vector<long double> re, im;
        vkfx::roots(n, re, im);
        if (re.size() != n || im.size() != n) return std::printf("FAIL size at %zu\n", n), 1;
        for (size_t k = 0; k < n; ++k, ++total) {
            long double c, s;
            vkfx::root((long double)k, (long double)n, c, s);
            // the direct evaluation's angle is rounded to 2 pi * 2^-64, the products add 3 * 2^-64
            if (fabsl(re[k] - c) > 1e-18L || fabsl(im[k] - s) > 1e-18L) {
                std::printf("FAIL n %zu k %zu: %Lg %Lg, want %Lg %Lg\n", n, k, re[k], im[k], c, s);
                return 1;
            }
        }
        // the axes and diagonals of the circle
        if (re[0] != 1.0L || im[0] != 0.0L) return std::printf("FAIL root 0 of %zu\n", n), 1;
        if (n % 2 == 0 && (re[n / 2] != -1.0L || im[n / 2] != 0.0L)) return std::printf("FAIL half of %zu\n", n), 1;
        for (size_t count : {(size_t)0, (size_t)1, n / 4 + 1, n / 2, n - 1, n + 5}) {
            std::vector<long double> a, b;
            vkfx::roots(n, a, b, count);
            if (a.size() != (count < n ? count : n)) return std::printf("FAIL count %zu of %zu\n", count, n), 1;
            for (size_t k = 0; k < a.size(); ++k)
                if (a[k] != re[k] || b[k] != im[k]) return std::printf("FAIL root %zu of %zu, first %zu\n", k, n, count), 1;
        }
        if (n % 4 == 0 && (re[n / 4] != 0.0L || im[n / 4] != -1.0L)) return std::printf("FAIL quarter of %zu\n", n), 1;
    }
    std::printf("ok %zu\n", total);
    return 0;
}
