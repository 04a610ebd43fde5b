// roots.hpp -- roots of unity in long double, host side.
#pragma once
#include <cmath>
#include <cstddef>
#include <vector>

namespace vkfx {

constexpr long double kPiL = 3.141592653589793238462643383279502884L;

// exp(-2 pi i k / n) with exact integer reduction of k.
inline void root(long double k, long double n, long double& c, long double& s) {
    const long double a = -2.0L * kPiL * k / n;
    c = cosl(a);
    s = sinl(a);
}

// exp(-2 pi i k / n) for all k < n, or the first `count` of them. The first eighth of the circle (n a multiple of
// 4), the first quarter (other even n) or half (odd n) is formed, each root as a
// product of two of about 2 sqrt(n) evaluated ones (within 3 units of 2^-64, the
// error of the evaluations' angle); the rest are its reflections, exact in every
// bit. The evaluations were the larger part of a plan's creation (1080 roots one by
// one: 223 us; the plan of 1080 x 1920 700 us, 130 this way).
inline void roots(size_t n, std::vector<long double>& re, std::vector<long double>& im, size_t count = (size_t)-1) {
    count = count < n ? count : n;
    re.assign(count, 0.0L);
    im.assign(count, 0.0L);
    const size_t half = n / 2, quarter = n / 4;
    const size_t first = n % 4 == 0 ? n / 8 : n % 2 == 0 ? quarter : half;
    size_t block = 1;
    while (block * block <= first) block *= 2;
    for (size_t k = 0; k <= first && k < count; ++k) {
        const size_t a = k / block * block, b = k - a;
        if (a == 0 || b == 0) {
            root((long double)k, (long double)n, re[k], im[k]);
        } else {
            re[k] = re[a] * re[b] - im[a] * im[b];
            im[k] = re[a] * im[b] + im[a] * re[b];
        }
    }
    size_t k = first + 1;
    if (n % 4 == 0)
        for (; k <= quarter && k < count; ++k) re[k] = -im[quarter - k], im[k] = -re[quarter - k];
    if (n % 2 == 0)
        for (; k <= half && k < count; ++k) re[k] = -re[half - k], im[k] = im[half - k];
    for (; k < count; ++k) re[k] = re[n - k], im[k] = -im[n - k];
}

}  // namespace vkfx
