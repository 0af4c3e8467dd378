// The arithmetic that stands for divisions in the embedding (pl_device.h), compiled for the host, against the
// divisions: bit for bit over the range that the comments there name, and an ulp beyond it.
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <random>

#include "pl_device.h"

namespace {

using plk::device::divided;
using plk::device::scaled_down;

long g_failures = 0;
std::mt19937_64 g_random(1);

// a number with random sign and mantissa and an exponent from `low` to `high`
template <typename T>
T random_number(int low, int high) {
    const double mantissa = 1.0 + (double)(g_random() >> 12) * 0x1p-52;   // (all 53 bits)
    const int exponent = low + (int)(g_random() % (uint64_t)(high - low + 1));
    return (T)((g_random() & 1 ? -1.0 : 1.0) * std::ldexp((double)(T)mantissa, exponent));
}

template <typename T>
void same(T got, T want, const char *what, double a, double b) {
    if (got == want || (std::isnan(got) && std::isnan(want))) return;
    if (++g_failures <= 10) std::printf("%s: %a and %a give %a, not %a\n", what, a, b, (double)got, (double)want);
}
template <typename T>
void an_ulp_apart(T got, T want, const char *what, double a, double b) {
    if (got == std::nextafter(want, (T)INFINITY) || got == std::nextafter(want, (T)-INFINITY)) return;
    same(got, want, what, a, b);
}

template <typename T>
void divisions(long n) {
    const T ordinary[] = {8, (T)0.125, (T)3.3, (T)0.07, (T)0.37, 13, 80, 3, 5, (T)0.1, (T)-1.7, (T)0x1p-40, (T)0x1p40,
                          std::nextafter((T)2, (T)1), std::nextafter((T)1, (T)2)};
    for (const T b : ordinary) {
        const T inverse = (T)1 / b;
        for (int i = 0; i < 70000; ++i) same(divided((T)i, b, inverse), (T)i / b, "coordinate", i, (double)b);
        for (long i = 0; i < n / 16; ++i) {
            const T a = random_number<T>(-100, 60);
            same(divided(a, b, inverse), a / b, "channel", (double)a, (double)b);
        }
    }
    for (long i = 0; i < n; ++i) {
        const T b = random_number<T>(-40, 39), a = random_number<T>(-100, 39);
        same(divided(a, b, (T)1 / b), a / b, "channel", (double)a, (double)b);
    }
    // smaller channels, down to the smallest of all
    for (long i = 0; i < n; ++i) {
        const T b = random_number<T>(-40, 39), a = random_number<T>(-149, -101);
        an_ulp_apart(divided(a, b, (T)1 / b), a / b, "small channel", (double)a, (double)b);
    }
    same(divided((T)0, (T)3, (T)1 / (T)3), (T)0, "zero", 0, 3);
    same(divided((T)NAN, (T)3, (T)1 / (T)3), (T)NAN, "NaN", NAN, 3);
}

template <int D1>
void scaling(long n) {
    auto want = [](float x) { return (float)((double)x * (1.0 / (double)D1)); };
    for (const int exponent : {0, 1, -90, 60, 100})
        for (uint32_t m = 0; m < 1u << 23; m += 1 + (exponent != 0) * 7) {
            const float x = std::ldexp(1.0f + (float)m * 0x1p-23f, exponent);
            same(scaled_down<D1>(x), want(x), "scaled", x, D1);
        }
    for (long i = 0; i < n; ++i) {
        const float x = random_number<float>(-90, 126), tiny = random_number<float>(-126, -90);
        same(scaled_down<D1>(x), want(x), "scaled", x, D1);
        an_ulp_apart(scaled_down<D1>(tiny), want(tiny), "small, scaled", tiny, D1);
    }
    for (const float x : {0.0f, INFINITY, -INFINITY, NAN}) same(scaled_down<D1>(x), want(x), "scaled", x, D1);
}

}  // namespace

int main() {
    divisions<float>(1000000);
    divisions<double>(1000000);
    scaling<2>(1000000);
    scaling<3>(1000000);
    scaling<4>(1000000);
    scaling<5>(1000000);
    scaling<6>(1000000);
    scaling<7>(1000000);
    scaling<8>(1000000);
    scaling<9>(1000000);
    std::printf("%ld differ\n", g_failures);
    return g_failures ? 1 : 0;
}
