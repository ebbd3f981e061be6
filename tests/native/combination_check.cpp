// Host driver for combination_coefficients (tm_internal.hpp): prints the
// coefficients of K iterations.  alpha_i = 1 / (i + 1), beta_i = i / 8, at the
// given stride; every value the K iterations do not write is NaN.
// Usage: combination_check K STRIDE
#include "tm_internal.hpp"

#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <vector>

int main(int argc, char** argv) {
    if (argc < 3) return 2;
    const int K = std::atoi(argv[1]), stride = std::atoi(argv[2]);
    std::vector<double> ah((size_t)(K + 1) * stride, NAN), bh(ah), c((size_t)K, 0.0);
    for (int i = 0; i < K; ++i) {
        ah[(size_t)i * stride] = 1.0 / (i + 1);
        bh[(size_t)i * stride] = i / 8.0;
    }
    tmh::combination_coefficients(K, ah.data(), bh.data(), stride, [&](int i, double v) { c[i] = v; });
    for (double v : c) std::printf("%.17g\n", v);
    return 0;
}
