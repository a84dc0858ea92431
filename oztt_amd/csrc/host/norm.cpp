// See norm.hpp. Compiled with -ffp-contract=off, like the reference (its Makefile:51-53).
#include "norm.hpp"

#include <algorithm>
#include <cstdint>
#include <cmath>
#include <limits>
#include <random>
#include <vector>

namespace ozTTgemm::detail {

static_assert(std::numeric_limits<long double>::digits == 64,
              "the norm estimate accumulates in x86 extended precision, like the reference (bits.hpp:18-19)");

double pow2_scale(const double* v, std::size_t n) {
    // the maximum does not depend on the order of the comparisons: blocks in parallel
    double mx = 0;
#pragma omp parallel for schedule(static) reduction(max : mx)
    for (std::int64_t i = 0; i < (std::int64_t)n; i++) mx = std::max(mx, std::fabs(v[i]));
    if (!(mx > 0) || !std::isfinite(mx)) return 1.0;
    int e;
    std::frexp(mx, &e);
    e = std::min(std::max(e, -1000), 1000);
    return std::ldexp(1.0, e);
}

namespace {

constexpr std::uint32_t kProbes = 8;

// out[kProbes r + l] = sum_c (X[r][c] * rg) * v[kProbes c + l] for every row r < rows and probe l, each sum
// in column order in x86 extended precision (norm_estimate.hpp:35-44). All probes take one pass over X, four
// of them at a time: X[r][c] * rg is computed and moved to the x87 registers once for four, the four
// chains overlap, X is read from memory once, and one parallel loop does for eight. A sum's own sequence
// of operations, and so its value, does not depend on that. The whole plan of 2048^3 went from 5.75-5.87 to
// 4.94-5.28 ms, of 1024^3 (with the shorter search for the last moduli, plan2.cpp) from 1.73 to 1.35.
void matvecs_x87(const double* X, std::uint32_t rows, std::uint32_t cols, double rg, const double* v, double* out) {
#pragma omp parallel for schedule(static)
    for (std::int64_t r = 0; r < (std::int64_t)rows; r++) {
        const double* x = X + (std::size_t)r * cols;
        for (std::uint32_t l = 0; l < kProbes; l += 4) {
            const double* p = v + l;
            long double s0 = 0, s1 = 0, s2 = 0, s3 = 0;
            for (std::uint32_t c = 0; c < cols; c++, p += kProbes) {
                const long double xc = x[c] * rg;
                s0 += xc * p[0];
                s1 += xc * p[1];
                s2 += xc * p[2];
                s3 += xc * p[3];
            }
            double* o = out + (std::size_t)r * kProbes + l;
            o[0] = (double)s0;
            o[1] = (double)s1;
            o[2] = (double)s2;
            o[3] = (double)s3;
        }
    }
}

}  // namespace

double estimate_product_norm(const double* A, const double* B, std::uint32_t M, std::uint32_t N, std::uint32_t K,
                             double rgA, double rgB) {
    constexpr std::uint32_t L = kProbes;
    std::mt19937 rg(12345);
    std::normal_distribution<double> nd(0.0, 1.0);
    std::vector<double> g((std::size_t)L * N), y((std::size_t)L * K), p((std::size_t)L * M);
    for (std::uint32_t l = 0; l < L; l++)  // the probes in the reference's order
        for (std::uint32_t j = 0; j < N; j++) g[(std::size_t)L * j + l] = nd(rg);
    matvecs_x87(B, K, N, rgB, g.data(), y.data());
    matvecs_x87(A, M, K, rgA, y.data(), p.data());
    double cs2 = 0, cmax = 0;
    for (std::uint32_t l = 0; l < L; l++) {
        double q = 0;
        for (std::uint32_t i = 0; i < M; i++) q += p[(std::size_t)L * i + l] * p[(std::size_t)L * i + l];
        cs2 += q;
        cmax = std::max(cmax, q);
    }
    return (cs2 - cmax) / (L - 1) / (1.0 + 2.0 * std::sqrt(2.0 / (double)L));
}

}  // namespace ozTTgemm::detail
