// analytic_terms.hpp - H(k) of an analytic tight-binding class as a short
// trigonometric sum, the form the time-fused N-band kernel evaluates per
// matrix element (nband_evolve.hip).
#pragma once

#include <vector>

#include "antelope/sbe_c.h"

namespace sbe {

constexpr int kMaxTerms = 9;  // TMDCs.h: third neighbours, nine +-v pairs

// H(k) = m0 + sum_t p_t cos(k.v_t) + q_t sin(k.v_t) with Hermitian N x N
// matrices (row-major [re, im]), and the Hermitian part of the class's current
// J_a(k) = scale o sum_t grad_t[a] (q_t cos(k.v_t) - p_t sin(k.v_t)): scale is
// one complex factor per element (-1 where J = -dH/dk, +1 where it is +dH/dk).
struct AnalyticTerms {
    int T = 0;
    double vec[kMaxTerms][3] = {}, grad[kMaxTerms][3] = {};
    std::vector<double> m0, p, q;  // [N*N*2], [T][N*N*2]
    std::vector<double> scale;     // [N*N*2]
};

// false when the class (or its current) has no such form: MultiWSM (powers of
// k), Haldane2L with a distinct bottom layer, or more than kMaxTerms pairs.
// The form found is compared with the class's own H and J at points off the
// sampling grid and refused beyond 1e-12 of their size.
bool analytic_terms(int kind, int N, const double *params, AnalyticTerms &out);

}  // namespace sbe
