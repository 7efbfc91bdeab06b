// hc_coef.hpp - device code of the (h, g)-derived coefficients of the H.C
// kernels: the block of the one-stage rows (hamiltonian.hpp) and the pair
// matrix of the two-stage form (hamiltonian_two.hpp).
#pragma once

#include "hamiltonian.hpp"

namespace mctdhb {

// With sum_m n_m = N the last occupation is folded into the single-jump
// coefficients: A'_kl = A_kl + N B_kl,M-1 and B'_klm = B_klm - B_kl,M-1, so
// F_kl(n) = A'_kl + sum_{m < M-1} n_m B'_klm.
// Entries t, t + stride, ...
__device__ __forceinline__ void hc_coefficients_part(int t, int stride, int M, int N, const double2* __restrict__ hob,
                                                     const double2* __restrict__ hint, double2* __restrict__ cf64,
                                                     float2* __restrict__ cf32) {
    const int M2 = M * M, M3 = M2 * M;
    auto G = [&](int a, int b, int c, int d) { return hint[a + b * M + c * M2 + d * M3]; };
    double2* d64 = cf32 ? (double2*) (cf32 + cf_f64_off(M)) : nullptr;
    auto put = [&](int idx, double2 v) {
        cf64[idx] = v;
        if (cf32) {
            cf32[idx] = make_float2((float) v.x, (float) v.y);
            // the one-body and diagonal sections once more in FP64
            if (idx < cf_f64_count(M)) d64[idx] = v;
        }
    };
    const int total = cf_size(M);
    for (int idx = t; idx < total; idx += stride) {
        double2 v = make_double2(0, 0);
        // B_klm = g_kkkl (m = k), g_klll (m = l), 2 g_kmml (otherwise)
        auto B = [&](int k, int l, int m) {
            if (m == k) return G(k, k, k, l);
            if (m == l) return G(k, l, l, l);
            return cscale(G(k, m, m, l), 2.0);
        };
        if (idx < cf_off_B(M)) {  // A'_kl = h_kl - g_kkkl + N B_kl,M-1
            int k = idx / M, l = idx % M;
            if (k != l) v = hob[k * M + l] - G(k, k, k, l) + cscale(B(k, l, M - 1), (double) N);
        } else if (idx < cf_off_d1(M)) {  // B'_klm = B_klm - B_kl,M-1
            int r = idx - cf_off_B(M);
            int k = r / M2, l = (r / M) % M, m = r % M;
            if (k != l && m < M - 1) v = B(k, l, m) - B(k, l, M - 1);
        } else if (idx < cf_off_d2(M)) {  // d1_k = h_kk - g_kkkk / 2
            int k = idx - cf_off_d1(M);
            v = hob[k * M + k] - cscale(G(k, k, k, k), 0.5);
        } else if (idx < cf_off_d3(M)) {  // d2_k = g_kkkk / 2
            int k = idx - cf_off_d2(M);
            v = cscale(G(k, k, k, k), 0.5);
        } else if (idx < cf_off_ot(M)) {  // d3_ks = 2 g_ksks (k < s)
            int r = idx - cf_off_d3(M);
            int k = r / M, s = r % M;
            if (k < s) v = cscale(G(k, s, k, s), 2.0);
        } else if (idx < cf_off_tt(M)) {  // Got[k][q][l]
            int r = idx - cf_off_ot(M);
            int k = r / M2, q = (r / M) % M, l = r % M;
            if (q != k && l != k && q <= l) v = (q == l) ? cscale(G(k, k, q, q), 0.5) : G(k, k, q, l);
        } else {  // Gtt[k][s][q][l]
            int r = idx - cf_off_tt(M);
            int k = r / M3, s = (r / M2) % M, q = (r / M) % M, l = r % M;
            if (k < s && q <= l && q != k && q != s && l != k && l != s)
                v = (q == l) ? G(k, s, q, q) : cscale(G(k, s, q, l), 2.0);
        }
        put(idx, v);
    }
}

// Entry X[a][b] for row pair (k <= s), column pair (q <= l), from the entries
// the fused row uses (so the result does not depend on symmetries of h and g
// that row does not need).  rn = 1 / (N - 1).
__device__ __forceinline__ double2 pair_element(int M, int k, int s, int q, int l, double rn,
                                                const double2* __restrict__ hob, const double2* __restrict__ hint) {
    const int M2 = M * M, M3 = M2 * M;
    auto G = [&](int a, int b, int c, int d) { return hint[a + b * M + c * M2 + d * M3]; };
    auto h = [&](int a, int b) { return cscale(hob[a * M + b], rn); };
    if (k == q && s == l) {  // the pair stays
        if (k == s) return cscale(G(k, k, k, k), 0.5) + h(k, k);
        return cscale(G(k, s, k, s), 2.0) + h(k, k) + h(s, s);
    }
    if (k == s && (q == k || l == k)) {  // k, k <- k, b
        const int b = q == k ? l : q;
        return G(k, k, k, b) + h(k, b);
    }
    if (q == l && (q == k || q == s)) {  // a, q <- q, q
        const int a = q == k ? s : k;
        return G(a, q, q, q) + h(a, q);
    }
    if (k != s && q != l && (k == q || k == l || s == q || s == l)) {  // a, m <- m, b
        const int m = k == q || k == l ? k : s, a = m == k ? s : k, b = m == q ? l : q;
        return cscale(G(a, m, m, b), 2.0) + h(a, b);
    }
    if (k == s) return q == l ? cscale(G(k, k, q, q), 0.5) : G(k, k, q, l);
    return q == l ? G(k, s, q, q) : cscale(G(k, s, q, l), 2.0);
}

// X (P x P; h alone, M x M, for one particle), entries t, t + stride, ...
__device__ __forceinline__ void pair_matrix_part(int t, int stride, int M, int N, const double2* __restrict__ hob,
                                                 const double2* __restrict__ hint, double2* __restrict__ X) {
    const int P = M * (M + 1) / 2;
    if (N == 1) {
        for (int e = t; e < M * M; e += stride) X[e] = hob[e];
        return;
    }
    auto pair = [&](int p, int& a, int& b) {
        a = 0;
        while (p >= M - a) p -= M - a++;
        b = a + p;
    };
    for (int e = t; e < P * P; e += stride) {
        int k, s, q, l;
        pair(e / P, k, s);
        pair(e % P, q, l);
        X[e] = pair_element(M, k, s, q, l, 1.0 / (N - 1), hob, hint);
    }
}

}  // namespace mctdhb
