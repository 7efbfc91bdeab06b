// pairs.hpp - the space of N - 2 particles seen from N: with
// phi_ql = a_q a_l C (q <= l, P = M (M + 1) / 2 pairs), every two-body
// quantity is a small dense contraction over pairs at each of its
// configurations n' (rho2 = sum conj(phi_ks) phi_ql, and
// H C = sum a+_k a+_s sum G phi_ql), with P coefficient reads per n'.
//
// phi_ql(n') = sqrt((n'_q + 1)(n'_l + 1 + [q = l])) C[rank(n' + e_q + e_l)],
// rank(n) = NC - 1 - sum_m W_m(P_m) (fock.hpp): adding the pair raises the
// prefix occupation P'_m by [q <= m] + [l <= m].
#pragma once

#include "fock.hpp"

namespace mctdhb {

constexpr int pair_count(int M) { return M * (M + 1) / 2; }
// position of the pair q <= l in lexicographic order
__host__ __device__ constexpr int pair_index(int M, int q, int l) { return q * M - q * (q - 1) / 2 + (l - q); }
// its orbitals, as tables: indices of unrolled loops fold to constants
template <int M> struct PairTable {
    int q[pair_count(M)], l[pair_count(M)];
    constexpr PairTable() : q{}, l{} {
        int p = 0;
        for (int a = 0; a < M; a++)
            for (int b = a; b < M; b++) {
                q[p] = a;
                l[p++] = b;
            }
    }
};
template <int M> constexpr PairTable<M> kPairTable{};

// A configuration of N - 2 particles is stored as its M prefix occupations
// P'_0 .. P'_{M-1} = N - 2 in one 64-bit word, fields of low_bits(M) bits:
// spaces below 2^32 / M configurations have N <= 10000, 1860, 378, 150 and
// 85 for M = 3 .. 7 (and N <= 10000 at M = 2).
constexpr int low_bits(int M) { return M <= 4 ? 16 : M == 5 ? 12 : 8; }
constexpr uint64_t low_mask(int M) { return (1ull << low_bits(M)) - 1; }

struct LowCtx {
    const uint64_t* rows;  // prefix words of the N - 2 space
    uint32_t dim;          // its size (0 for N = 1)
    uint32_t top;          // NC of the N space
    int npar;              // N
};

// One configuration n' in a lane: the ranks of n' + e_q + e_l and the roots.
// Adding the pair raises P'_m by one for q <= m < l and by two for m >= l, so
// with d1_m, d2_m the falls of the rank for one and two at level m,
//   rank(n' + e_q + e_l) = from[q] + to[l],
//   from[q] = rank(n') - sum_{m >= q} d1_m,  to[l] = sum_{m >= l} (d1_m - d2_m).
template <int M> struct LowRow {
    uint32_t from[M], to[M];
    uint32_t n[M];  // occupations of n'

    __device__ __forceinline__ void set(uint64_t row, const uint32_t* __restrict__ Wl, int ldw, uint32_t top) {
        constexpr int B = low_bits(M);
        constexpr uint32_t mask = (uint32_t) low_mask(M);
        uint32_t P[M], d1[M], d2[M];
#pragma unroll
        for (int m = 0; m < M; m++) {
            P[m] = (uint32_t) (row >> (B * m)) & mask;
            n[m] = m ? P[m] - P[m - 1] : P[0];
        }
        uint32_t base = top - 1u;
#pragma unroll
        for (int m = 0; m < M - 1; m++) {
            const uint32_t* w = Wl + m * ldw + kWOff + P[m];
            const uint32_t w0 = w[0];
            d1[m] = w[1] - w0;
            d2[m] = w[2] - w0;
            base -= w0;
        }
        from[M - 1] = base;
        to[M - 1] = 0;
#pragma unroll
        for (int m = M - 2; m >= 0; m--) {
            from[m] = from[m + 1] - d1[m];
            to[m] = to[m + 1] + d1[m] - d2[m];
        }
    }
};

// FP64 matrix product of the wave: D[4 i + g][c] += sum_k A[.][k] B[k][.],
// lane (g = lane / 16, c = lane % 16) holding A[c][g], B[g][c] and, in
// element i, D[4 i + g][c].
typedef double mat4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ mat4 mma(double a, double b, mat4 d) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, d, 0, 0, 0);
}

}  // namespace mctdhb
