// hamiltonian_two.hpp - H.C in two stages over the space of N - 2 particles
// (pairs.hpp), instantiated once per orbital count in h2_m<M>.hip.
//
// With phi_b = a_q a_l C (pair b = q <= l),
//   psi_a(n') = sum_b X[a][b] phi_b(n')          (first stage, P x P per n')
//   (H C)(n)  = sum_{a = k <= s} f_a(n) psi_a(n - e_k - e_s)   (second stage)
//   f_ks = sqrt(n_k n_s), f_kk = sqrt(n_k (n_k - 1)).
// X holds the two-body factors of hamiltonian.hpp and, spread over the
// spectators as h_kl / (N - 1), the one-body matrix, so nothing else is left
// to add (N >= 2).
//
// Everything but the stored vectors and psi is FP64 in both forms: FP64 and
// FP32 operations with a scalar operand (the entries of X come from scalar
// registers) take the same time on this card, and the mixed product is then
// closer to the FP64 one than the one-stage form (relative error of a SIL step
// at N=30, M=7 1.7e-8 against 6.8e-8).  One lane per configuration, one row of
// X at a time: X is read through the scalar cache, phi stays in registers.
// The first stage is bound by its FP64 vector instructions (4 P^2 of about
// 4 P^2 + 230 per wave; 178 us of 179 at that rate at N=30, M=7), the second
// by reading psi.
#pragma once

#include "hamiltonian_impl.hpp"

namespace mctdhb {

constexpr int kTwoBlock = 256;

// phi_b of one configuration n' into registers.
template <int M, typename Z>
__device__ __forceinline__ void pair_states(double2 (&phi)[pair_count(M)], uint64_t row, uint32_t top,
                                            const Z* __restrict__ c, const uint32_t* __restrict__ Wl, int ldw,
                                            const double* __restrict__ sql) {
    constexpr int P = pair_count(M);
    LowRow<M> x;
    x.set(row, Wl, ldw, top);
    Z v[P];
#pragma unroll
    for (int p = 0; p < P; p++) v[p] = c[x.from[kPairTable<M>.q[p]] + x.to[kPairTable<M>.l[p]]];
    double r1[M], r2[M];
#pragma unroll
    for (int k = 0; k < M; k++) {
        r1[k] = sql[x.n[k] + 1];
        r2[k] = sql[x.n[k] + 2];
    }
#pragma unroll
    for (int p = 0; p < P; p++) {
        const int q = kPairTable<M>.q[p], l = kPairTable<M>.l[p];
        phi[p] = cscale(to_d2(v[p]), r1[q] * (q == l ? r2[q] : r1[l]));
    }
}

// Tables in LDS: W, then the roots 0 .. N + 2; behind `front` bytes.
template <int M>
__device__ __forceinline__ void two_tables(unsigned char* smem, size_t front, const uint32_t* __restrict__ Wg, int ldw,
                                           int npar, uint32_t*& Wl, double*& sql) {
    const int wsz = (M - 1) * ldw;
    Wl = (uint32_t*) (smem + front);
    sql = (double*) (smem + front + (((size_t) wsz * 4 + 15) & ~(size_t) 15));
    for (int t = threadIdx.x; t < wsz; t += blockDim.x) Wl[t] = Wg[t];
    for (int t = threadIdx.x; t < npar + 3; t += blockDim.x) sql[t] = sqrt((double) t);
    __syncthreads();
}

// First stage: psi[a * ld + n'].
template <int M, typename Z>
__global__ __launch_bounds__(kTwoBlock) void k_pair_product(LowCtx low, const Z* __restrict__ c,
                                                            const double2* __restrict__ X,
                                                            const uint32_t* __restrict__ Wg, int ldw, size_t ld,
                                                            int stop_check, const SilState* st,
                                                            Z* __restrict__ psi) {
    extern __shared__ __align__(16) unsigned char smem[];
    if (stop_check && st->stop) return;
    constexpr int P = pair_count(M);
    uint32_t* Wl;
    double* sql;
    two_tables<M>(smem, 0, Wg, ldw, low.npar, Wl, sql);
    const uint32_t i = xcd_block(blockIdx.x, gridDim.x) * kTwoBlock + threadIdx.x;
    if (i >= low.dim) return;
    double2 phi[P];
    pair_states<M, Z>(phi, low.rows[i], low.top, c, Wl, ldw, sql);
#pragma unroll 1
    for (int a = 0; a < P; a++) {
        double2 v = make_double2(0, 0);
#pragma unroll
        for (int b = 0; b < P; b++) v = cfma(X[a * P + b], phi[b], v);
        psi[a * ld + i] = from_d2<Z>(v);
    }
}

// <c, H c>, one sum per block, from the upper triangle of the Hermitian X:
// the last Lanczos iteration of every orbital count (N=100, M=5: 217 -> 117 us
// FP64, 143 -> 100 us mixed against half a one-stage row).
template <int M, typename Z>
__global__ __launch_bounds__(kTwoBlock) void k_pair_rayleigh(LowCtx low, const Z* __restrict__ c,
                                                             const double2* __restrict__ X,
                                                             const uint32_t* __restrict__ Wg, int ldw, int stop_check,
                                                             const SilState* st, double* __restrict__ part) {
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ double red[kTwoBlock / 64];
    if (stop_check && st->stop) return;
    constexpr int P = pair_count(M);
    uint32_t* Wl;
    double* sql;
    two_tables<M>(smem, 0, Wg, ldw, low.npar, Wl, sql);
    const uint32_t i = xcd_block(blockIdx.x, gridDim.x) * kTwoBlock + threadIdx.x;
    double e[1] = {0};
    if (i < low.dim) {
        double2 phi[P];
        pair_states<M, Z>(phi, low.rows[i], low.top, c, Wl, ldw, sql);
#pragma unroll
        for (int a = 0; a < P; a++) {
            double2 v = cscale(phi[a], 0.5 * X[a * P + a].x);
#pragma unroll
            for (int b = a + 1; b < P; b++) v = cfma(X[a * P + b], phi[b], v);
            e[0] += phi[a].x * v.x + phi[a].y * v.y;
        }
        e[0] *= 2.0;
    }
    block_sum<1>(e, red);
    if (threadIdx.x == 0) part[blockIdx.x] = e[0];
}

// One configuration n in a lane: byte offsets of n - e_k - e_s in an array of
// psi values and the annihilation roots.  Removing the pair lowers P_m by one
// for k <= m < s and by two for m >= s:
//   rank(n - e_k - e_s) = from[k] + to[s],
// with every jump out of an empty orbital sent past the end of the array by
// gone1 (one particle) or gone2 (two from one orbital), where a buffer load
// gives zero.
template <int M> struct HighRow {
    uint32_t from[M], to[M], gone1[M], gone2[M];
    double r0[M], rm[M];  // sqrt(n), sqrt(n - 1)

    __device__ __forceinline__ void set(uint32_t i, const RowCtx& ctx, uint32_t low_dim, int shift,
                                        const uint32_t* __restrict__ Wl, int ldw, const double* __restrict__ sql) {
        uint32_t n[M], P = 0;
        if (ctx.occ8) {
            const uint2 w = *(const uint2*) (ctx.occ8 + (size_t) i * 8);
#pragma unroll
            for (int k = 0; k < M; k++) n[k] = ((k < 4 ? w.x : w.y) >> (8 * (k & 3))) & 255u;
        } else {
#pragma unroll
            for (int k = 0; k < M; k++) n[k] = ctx.ht[(size_t) i * M + k];
        }
        uint32_t e1[M], e2[M], base = low_dim - 1u;
#pragma unroll
        for (int m = 0; m < M - 1; m++) {
            P += n[m];
            const uint32_t* w = Wl + m * ldw + kWOff + P;
            const uint32_t w0 = w[0];
            e1[m] = w0 - w[-1];
            e2[m] = w0 - w[-2];
            base -= w0;
        }
        from[M - 1] = base;
        to[M - 1] = 0;
#pragma unroll
        for (int m = M - 2; m >= 0; m--) {
            from[m] = from[m + 1] + e1[m];
            to[m] = to[m + 1] + e2[m] - e1[m];
        }
#pragma unroll
        for (int k = 0; k < M; k++) {
            from[k] <<= shift;
            to[k] <<= shift;
            gone1[k] = n[k] >= 1 ? 0u : ~0u;
            gone2[k] = n[k] >= 2 ? 0u : ~0u;
            r0[k] = sql[n[k]];
            rm[k] = sql[n[k] ? n[k] - 1 : 0];
        }
    }
};

template <typename Z> __device__ __forceinline__ double2 ld_psi(__amdgpu_buffer_rsrc_t r, uint32_t off);
template <> __device__ __forceinline__ double2 ld_psi<float2>(__amdgpu_buffer_rsrc_t r, uint32_t off) {
    return to_d2(ld8(r, off));
}
template <> __device__ __forceinline__ double2 ld_psi<double2>(__amdgpu_buffer_rsrc_t r, uint32_t off) {
    const u32x4_t v = __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0);
    return make_double2(__hiloint2double((int) v.y, (int) v.x), __hiloint2double((int) v.w, (int) v.z));
}

// Second stage: row i of H C to the epilogue.
template <int M, typename Z, typename Epi>
__global__ __launch_bounds__(kTwoBlock) void k_pair_collect(RowCtx ctx, uint32_t low_dim, const Z* __restrict__ c,
                                                            const Z* __restrict__ psi, size_t ld,
                                                            const uint32_t* __restrict__ Wg, int ldw, int stop_check,
                                                            const SilState* st, Epi epi) {
    extern __shared__ __align__(16) unsigned char smem[];
    if (stop_check && st->stop) return;
    constexpr int P = pair_count(M), SHIFT = sizeof(Z) == 16 ? 4 : 3;
    uint32_t* Wl;
    double* sql;
    two_tables<M>(smem, kRedBytes, Wg, ldw, ctx.npar, Wl, sql);
    const uint32_t i = xcd_block(blockIdx.x, gridDim.x) * kTwoBlock + threadIdx.x;
    const bool valid = i < ctx.dim;
    const auto pre = epi.prefetch(i, valid);
    HighRow<M> x;
    x.set(valid ? i : ctx.dim - 1, ctx, low_dim, SHIFT, Wl, ldw, sql);
    const double2 ci = to_d2(c[valid ? i : ctx.dim - 1]);
    double2 row = make_double2(0, 0);
#pragma unroll
    for (int p = 0; p < P; p++) {
        const int k = kPairTable<M>.q[p], s = kPairTable<M>.l[p];
        const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(
            (void*) (psi + p * ld), (short) 0, (int) (low_dim * (uint32_t) sizeof(Z)), 0x00020000);
        const uint32_t off = (x.from[k] + x.to[s]) | (k == s ? x.gone2[k] : x.gone1[k] | x.gone1[s]);
        const double2 v = ld_psi<Z>(r, off);
        const double f = x.r0[k] * (k == s ? x.rm[k] : x.r0[s]);
        row.x = fma(f, v.x, row.x);
        row.y = fma(f, v.y, row.y);
    }
    epi(i, valid, row, ci, (double*) smem, pre);
}

// ---------------------------------------------------------------- launches

inline size_t two_table_bytes(const Space* S) {
    return ((((size_t) (S->norb - 1) * S->ldw * 4) + 15) & ~(size_t) 15) + sizeof(double) * (S->npar + 3);
}
inline LowCtx two_low(const Space* S) { return LowCtx{S->d_low, S->low_dim, S->dim, S->npar}; }

template <int M, typename Z>
static int two_product(const Space* S, const Z* c, const double2* X, Z* psi, int stop_check, const SilState* st,
                       hipStream_t stream) {
    k_pair_product<M, Z><<<div_up(S->low_dim, kTwoBlock), kTwoBlock, two_table_bytes(S), stream>>>(
        two_low(S), c, X, S->d_W, S->ldw, two_ld(S), stop_check, st, psi);
    MCTDHB_HIP_CHECK(hipGetLastError());
    return kOk;
}

template <int M, typename Z, typename Epi>
static int two_collect(const Space* S, const Z* c, const Z* psi, int stop_check, const SilState* st, Epi epi,
                       hipStream_t stream) {
    k_pair_collect<M, Z, Epi><<<div_up(S->dim, kTwoBlock), kTwoBlock, kRedBytes + two_table_bytes(S), stream>>>(
        row_ctx(S), S->low_dim, c, psi, two_ld(S), S->d_W, S->ldw, stop_check, st, epi);
    MCTDHB_HIP_CHECK(hipGetLastError());
    return kOk;
}

template <int M>
int HcTwoRows<M>::plain(const Space* S, const void* c, const double2* X, void* psi, void* out, int prec, hipStream_t st) {
    int rc;
    if (prec == kPrecFP64) {
        if ((rc = two_product<M>(S, (const double2*) c, X, (double2*) psi, 0, nullptr, st))) return rc;
        return two_collect<M>(S, (const double2*) c, (const double2*) psi, 0, nullptr,
                              EpiPlain<double2>{(double2*) out}, st);
    }
    if ((rc = two_product<M>(S, (const float2*) c, X, (float2*) psi, 0, nullptr, st))) return rc;
    return two_collect<M>(S, (const float2*) c, (const float2*) psi, 0, nullptr, EpiPlain<float2>{(float2*) out}, st);
}

template <int M>
int HcTwo<M>::rayleigh(const Space* S, const double2* X, const LanczosHcArgs& a, int prec, hipStream_t st) {
    const unsigned nb = two_rayleigh_blocks(S);
    double* part = a.part + (size_t) 2 * a.it * nb;  // slot 2 it
    if (prec == kPrecFP64)
        k_pair_rayleigh<M, double2><<<nb, kTwoBlock, two_table_bytes(S), st>>>(
            two_low(S), (const double2*) a.w[a.it], X, S->d_W, S->ldw, 1, a.st, part);
    else
        k_pair_rayleigh<M, float2><<<nb, kTwoBlock, two_table_bytes(S), st>>>(
            two_low(S), (const float2*) a.w[a.it], X, S->d_W, S->ldw, 1, a.st, part);
    MCTDHB_HIP_CHECK(hipGetLastError());
    return kOk;
}

template <int M>
int HcTwoRows<M>::lanczos(const Space* S, const double2* X, void* psi, const LanczosHcArgs& a, int prec, hipStream_t st) {
    int rc;
    if (prec == kPrecFP64) {
        const double2* w = (const double2*) a.w[a.it];
        if ((rc = two_product<M>(S, w, X, (double2*) psi, 1, a.st, st))) return rc;
        return two_collect<M>(S, w, (const double2*) psi, 1, a.st, EpiLanczos<double2>{a}, st);
    }
    const float2* w = (const float2*) a.w[a.it];
    if ((rc = two_product<M>(S, w, X, (float2*) psi, 1, a.st, st))) return rc;
    return two_collect<M>(S, w, (const float2*) psi, 1, a.st, EpiLanczos<float2>{a}, st);
}

}  // namespace mctdhb
