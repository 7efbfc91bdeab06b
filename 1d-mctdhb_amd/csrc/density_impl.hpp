// density_impl.hpp - the pair-sum kernel of the density matrices,
// instantiated once per orbital count in dm_m<M>.hip.
//
// Gamma[a][b] = sum over n' of conj(phi_a(n')) phi_b(n') for the pairs
// a <= b (pairs.hpp) holds all of rho2, and rho1 is its partial trace over
// N - 1.  The sum is a product of the P x NC' matrix phi with its adjoint,
// taken on the FP64 matrix cores: lane (g, c) of a wave holds phi of pair c
// (and 16 + c for M >= 6) at the g-th of four configurations, which is the
// operand layout of both factors.
//
// Why this form: forming every element from the N space takes a gather and a
// product per jump (about 80 per configuration at M = 5, one sum per element
// on the vector ALU); here it is P = 15 gathers, and the sums are matrix
// work.  Measured on MI355X, whole call: N=100, M=5 in FP64 0.495 ms before,
// 0.149 ms now; N=30, M=7 from complex64 coefficients 1.81 ms before, 0.153 ms
// now.  What bounds it is the FP64 unit, which matrix and vector instructions
// share (run together they add up, they do not overlap): 3 products of
// 16 x 16 x 4 per four configurations (10 at M >= 6) are 0.083 and 0.087 ms at
// those sizes, the addressing and scaling about a third of that again.  Hence
// a lane forms its configuration's addresses once for all pairs; with one
// pair per lane (every lane ranking for itself, no LDS) the same loop took
// 0.205 ms at both sizes.
//
// Complex64 coefficients are widened when read: products and sums are FP64
// in both forms.
#pragma once

#include "density.hpp"
#include "mxm_wave.hpp"
#include "pack.hpp"

namespace mctdhb {

// Gamma[a][b], a <= b, of the totals tot (row by row over the upper triangle).
__device__ __forceinline__ double2 gamma_at(const double2* tot, int P, int a, int b) {
    const bool up = a <= b;
    const int i = up ? a : b, j = up ? b : a;
    const double2 v = tot[i * P - i * (i - 1) / 2 + (j - i)];
    return up ? v : make_double2(v.x, -v.y);
}

__device__ __forceinline__ int pair_of(int M, int a, int b) { return a <= b ? pair_index(M, a, b) : pair_index(M, b, a); }

// rho1 and rho2 from the pair sums (every entry written once), then with
// sy.rinv set the synchronisation of rho1.  One block; tot is in LDS and
// visible to it.  Wave 0 forms rho1, one element per lane, and inverts it in
// its registers while the other waves write rho2; the eigenvalues, or a rho1
// that may need regularisation, take the whole block (density_sync_body).
// N = 1 has no pairs: rho1 = conj(c_k) c_l, rho2 = 0.
template <typename Z>
__device__ __forceinline__ void dm_fill_block(int M, int npar, const double2* tot, const DmOut& o, double2* work) {
    const int M2 = M * M, P = M * (M + 1) / 2;
    __shared__ int done;
    if (threadIdx.x < 64) {
        const int k = threadIdx.x >> 3, l = threadIdx.x & 7;
        const bool in = k < M && l < M;
        double2 v = make_double2(0, 0);
        if (in && npar < 2) {
            const Z* c = (const Z*) o.c;
            v = cconjmul(to_d2(c[k]), to_d2(c[l]));
        } else if (in) {
            for (int s = 0; s < M; s++) v = v + gamma_at(tot, P, pair_of(M, k, s), pair_of(M, s, l));
            v = cscale(v, 1.0 / (npar - 1));
        }
        if (in) o.rho1[k * M + l] = v;
        bool ok = !o.sy.rinv;
        if (o.sy.rinv && !o.sy.eig) {
            if (k == l) v.y = 0;
            ok = hpd_inverse_wave(M, v, o.sy.reg);
            if (ok && in) o.sy.rinv[k * M + l] = v;
        }
        if (threadIdx.x == 0) done = ok;
    } else if (o.rho2) {
        for (int e = threadIdx.x - 64; e < M2 * M2; e += blockDim.x - 64) {
            const int k = e % M, s = (e / M) % M, q = (e / M2) % M, l = e / (M2 * M);
            o.rho2[e] = npar < 2 ? make_double2(0, 0) : gamma_at(tot, P, pair_of(M, k, s), pair_of(M, q, l));
        }
    }
    __syncthreads();
    if (!done) density_sync_body(M, o.rho1, o.sy.rinv, o.sy.eig, o.sy.reg, work);
}

// Accumulators of a wave: for M <= 5 one tile of 16 pairs, Re = S and
// Im = Q - Q^T with Q = Xr Xi^T; for M >= 6 two tiles, Re of (0,0), (0,1),
// (1,1), Q of (0,0) and (1,1), and Im of (0,1).
template <int M> struct GramAcc {
    static constexpr int T = pair_count(M) <= 16 ? 1 : 2;
    static constexpr int N = T == 1 ? 2 : 6;
    mat4 a[N];
    __device__ __forceinline__ void zero() {
#pragma unroll
        for (int t = 0; t < N; t++) a[t] = mat4{0, 0, 0, 0};
    }
    __device__ __forceinline__ void add(const double2 (&x)[T]) {
        if constexpr (T == 1) {
            a[0] = mma(x[0].x, x[0].x, a[0]);
            a[1] = mma(x[0].x, x[0].y, a[1]);
            a[0] = mma(x[0].y, x[0].y, a[0]);
        } else {
            a[0] = mma(x[0].x, x[0].x, a[0]);
            a[1] = mma(x[0].x, x[1].x, a[1]);
            a[2] = mma(x[1].x, x[1].x, a[2]);
            a[3] = mma(x[0].x, x[0].y, a[3]);
            a[4] = mma(x[1].x, x[1].y, a[4]);
            a[5] = mma(x[0].x, x[1].y, a[5]);
            a[0] = mma(x[0].y, x[0].y, a[0]);
            a[1] = mma(x[0].y, x[1].y, a[1]);
            a[2] = mma(x[1].y, x[1].y, a[2]);
            a[5] = mma(-x[0].y, x[1].x, a[5]);
        }
    }
};

// A wave works on 64 configurations at a time for M <= 5 (a lane forms all
// the pairs of its configuration) and on 32 for M >= 6 (lane i and lane
// i + 32 share one and take half of the pairs each).  The values go through
// the wave's own LDS buffer, row p the configurations of pair p, padded by
// one so that the 16 rows a matrix operand reads start in different banks.
template <int M> struct GramShape {
    static constexpr int P = pair_count(M);
    static constexpr int H = P <= 16 ? 1 : 2;
    static constexpr int C = 64 / H;         // configurations per pass
    static constexpr int S = (P + H - 1) / H;  // pairs per lane
    static constexpr int LD = C + 1;
    static constexpr size_t wave_bytes = sizeof(double2) * P * LD;
};

// Passes w0 .. w1, in a pipeline: while pass s is multiplied, the
// coefficients of s + 1 and the rows of s + 2 are on their way.  Reads past
// the end repeat the last row and count as zero.
template <int M, bool LUT, typename Z>
__device__ __forceinline__ void gram_loop(GramAcc<M>& acc, double2* __restrict__ buf, const LowCtx& low,
                                          const Z* __restrict__ c, const uint32_t* __restrict__ Wl, int ldw,
                                          const double* __restrict__ sql, uint32_t w0, uint32_t w1) {
    using G = GramShape<M>;
    constexpr int T = GramAcc<M>::T;
    if (w0 >= w1) return;
    const int lane = threadIdx.x & 63, col = lane & 15, grp = lane >> 4;
    const uint32_t mine = lane % G::C;
    const bool second = G::H == 2 && lane >= G::C;
    LowRow<M> x;
    Z v[G::S];
    uint32_t num[G::S];  // the numbers under the roots, 16 bits each
    // slot t of this lane is pair t, or S + t in the second half (pair P - 1 again past the end)
    auto gather = [&](uint64_t row) {
        x.set(row, Wl, ldw, low.top);
#pragma unroll
        for (int t = 0; t < G::S; t++) {
            constexpr int last = G::P - 1;
            const int p0 = t, p1 = G::S + t < G::P ? G::S + t : last;
            const int q0 = kPairTable<M>.q[p0], l0 = kPairTable<M>.l[p0];
            const int q1 = kPairTable<M>.q[p1], l1 = kPairTable<M>.l[p1];
            uint32_t j = x.from[q0] + x.to[l0];
            uint32_t a = (x.n[q0] + 1) | (x.n[l0] + 1 + (q0 == l0)) << 16;
            if (G::H == 2) {
                const uint32_t j1 = x.from[q1] + x.to[l1];
                const uint32_t a1 = (x.n[q1] + 1) | (x.n[l1] + 1 + (q1 == l1)) << 16;
                j = second ? j1 : j;
                a = second ? a1 : a;
            }
            num[t] = a;
            v[t] = c[j];
        }
    };
    auto fetch = [&](uint32_t s) { return low.rows[min(s * G::C + mine, low.dim - 1)]; };
    uint64_t next = fetch(w0 + 1);
    gather(fetch(w0));
    for (uint32_t s = w0; s < w1; s++) {
        const bool in = s * G::C + mine < low.dim;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();  // the previous pass has been read
#pragma unroll
        for (int t = 0; t < G::S; t++) {
            const uint32_t a = num[t] & 0xffffu, b = num[t] >> 16;
            const double f = LUT ? sql[a] * sql[b] : sqrt((double) a * (double) b);
            const int p = second ? (G::S + t < G::P ? G::S + t : G::P - 1) : t;
            buf[p * G::LD + mine] = cscale(to_d2(v[t]), in ? f : 0.0);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        const uint64_t row = next;
        next = fetch(s + 2);
        gather(row);
        // the loads stay on this side of the products (moved to where their
        // values are used, they would be waited for at once)
        asm volatile("" ::: "memory");
#pragma unroll 4
        for (int u = 0; u < G::C / 4; u++) {
            double2 o[T];
#pragma unroll
            for (int t = 0; t < T; t++) o[t] = buf[min(t * 16 + col, G::P - 1) * G::LD + 4 * u + grp];
            acc.add(o);
        }
    }
}

// Dynamic LDS: the tables and one buffer per wave in the loop; after it the
// waves' values of one accumulator and the block sums of all of them.
template <int M> constexpr size_t gram_loop_lds() { return kDmWaves * GramShape<M>::wave_bytes; }
template <int M> constexpr size_t gram_sum_lds() { return sizeof(double) * 256 * (kDmWaves + GramAcc<M>::N); }
constexpr int gram_elements(int M) { return pair_count(M) * (pair_count(M) + 1) / 2; }

// Block bid of nb: sums its share of the N - 2 space and leaves
// Gamma (upper triangle) in part[e * nb + bid].
template <int M, typename Z>
__device__ __forceinline__ void gram_block(unsigned char* smem, uint32_t bid, uint32_t nb, const LowCtx& low,
                                           const Z* __restrict__ c, const uint32_t* __restrict__ Wg, int ldw,
                                           int use_sq, double2* part) {
    using G = GramShape<M>;
    constexpr int P = G::P, T = GramAcc<M>::T;
    uint32_t* Wl = (uint32_t*) smem;
    const int wsz = (M - 1) * ldw;
    double* sql = (double*) (smem + ((wsz * 4 + 15) & ~15));
    for (int t = threadIdx.x; t < wsz; t += blockDim.x) Wl[t] = Wg[t];
    if (use_sq)
        for (int t = threadIdx.x; t < low.npar + 3; t += blockDim.x) sql[t] = sqrt((double) t);
    __syncthreads();
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, col = lane & 15, grp = lane >> 4;
    size_t off = (wsz * 4 + 15) & ~(size_t) 15;
    if (use_sq) off += (sizeof(double) * (low.npar + 3) + 15) & ~(size_t) 15;
    double2* buf = (double2*) (smem + off + wid * G::wave_bytes);
    GramAcc<M> acc;
    acc.zero();
    // passes of C configurations, a contiguous run of them per wave
    const uint32_t nsub = (low.dim + G::C - 1) / G::C, nw = nb * kDmWaves;
    const uint32_t per = (nsub + nw - 1) / nw, w0 = (bid * kDmWaves + wid) * per;
    const uint32_t w1 = min(w0 + per, nsub);
    if (use_sq) gram_loop<M, true>(acc, buf, low, c, Wl, ldw, sql, w0, w1);
    else gram_loop<M, false>(acc, buf, low, c, Wl, ldw, sql, w0, w1);
    // block sums in a fixed order
    double* wave = (double*) smem;           // [kDmWaves][256]
    double* sum = wave + 256 * kDmWaves;     // [accumulator][256]
    for (int t = 0; t < GramAcc<M>::N; t++) {
        __syncthreads();
        mat4 v = acc.a[0];
#pragma unroll
        for (int j = 1; j < GramAcc<M>::N; j++)
            if (j == t) v = acc.a[j];
#pragma unroll
        for (int i = 0; i < 4; i++) wave[wid * 256 + (4 * i + grp) * 16 + col] = v[i];
        __syncthreads();
        for (int e = threadIdx.x; e < 256; e += blockDim.x) {
            double v = wave[e];
#pragma unroll
            for (int w = 1; w < kDmWaves; w++) v += wave[w * 256 + e];
            sum[t * 256 + e] = v;
        }
    }
    __syncthreads();
    for (int e = threadIdx.x; e < P * P; e += blockDim.x) {
        const int a = e / P, b = e % P;
        if (a > b) continue;
        const int i = a & 15, j = b & 15;
        double re, im;
        if (T == 1 || b < 16) {
            re = sum[i * 16 + j];
            im = sum[(T == 1 ? 1 : 3) * 256 + i * 16 + j] - sum[(T == 1 ? 1 : 3) * 256 + j * 16 + i];
        } else if (a < 16) {
            re = sum[256 + i * 16 + j];
            im = sum[5 * 256 + i * 16 + j];
        } else {
            re = sum[2 * 256 + i * 16 + j];
            im = sum[4 * 256 + i * 16 + j] - sum[4 * 256 + j * 16 + i];
        }
        part[(size_t) (a * P - a * (a - 1) / 2 + (b - a)) * nb + bid] = make_double2(re, im);
    }
}

// One block (nb = 1) also fills rho1 and rho2 and synchronises rho1: its sums
// go to LDS behind those of the waves.  arrive (may be null): cleared for the
// last stage.
template <int M, typename Z>
__global__ __launch_bounds__(kDmThreads) void k_gram(LowCtx low, const Z* __restrict__ c,
                                                     const uint32_t* __restrict__ Wg, int ldw, int use_sq,
                                                     double2* part, unsigned* arrive, DmOut out) {
    extern __shared__ __align__(16) unsigned char smem[];
    double2* tot = (double2*) (smem + gram_sum_lds<M>());
    const bool one = gridDim.x == 1;
    if (arrive && blockIdx.x == 0 && threadIdx.x == 0) *arrive = 0;
    gram_block<M, Z>(smem, xcd_block(blockIdx.x, gridDim.x), gridDim.x, low, c, Wg, ldw, use_sq, one ? tot : part);
    if (one) {
        __syncthreads();
        dm_fill_block<Z>(M, low.npar, tot, out, (double2*) smem);
    }
}

// Packed form: instance blockIdx.y; blocks past its own count return.
template <int M> __global__ __launch_bounds__(kDmThreads) void k_gram_pk(const PkDm* __restrict__ tab) {
    extern __shared__ __align__(16) unsigned char smem[];
    const PkDm& p = tab[blockIdx.y];
    if (blockIdx.x >= p.nb) return;
    gram_block<M, double2>(smem, xcd_block(blockIdx.x, p.nb), p.nb, p.low, p.c, p.W, p.ldw, p.use_sq, p.part);
}

template <int M>
int DmPairs<M>::run_pk(const PkDm* tab, int count, unsigned max_nb, size_t smem, hipStream_t st) {
    k_gram_pk<M><<<dim3(max_nb, count), kDmThreads, smem, st>>>(tab);
    MCTDHB_HIP_CHECK(hipGetLastError());
    return kOk;
}

template <int M>
int DmPairs<M>::run(const Space* S, const void* c, int prec, double2* part, unsigned* arrive, const DmPlan& plan,
                    const DmOut& out, hipStream_t st) {
    const size_t smem = dm_pair_smem(S);
    if (!smem) {
        set_error("density kernel LDS budget exceeded for this (N, M)");
        return kInvalidArgument;
    }
    const int use_sq = dm_root_table(S) ? 1 : 0;
    if (prec == kDmMixed)
        k_gram<M, float2><<<plan.nb, kDmThreads, smem, st>>>(low_ctx(S), (const float2*) c, S->d_W, S->ldw, use_sq,
                                                             part, arrive, out);
    else
        k_gram<M, double2><<<plan.nb, kDmThreads, smem, st>>>(low_ctx(S), (const double2*) c, S->d_W, S->ldw, use_sq,
                                                              part, arrive, out);
    MCTDHB_HIP_CHECK(hipGetLastError());
    return kOk;
}

}  // namespace mctdhb
