// density.hip - one- and two-body density matrices on the device.
//
// Replaces reference src/configurational/density_matrices.c:8-443
// (set_onebody_dm, set_twobody_dm).  The reference runs one OpenMP
// reduction over all configurations per unique element (~155 sweeps at
// M = 5).  For 2 <= M <= 7 both matrices come from one pass over the space of
// N - 2 particles (density_impl.hpp); a deterministic second stage sums the
// per-block partials and fills rho1 and rho2.
//
// Other orbital counts take the generic kernel, one element at a time over
// the jump tables (e = layout index, see DmLayout):
//   D1[k]    = sum |c|^2 n_k                        -> rho1[k][k]
//   D2[k]    = sum |c|^2 n_k (n_k - 1)              -> rho2[kkkk]          (Rule 1)
//   D3[k<s]  = sum |c|^2 n_k n_s                    -> rho2[ksks] & perms  (Rule 2)
//   pair (k<l), t = conj(c_i) c[i-e_k+e_l] sqrt(n_k (n_l+1)):
//     T0 = sum t                                    -> rho1[k][l]
//     T_m = sum n_m t                               -> rho2[kkkl] = T_k - T0 (Rule 4),
//                                                      rho2[klll] = T_l (Rule 5),
//                                                      rho2[kssl] = T_s (Rule 7)
//   O3 (k<q)      = sum conj(c_i) c[i-2e_k+2e_q] sqrt((n_k-1) n_k (n_q+1)(n_q+2))   (Rule 3)
//   O6 (k; q<l)   = sum conj(c_i) c[i-2e_k+e_q+e_l] sqrt(n_k (n_k-1)(n_q+1)(n_l+1)) (Rule 6)
//   T8 (k<s; q<l) = sum conj(c_i) c[i-e_k-e_s+e_q+e_l] sqrt(n_k n_s (n_q+1)(n_l+1)) (Rule 8)
// and the reference's symmetric fill assembles rho1 (M x M) and rho2 (M^4,
// element k + sM + qM^2 + lM^3 = <a+_k a+_s a_q a_l>).
#include <algorithm>
#include <vector>

#include "density_impl.hpp"
#include "orbital.hpp"
#include "rowctx.hpp"

namespace mctdhb {

constexpr int kDmBlock = 256;
constexpr int kDmCPT = 16;  // configurations per thread per tile (generic kernel)
constexpr int kDmTile = kDmBlock * kDmCPT;

// ---------------------------------------------------------------- layout
__host__ __device__ constexpr int c2(int m) { return m * (m - 1) / 2; }
struct DmLayout {
    int M;
    __host__ __device__ constexpr int d1() const { return 0; }
    __host__ __device__ constexpr int d2() const { return M; }
    __host__ __device__ constexpr int d3() const { return 2 * M; }
    __host__ __device__ constexpr int pair() const { return 2 * M + c2(M); }
    __host__ __device__ constexpr int o3() const { return pair() + c2(M) * (M + 1); }
    __host__ __device__ constexpr int o6() const { return o3() + c2(M); }
    __host__ __device__ constexpr int t8() const { return o6() + M * c2(M - 1); }
    __host__ __device__ constexpr int total() const { return t8() + c2(M) * c2(M > 2 ? M - 2 : 0); }
    // lexicographic index of the pair a < b among 0..M-1
    __host__ __device__ constexpr int pidx(int a, int b) const { return a * M - a * (a + 1) / 2 + (b - a - 1); }
    // index of the pair q < l among the orbitals other than x (lexicographic)
    __host__ __device__ constexpr int pidx_excl1(int x, int q, int l) const {
        const int qq = q - (q > x), ll = l - (l > x);
        const int m = M - 1;
        return qq * m - qq * (qq + 1) / 2 + (ll - qq - 1);
    }
    __host__ __device__ constexpr int pidx_excl2(int x, int y, int q, int l) const {
        const int qq = q - (q > x) - (q > y), ll = l - (l > x) - (l > y);
        const int m = M - 2;
        return qq * m - qq * (qq + 1) / 2 + (ll - qq - 1);
    }
};

// -------------------------------------------------- generic (any M, FP64)
// One block per (tile, element); the element is described at run time.
struct ElemDesc {
    int type;  // 0 d1, 1 d2, 2 d3, 3 pair T0, 4 pair Tm, 5 o3, 6 o6, 7 t8
    int k, s, q, l, m;
};

static std::vector<ElemDesc> element_list(int M) {
    DmLayout L{M};
    std::vector<ElemDesc> v(L.total());
    for (int k = 0; k < M; k++) {
        v[L.d1() + k] = {0, k, 0, 0, 0, 0};
        v[L.d2() + k] = {1, k, 0, 0, 0, 0};
    }
    for (int k = 0; k < M; k++)
        for (int s = k + 1; s < M; s++) {
            v[L.d3() + L.pidx(k, s)] = {2, k, s, 0, 0, 0};
            const int o = L.pair() + L.pidx(k, s) * (M + 1);
            v[o] = {3, k, 0, 0, s, 0};
            for (int m = 0; m < M; m++) v[o + 1 + m] = {4, k, 0, 0, s, m};
            v[L.o3() + L.pidx(k, s)] = {5, k, 0, s, s, 0};
        }
    for (int k = 0; k < M; k++)
        for (int q = 0; q < M; q++)
            for (int l = q + 1; l < M; l++)
                if (q != k && l != k) v[L.o6() + k * c2(M - 1) + L.pidx_excl1(k, q, l)] = {6, k, 0, q, l, 0};
    for (int k = 0; k < M; k++)
        for (int s = k + 1; s < M; s++)
            for (int q = 0; q < M; q++)
                for (int l = q + 1; l < M; l++)
                    if (q != k && q != s && l != k && l != s)
                        v[L.t8() + L.pidx(k, s) * c2(M - 2) + L.pidx_excl2(k, s, q, l)] = {7, k, s, q, l, 0};
    return v;
}

__global__ __launch_bounds__(kDmBlock) void k_density_generic(int M, RowCtx ctx, const double2* __restrict__ c,
                                                              const ElemDesc* __restrict__ elems, int E,
                                                              double2* __restrict__ part) {
    __shared__ double red[2 * (kDmBlock / 64)];
    const ElemDesc d = elems[blockIdx.y];
    const uint32_t base = blockIdx.x * kDmTile;
    const uint32_t M2 = M * M;
    double2 acc = make_double2(0, 0);
    for (int r = 0; r < kDmCPT; r++) {
        const uint32_t i = base + threadIdx.x + r * kDmBlock;
        if (i >= ctx.dim) break;
        uint16_t occ[kMaxOrb];
        for (int k = 0; k < M; k++) occ[k] = ctx.ht[(size_t) i * M + k];
        const double2 ci = c[i];
        const double w = ci.x * ci.x + ci.y * ci.y;
        auto otc = [&](int k) {
            uint32_t cnt = 0;
            for (int h = 0; h < k; h++) cnt += occ[h] > 1;
            return cnt;
        };
        auto ttc = [&](int k, int s) {
            uint32_t cnt = 0;
            for (int h = 0; h < k; h++)
                for (int g = h + 1; g < M; g++) cnt += (occ[h] > 0 && occ[g] > 0);
            for (int g = k + 1; g < s; g++) cnt += occ[g] > 0;
            return cnt;
        };
        const int k = d.k;
        switch (d.type) {
            case 0: acc.x += w * occ[k]; break;
            case 1: acc.x += w * (double) (occ[k] * (occ[k] - 1)); break;
            case 2: acc.x += w * (double) (occ[k] * occ[d.s]); break;
            case 3:
            case 4:
                if (occ[k] >= 1) {
                    const uint32_t j = ctx.map[i + k * ctx.dim + d.l * M * ctx.dim];
                    double2 t = cscale(cconjmul(ci, c[j]), sqrt((double) occ[k] * (occ[d.l] + 1)));
                    if (d.type == 4) t = cscale(t, (double) occ[d.m]);
                    acc = acc + t;
                }
                break;
            case 5:
                if (occ[k] >= 2) {
                    const uint32_t j = ctx.mapot[ctx.sot[i] + otc(k) * M2 + d.q + d.q * M];
                    acc = acc + cscale(cconjmul(ci, c[j]),
                                       sqrt((double) (occ[k] - 1) * occ[k] * (occ[d.q] + 1) * (occ[d.q] + 2)));
                }
                break;
            case 6:
                if (occ[k] >= 2) {
                    const uint32_t j = ctx.mapot[ctx.sot[i] + otc(k) * M2 + d.q + d.l * M];
                    acc = acc + cscale(cconjmul(ci, c[j]),
                                       sqrt((double) occ[k] * (occ[k] - 1) * (occ[d.q] + 1) * (occ[d.l] + 1)));
                }
                break;
            case 7:
                if (occ[k] >= 1 && occ[d.s] >= 1) {
                    const uint32_t j = ctx.maptt[ctx.stt[i] + ttc(k, d.s) * M2 + d.q + d.l * M];
                    acc = acc + cscale(cconjmul(ci, c[j]),
                                       sqrt((double) occ[k] * occ[d.s] * (occ[d.q] + 1) * (occ[d.l] + 1)));
                }
                break;
        }
    }
    double v[2] = {acc.x, acc.y};
    block_sum<2>(v, red);
    if (threadIdx.x == 0) part[(size_t) blockIdx.x * E + blockIdx.y] = make_double2(v[0], v[1]);
}

// ------------------------------------- generic second stage and fill

__global__ __launch_bounds__(256) void k_generic_reduce(const double2* __restrict__ part, int nblocks, int E,
                                                        double2* __restrict__ tot) {
    __shared__ double red[2 * 4];
    const int e = blockIdx.x;
    double v[2] = {0, 0};
    for (int b = threadIdx.x; b < nblocks; b += blockDim.x) {
        const double2 p = part[(size_t) b * E + e];
        v[0] += p.x;
        v[1] += p.y;
    }
    block_sum<2>(v, red);
    if (threadIdx.x == 0) tot[e] = make_double2(v[0], v[1]);
}

__device__ __forceinline__ double2 dconj(double2 a) { return make_double2(a.x, -a.y); }

// Symmetric fill of reference density_matrices.c:23-50 and :76-442.  Every
// element of rho1 and rho2 is written exactly once, so the fill is spread
// over the threads of one block with no ordering: work item t is a diagonal
// index k (t < M), an orbital pair k < l (Rules 1-5, 7 and 3), a (k, q < l)
// triple of Rule 6 or a (k < s, q < l) quadruple of Rule 8.
__device__ __forceinline__ void dm_assemble_block(int M, const double2* __restrict__ tot, double2* __restrict__ rho1,
                                                  double2* __restrict__ rho2) {
    const DmLayout L{M};
    const int M2 = M * M, M3 = M2 * M, np = c2(M);
    auto R2 = [&](int a, int b, int cc, int d) -> double2& { return rho2[a + b * M + cc * M2 + d * M3]; };
    auto pair_of = [&](int p, int& a, int& b) {
        a = 0;
        while (p >= M - 1 - a) p -= M - 1 - a++;
        b = a + 1 + p;
    };
    const int n_diag = M, n_pair = np, n_r6 = rho2 ? M * np : 0, n_r8 = rho2 ? np * np : 0;
    for (int t = threadIdx.x; t < n_diag + n_pair + n_r6 + n_r8; t += blockDim.x) {
        if (t < n_diag) {
            const int k = t;
            rho1[k * M + k] = make_double2(tot[L.d1() + k].x, 0);
            if (rho2) R2(k, k, k, k) = make_double2(tot[L.d2() + k].x, 0);
        } else if (t < n_diag + n_pair) {
            const int p = t - n_diag;
            int k, l;
            pair_of(p, k, l);
            const double2* T = tot + L.pair() + p * (M + 1);
            rho1[k * M + l] = T[0];
            rho1[l * M + k] = dconj(T[0]);
            if (!rho2) continue;
            const double2 d3 = make_double2(tot[L.d3() + p].x, 0);  // Rule 2
            R2(k, l, k, l) = d3;
            R2(l, k, k, l) = d3;
            R2(l, k, l, k) = d3;
            R2(k, l, l, k) = d3;
            const double2 r4 = T[1 + k] - T[0];  // Rule 4
            R2(k, k, k, l) = r4;
            R2(k, k, l, k) = r4;
            R2(l, k, k, k) = dconj(r4);
            R2(k, l, k, k) = dconj(r4);
            const double2 r5 = T[1 + l];  // Rule 5
            R2(k, l, l, l) = r5;
            R2(l, k, l, l) = r5;
            R2(l, l, l, k) = dconj(r5);
            R2(l, l, k, l) = dconj(r5);
            for (int s = 0; s < M; s++) {  // Rule 7 (element k s s l)
                if (s == k || s == l) continue;
                const double2 r7 = T[1 + s];
                R2(k, s, s, l) = r7;
                R2(s, k, s, l) = r7;
                R2(s, k, l, s) = r7;
                R2(k, s, l, s) = r7;
                R2(l, s, s, k) = dconj(r7);
                R2(s, l, s, k) = dconj(r7);
                R2(s, l, k, s) = dconj(r7);
                R2(l, s, k, s) = dconj(r7);
            }
            const double2 r3 = tot[L.o3() + p];  // Rule 3 (k < q = l)
            R2(k, k, l, l) = r3;
            R2(l, l, k, k) = dconj(r3);
        } else if (t < n_diag + n_pair + n_r6) {  // Rule 6
            const int u = t - n_diag - n_pair, k = u / np;
            int q, l;
            pair_of(u % np, q, l);
            if (q == k || l == k) continue;
            const double2 r = tot[L.o6() + k * c2(M - 1) + L.pidx_excl1(k, q, l)];
            R2(k, k, q, l) = r;
            R2(k, k, l, q) = r;
            R2(l, q, k, k) = dconj(r);
            R2(q, l, k, k) = dconj(r);
        } else {  // Rule 8
            const int u = t - n_diag - n_pair - n_r6;
            int k, s, q, l;
            pair_of(u / np, k, s);
            pair_of(u % np, q, l);
            if (q == k || q == s || l == k || l == s) continue;
            const double2 r = tot[L.t8() + L.pidx(k, s) * c2(M - 2) + L.pidx_excl2(k, s, q, l)];
            R2(k, s, q, l) = r;
            R2(s, k, q, l) = r;
            R2(k, s, l, q) = r;
            R2(s, k, l, q) = r;
        }
    }
}

__global__ __launch_bounds__(256) void k_generic_assemble(int M, const double2* __restrict__ tot,
                                                     double2* __restrict__ rho1, double2* __restrict__ rho2) {
    dm_assemble_block(M, tot, rho1, rho2);
}

// ------------------------------------------- second stage of the pair sums

// Up to kDmFinishBlocks = 64 partials per element: one block sums them, a
// wave per element (one load per lane), and fills.
constexpr int kDmFinishThreads = 1024;
constexpr size_t dm_finish_lds(int M) { return sizeof(double2) * (gram_elements(M) + 4 * M * M); }

template <typename Z>
__device__ __forceinline__ void dm_finish_block(double2* lds, int M, int npar, const double2* __restrict__ part,
                                                int nb, const DmOut& out) {
    const int E = gram_elements(M), lane = threadIdx.x & 63;
    for (int e = threadIdx.x >> 6; e < E; e += blockDim.x >> 6) {
        const double2 p = lane < nb ? part[(size_t) e * nb + lane] : make_double2(0, 0);
        const double re = wave_sum(p.x), im = wave_sum(p.y);
        if (lane == 0) lds[e] = make_double2(re, im);
    }
    __syncthreads();
    dm_fill_block<Z>(M, npar, lds, out, lds + E);
}

template <typename Z>
__global__ __launch_bounds__(kDmFinishThreads) void k_dm_finish(int M, int npar, const double2* __restrict__ part,
                                                                int nb, DmOut out) {
    extern __shared__ double2 lds[];
    dm_finish_block<Z>(lds, M, npar, part, nb, out);
}

// Packed form: one block per instance.
__global__ __launch_bounds__(kDmFinishThreads) void k_dm_finish_pk(const PkDmFin* __restrict__ tab, int M) {
    extern __shared__ double2 lds[];
    const PkDmFin& a = tab[blockIdx.x];
    dm_finish_block<double2>(lds, M, a.npar, a.part, a.nb, a.out);
}

// More partials: one block per element sums them, and the last block to
// arrive fills.  Blocks count themselves in *arrive (a vector atomic), which
// k_gram has cleared: a count left over from calls that overlapped on one
// workspace spoils those calls only.  Each block writes one element before it
// counts, so the release it makes is cheap.
template <typename Z>
__global__ __launch_bounds__(256) void k_dm_reduce(int M, int npar, const double2* __restrict__ part, int nb,
                                                   double2* tot, unsigned* arrive, DmOut out) {
    extern __shared__ double2 lds[];
    __shared__ double red[2 * 4];
    __shared__ int last;
    const int e = blockIdx.x;
    double v[2] = {0, 0};
    for (int b = threadIdx.x; b < nb; b += blockDim.x) {
        const double2 p = part[(size_t) e * nb + b];
        v[0] += p.x;
        v[1] += p.y;
    }
    block_sum<2>(v, red);
    if (threadIdx.x == 0) {
        tot[e] = make_double2(v[0], v[1]);
        __threadfence();
        last = atomicAdd(arrive, 1u) == gridDim.x - 1;
    }
    __syncthreads();
    if (!last) return;
    __threadfence();
    for (int t = threadIdx.x; t < (int) gridDim.x; t += blockDim.x) lds[t] = tot[t];
    __syncthreads();
    dm_fill_block<Z>(M, npar, lds, out, lds + gridDim.x);
}

int pk_dm_finish(const PkDmFin* tab, int count, int M, hipStream_t st) {
    k_dm_finish_pk<<<count, kDmFinishThreads, dm_finish_lds(M), st>>>(tab, M);
    MCTDHB_HIP_CHECK(hipGetLastError());
    return kOk;
}

// instantiated once each in dm_m<M>.hip
extern template struct DmPairs<2>;
extern template struct DmPairs<3>;
extern template struct DmPairs<4>;
extern template struct DmPairs<5>;
extern template struct DmPairs<6>;
extern template struct DmPairs<7>;

int pk_density(const PkDm* tab, int count, int M, unsigned max_nb, size_t smem, hipStream_t st) {
    switch (M) {
        case 2: return DmPairs<2>::run_pk(tab, count, max_nb, smem, st);
        case 3: return DmPairs<3>::run_pk(tab, count, max_nb, smem, st);
        case 4: return DmPairs<4>::run_pk(tab, count, max_nb, smem, st);
        case 5: return DmPairs<5>::run_pk(tab, count, max_nb, smem, st);
        case 6: return DmPairs<6>::run_pk(tab, count, max_nb, smem, st);
        case 7: return DmPairs<7>::run_pk(tab, count, max_nb, smem, st);
        default: set_error("packed density kernels cover 2 <= norb <= 7"); return kInvalidArgument;
    }
}

static bool dm_generic(int M) { return M == 1 || M > 7; }

// Runs of configurations go to waves.  Up to 1024 configurations of N - 2
// particles one block of 8 waves does it all and the separate finish (a
// launch) is saved (1001 at M = 5: 13.2 us, two blocks 15.3; 1225 at M = 3:
// 13.8 in one block, 10.3 in several; at M = 6 several win earlier, 792: 29.0
// and 26.8).  Then 64 per wave, so a middling space still reaches many CUs.
// From 256 blocks on, one per CU (the LDS buffers of M >= 4 hold a CU each),
// the runs get longer: 128, 256 and 512 blocks take 272, 149 and 155 us at
// N=100, M=5, 282, 153 and 165 us at N=30, M=7 (complex64).
DmPlan dm_plan(const Space* S) {
    if (dm_generic(S->norb)) return {div_up(S->dim, kDmTile)};
    return {S->low_dim <= 1024 ? 1u : std::min(256u, div_up(S->low_dim, 64 * kDmWaves))};
}

// The rank and root tables leave room for what the block sums need; at M = 3
// this is what bounds N (7027).
constexpr size_t kDmTableBytes = 64 * 1024 - 9280;

bool dm_root_table(const Space* S) { return S->npar + 3 <= 2048; }

size_t dm_pair_smem(const Space* S) {
    const int M = S->norb;
    size_t tables = ((size_t) (M - 1) * S->ldw * 4 + 15) & ~(size_t) 15;
    if (dm_root_table(S)) tables += (sizeof(double) * (S->npar + 3) + 15) & ~(size_t) 15;
    if (tables > kDmTableBytes) return 0;
    size_t loop = 0, sums = 0;
    switch (M) {
#define CASE(m) \
    case m:                                                               \
        loop = gram_loop_lds<m>();                                          \
        sums = gram_sum_lds<m>() + sizeof(double2) * gram_elements(m);      \
        break;
        CASE(2) CASE(3) CASE(4) CASE(5) CASE(6) CASE(7)
#undef CASE
        default: return 0;
    }
    return std::max(tables + loop, sums);
}

// counter | totals | partials | element list (generic)
struct DmWork {
    unsigned* arrive;
    double2* tot;
    double2* part;
    ElemDesc* elems;
    size_t bytes;
};
static DmWork dm_work(const Space* S, void* base) {
    const int M = S->norb;
    const size_t nb = dm_plan(S).nb;
    const size_t E = dm_generic(M) ? (size_t) DmLayout{M}.total() : (size_t) gram_elements(M);
    char* p = (char*) base;
    DmWork w;
    w.arrive = (unsigned*) p;
    w.tot = (double2*) (p + 256);
    w.part = w.tot + E;
    w.elems = (ElemDesc*) (w.part + nb * E);
    w.bytes = 256 + sizeof(double2) * (nb + 1) * E + sizeof(ElemDesc) * E;
    return w;
}

static int dispatch_dm(const Space* S, const void* c, int prec, const DmWork& w, const DmPlan& plan, const DmOut& out,
                       hipStream_t st) {
    unsigned* arrive = plan.nb > kDmFinishBlocks ? w.arrive : nullptr;
    switch (S->norb) {
        case 2: return DmPairs<2>::run(S, c, prec, w.part, arrive, plan, out, st);
        case 3: return DmPairs<3>::run(S, c, prec, w.part, arrive, plan, out, st);
        case 4: return DmPairs<4>::run(S, c, prec, w.part, arrive, plan, out, st);
        case 5: return DmPairs<5>::run(S, c, prec, w.part, arrive, plan, out, st);
        case 6: return DmPairs<6>::run(S, c, prec, w.part, arrive, plan, out, st);
        case 7: return DmPairs<7>::run(S, c, prec, w.part, arrive, plan, out, st);
        default: set_error("pair density kernels cover 2 <= norb <= 7"); return kInvalidArgument;
    }
}

int dm_workspace_create(const Space* S, void** work) {
    MCTDHB_HIP_CHECK(hipMalloc(work, dm_work(S, nullptr).bytes));
    return kOk;
}

double2* dm_partials(const Space* S, void* work) { return dm_work(S, work).part; }

static int density_generic(const Space* S, const void* coef, double2* rho1, double2* rho2, const DmWork& w,
                           const DmSync& sy, hipStream_t st) {
    const int M = S->norb, E = DmLayout{M}.total();
    const unsigned nb = dm_plan(S).nb;
    std::vector<ElemDesc> el = element_list(M);
    MCTDHB_HIP_CHECK(hipMemcpyAsync(w.elems, el.data(), sizeof(ElemDesc) * E, hipMemcpyHostToDevice, st));
    RowCtx ctx = make_row_ctx(S->dim, S->npar, S->d_ht, S->d_map, S->d_mapot, S->d_maptt, S->d_strideot,
                              S->d_stridett);
    k_density_generic<<<dim3(nb, E), kDmBlock, 0, st>>>(M, ctx, (const double2*) coef, w.elems, E, w.part);
    MCTDHB_HIP_CHECK(hipGetLastError());
    // the host vector must outlive the async copy
    MCTDHB_HIP_CHECK(hipStreamSynchronize(st));
    k_generic_reduce<<<E, 256, 0, st>>>(w.part, (int) nb, E, w.tot);
    k_generic_assemble<<<1, 256, 0, st>>>(M, w.tot, rho1, rho2);
    MCTDHB_HIP_CHECK(hipGetLastError());
    return sy.rinv ? density_sync_small(M, rho1, sy.rinv, sy.eig, sy.reg, st) : kOk;
}

int density_matrices(const Space* S, const void* coef, double2* rho1, double2* rho2, int prec, int index,
                     void* work, hipStream_t st, const DmSync* sync) {
    if (sync && sync->rinv && S->norb > 30) {
        set_error("norb exceeds 30");
        return kInvalidArgument;
    }
    const int M = S->norb;
    const bool generic = dm_generic(M);
    if (prec == kDmMixed && generic) {
        set_error("mixed precision density matrices cover 2 <= norb <= 7");
        return kInvalidArgument;
    }
    if ((generic || index == kIdxTables) && !S->tables) {
        set_error("this density-matrix form needs the jump tables; build the space with tables");
        return kNotBuilt;
    }
    const DmSync sy = sync ? *sync : DmSync{nullptr, nullptr, 0.0};
    const DmWork w = dm_work(S, work);
    if (generic) return density_generic(S, coef, rho1, rho2, w, sy, st);
    const DmPlan plan = dm_plan(S);
    const DmOut out{coef, rho1, rho2, sy};
    const int rc = dispatch_dm(S, coef, prec, w, plan, out, st);
    if (rc || plan.nb == 1) return rc;
    const int nb = (int) plan.nb, E = gram_elements(M);
    const size_t smem = dm_finish_lds(M);
    if (plan.nb <= kDmFinishBlocks) {
        if (prec == kDmMixed) k_dm_finish<float2><<<1, kDmFinishThreads, smem, st>>>(M, S->npar, w.part, nb, out);
        else k_dm_finish<double2><<<1, kDmFinishThreads, smem, st>>>(M, S->npar, w.part, nb, out);
    } else {
        if (prec == kDmMixed)
            k_dm_reduce<float2><<<E, 256, smem, st>>>(M, S->npar, w.part, nb, w.tot, w.arrive, out);
        else
            k_dm_reduce<double2><<<E, 256, smem, st>>>(M, S->npar, w.part, nb, w.tot, w.arrive, out);
    }
    MCTDHB_HIP_CHECK(hipGetLastError());
    return kOk;
}

}  // namespace mctdhb
