// sil_small.hpp - the whole SIL step in one workgroup, for spaces small
// enough that the multi-kernel step is a chain of launches whose work is a
// few microseconds each (the ground states of the reference's own example
// problems: NC in the hundreds or thousands).
//
// The recursion is the one of lanczos.hip (reference
// multiconfig_lanczos.c:11-90 and coefficients_integration.c:59-160) with
// the same unnormalised vectors and the same scalar updates
// (sil_device.hpp); the block does every pass in turn with barriers in
// between: H w_it in the two stages of hamiltonian_two.hpp, the dot products
// as block reductions, the reorthogonalisation pass, the tridiagonal
// exponential on wave 0 and the recombination.  FP64 only.
//
// The two stages pay here at every orbital count (their values stay in LDS or
// in the L2 cache): a row takes P values instead of 55 (M = 4) to 504 (M = 7)
// gathers from LDS, whose bandwidth bound the one-stage form together with
// its rank arithmetic.  Whole FP64 steps of 5 vectors, one stage -> two (us):
// NC 126, M = 5: 93 -> 48; NC 495: 102 -> 72; NC 7315: 1220 -> 721; NC 462,
// M = 6: 145 -> 75; NC 462, M = 7: 238 -> 102; NC 3003: 1006 -> 528; M = 4,
// NC 165: 66 -> 45 and 5456: 351 -> 356 (12 vectors: 1082 -> 1034).  Large
// spaces are bound by one CU's FP64 rate and its path to the L2 cache (psi),
// small ones by the chain of barriers and one-wave updates.
#pragma once

#include "hamiltonian_two.hpp"
#include "pack.hpp"
#include "sil_device.hpp"

namespace mctdhb {

constexpr int kSmallSlots = 2 * kMaxLanczos + 2;  // d_k (2 per k) and one norm

// tot[t] = sum of acc[t] over the first nw waves for t < nv (nv, nw uniform):
// one pass of wave sums, then thread t adds the wave partials of slot t.
__device__ __forceinline__ void block_sum_slots(const double (&acc)[kSmallSlots], int nv, int nw, double* red,
                                                double* tot) {
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    if (wid < nw) {
#pragma unroll
        for (int t = 0; t < kSmallSlots; t++) {
            if (t < nv) {
                const double v = wave_sum(acc[t]);
                if (lane == 0) red[t * nw + wid] = v;
            }
        }
    }
    __syncthreads();
    if ((int) threadIdx.x < nv) {
        double v = 0;
        for (int w = 0; w < nw; w++) v += red[threadIdx.x * nw + w];
        tot[threadIdx.x] = v;
    }
    __syncthreads();
}

// Threads: a small space does not fill more; where psi or the vectors come
// from the L2 cache and the registers suffice (M <= 6), 16 waves hide more of
// its latency (NC 7315, M = 5: 773 us at 512, 721 at 1024; NC 2002, M = 6: 298
// and 278; M = 3 and 4 within 3 % either way).
template <int M> constexpr int small_block(int form) { return form == kSmallAll || M > 6 ? 512 : 1024; }

template <int M, int FORM>
__device__ __forceinline__ void sil_small_block(unsigned char* smem, const SmallSilCtx& c, const SmallSilArgs& a) {
    constexpr bool PSIL = FORM >= kSmallPsi, ALL = FORM == kSmallAll;
    constexpr int P = pair_count(M);
    const uint32_t n = c.row.dim, T = blockDim.x, nlow = c.low.dim;
    uint32_t* Wl;
    double* sql;
    two_tables<M>(smem, 0, c.W, c.ldw, c.row.npar, Wl, sql);
    unsigned char* lds_l = (unsigned char*) sql + ((sizeof(double) * (c.row.npar + 3) + 15) & ~15);
    SmallSilLds& L = *(SmallSilLds*) lds_l;
    // ALL: lm vectors of n entries; otherwise the one H acts on, which becomes
    // out and then w_{it+1} in place (a thread's own rows)
    double2* Ws = (double2*) (lds_l + sizeof(SmallSilLds));
    double2* psi = PSIL ? Ws + (size_t) n * (ALL ? a.lm : 1) : c.psi;  // P arrays of ld entries
    const size_t ld = PSIL ? nlow : c.ld;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, nwv = T >> 6;
    const int nwr = min((int) ((n + 63) / 64), nwv);  // waves that hold rows
    // the scalars live in LDS (the one-wave updates then make no global
    // round trips) and are copied to a.st once the eigensolve is done
    SilState* st = &L.state;
    for (uint32_t t = threadIdx.x; t < sizeof(SilState) / sizeof(double); t += T) ((double*) st)[t] = 0;
    for (uint32_t t = threadIdx.x; t < n; t += T) Ws[t] = ((const double2*) a.w[0])[t];
    __syncthreads();
    if (threadIdx.x == 0) {
        st->s[0] = 1.0;
        st->iter_done = a.lm;
#pragma unroll
        for (int k = 0; k < kMaxLanczos; k++) L.w[k] = (double2*) a.w[k];  // constant indices: no private copy
    }
    __syncthreads();
    auto vec = [&](int k) -> double2* {
        if constexpr (ALL) return Ws + (size_t) k * n;
        else return L.w[k];
    };
    // the vectors' addresses in scalar registers, ahead of a pass over rows
    // (a store to LDS in it would have them read again for every row)
    typedef const __attribute__((address_space(1))) double2* GlobalVec;
    GlobalVec wp[kMaxLanczos];
    auto fetch = [&] {
        if constexpr (!ALL) {
#pragma unroll
            for (int k = 0; k < kMaxLanczos; k++) {
                const uint64_t p = (uint64_t) L.w[k];
                const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t) p);
                const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t) (p >> 32));
                wp[k] = (GlobalVec) ((uint64_t) hi << 32 | lo);
            }
        }
    };
    // rows i0, i0 + T, ... of w_k; past the end the last row (R of them in
    // flight: NC 1820, M = 5: 203 us at 1, 198 at 2, 223 at 4 with its spills)
    constexpr int R = ALL ? 1 : M > 6 ? 4 : 2;
    auto row_at = [&](uint32_t i0, int r) { return min(i0 + r * T, n - 1); };
    auto load = [&](double2 (&w)[R], int k, uint32_t i0) {
#pragma unroll
        for (int r = 0; r < R; r++) {
            const uint32_t i = row_at(i0, r);
            if constexpr (ALL) w[r] = Ws[(size_t) k * n + i];
            else w[r] = make_double2(wp[k][i].x, wp[k][i].y);
        }
    };
    // chunks of 64 configurations of N - 2 particles to waves; with fewer of
    // them than waves several waves share one and take its rows of X in turn
    const int nchunk = (int) ((nlow + 63) / 64), groups = nchunk && nchunk < nwv ? nwv / nchunk : 1;
    const int cstep = groups == 1 ? nwv : nchunk, grp = wid / cstep;
    // row i of H w: the sum of psi over pairs
    auto collect = [&](uint32_t i, const double2* src) {
        double2 row = make_double2(0, 0);
        if (nlow == 0) {  // N = 1: H is h itself, rank k the particle in orbital k
            for (int l = 0; l < M; l++) row = cfma(c.X[i * M + l], src[l], row);
            return row;
        }
        HighRow<M> x;
        x.set(i, c.row, nlow, 0, Wl, c.ldw, sql);
#pragma unroll
        for (int p = 0; p < P; p++) {
            const int k = kPairTable<M>.q[p], s = kPairTable<M>.l[p];
            // an empty orbital: any entry, times a zero root
            const uint32_t gone = k == s ? x.gone2[k] : x.gone1[k] | x.gone1[s];
            const double2 v = psi[p * ld + ((x.from[k] + x.to[s]) & ~gone)];
            const double f = x.r0[k] * (k == s ? x.rm[k] : x.r0[s]);
            row.x = fma(f, v.x, row.x);
            row.y = fma(f, v.y, row.y);
        }
        return row;
    };
    double acc[kSmallSlots];
    for (int it = 0; it < a.lm; it++) {
        const double2* src = ALL ? vec(it) : Ws;
        const double sit = st->s[it], bprev = it > 0 ? st->beta[it - 1] * st->s[it - 1] : 0.0;
        if (it == a.lm - 1) {
            // <w_it, H w_it> alone
            double e = 0;
            if (nlow == 0 && threadIdx.x < n) {
                const double2 h = collect(threadIdx.x, src);
                e = src[threadIdx.x].x * h.x + src[threadIdx.x].y * h.y;
            }
            for (int ch = wid % cstep; grp < groups && ch < nchunk; ch += cstep) {
                const uint32_t i = ch * 64 + lane;
                double2 phi[P];
                pair_states<M, double2>(phi, c.low.rows[min(i, nlow - 1)], c.low.top, src, Wl, c.ldw, sql);
                double part = 0;
#pragma unroll
                for (int x = 0; x < P; x++) {
                    if (x % groups != grp) continue;
                    double2 v = cscale(phi[x], 0.5 * c.X[x * P + x].x);
#pragma unroll
                    for (int y = x + 1; y < P; y++) v = cfma(c.X[x * P + y], phi[y], v);
                    part += phi[x].x * v.x + phi[x].y * v.y;
                }
                if (i < nlow) e += 2.0 * part;
            }
            e = wave_sum(e);
            if (lane == 0) L.red[wid] = e;
            __syncthreads();
            if (threadIdx.x < 64) {
                if (threadIdx.x == 0) {
                    double v = 0;
                    for (int w = 0; w < nwv; w++) v += L.red[w];
                    L.tot[2 * it] = v;
                }
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                __builtin_amdgcn_wave_barrier();
                sil_after_hc(st, L.tot, it, 2, threadIdx.x);
            }
            __syncthreads();
            break;
        }
        for (int ch = wid % cstep; grp < groups && ch < nchunk; ch += cstep) {
            const uint32_t i = ch * 64 + lane;
            double2 phi[P];
            pair_states<M, double2>(phi, c.low.rows[min(i, nlow - 1)], c.low.top, src, Wl, c.ldw, sql);
#pragma unroll 1
            for (int x = grp; x < P; x += groups) {
                double2 v = make_double2(0, 0);
#pragma unroll
                for (int y = 0; y < P; y++) v = cfma(c.X[x * P + y], phi[y], v);
                if (i < nlow) psi[x * ld + i] = v;
            }
        }
        __syncthreads();
        // out = s_it H w_it - beta_{it-1} s_{it-1} w_{it-1}, with the sums of
        // conj(w_k) out (k <= it) and, on the first pass, |w_0|^2
        double2* const wn = ALL ? vec(it + 1) : Ws;
        double2 one = make_double2(0, 0);
        if (nlow == 0) {  // N = 1 reads all of src first
            if (threadIdx.x < n) one = collect(threadIdx.x, src);
            __syncthreads();
        }
        for (uint32_t i = threadIdx.x; i < n; i += T) wn[i] = cscale(nlow ? collect(i, src) : one, sit);
        // A pass of its own: the sums' registers and a row's do not meet, and
        // R rows at a time keep R loads of a vector in flight.
#pragma unroll
        for (int t = 0; t < kSmallSlots; t++) acc[t] = 0;
        fetch();
        const double2* const wprev = it > 0 ? vec(it - 1) : nullptr;
        for (uint32_t i0 = threadIdx.x; i0 < n; i0 += R * T) {
            double2 o[R], w[R];
#pragma unroll
            for (int r = 0; r < R; r++) o[r] = wn[row_at(i0, r)];
            if (it > 0) {
#pragma unroll
                for (int r = 0; r < R; r++) w[r] = wprev[row_at(i0, r)];
#pragma unroll
                for (int r = 0; r < R; r++) o[r] = o[r] - cscale(w[r], bprev);
            }
#pragma unroll
            for (int r = 0; r < R; r++) {
                if (i0 + r * T < n) wn[i0 + r * T] = o[r];
                else o[r] = make_double2(0, 0);
            }
#pragma unroll
            for (int k = 0; k < kMaxLanczos; k++) {
                if (k <= it) {
                    load(w, k, i0);
#pragma unroll
                    for (int r = 0; r < R; r++) {
                        const double2 p = cconjmul(w[r], o[r]);
                        acc[2 * k] += p.x;
                        acc[2 * k + 1] += p.y;
                        if (k == 0 && it == 0 && i0 + r * T < n) acc[2] += w[r].x * w[r].x + w[r].y * w[r].y;
                    }
                }
            }
        }
        block_sum_slots(acc, 2 * (it + 1) + 1, nwr, L.red, L.tot);
        if (threadIdx.x < 64) {
            const int k = threadIdx.x;
            if (k <= it) {  // d_k = s_k <w_k, out>
                L.tot[2 * k] *= st->s[k];
                L.tot[2 * k + 1] *= st->s[k];
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            sil_after_hc(st, L.tot, it, 0, k);
        }
        __syncthreads();
        // w_{it+1} = out - sum_k cre_k w_k, with <w_k, w_{it+1}> and |w_{it+1}|^2
#pragma unroll
        for (int t = 0; t < kSmallSlots; t++) acc[t] = 0;
        double nrm = 0;
        double2* const wnew = ALL ? nullptr : L.w[it + 1];
        for (uint32_t i0 = threadIdx.x; i0 < n; i0 += R * T) {
            double2 o[R], w[R];
#pragma unroll
            for (int r = 0; r < R; r++) o[r] = wn[row_at(i0, r)];
#pragma unroll
            for (int k = 0; k < kMaxLanczos; k++) {
                if (k <= it) {
                    load(w, k, i0);
#pragma unroll
                    for (int r = 0; r < R; r++) o[r] = o[r] - cmul(st->cre[k], w[r]);
                }
            }
#pragma unroll
            for (int r = 0; r < R; r++) {
                if (i0 + r * T < n) {
                    wn[i0 + r * T] = o[r];
                    if constexpr (!ALL) wnew[i0 + r * T] = o[r];
                } else {
                    o[r] = make_double2(0, 0);
                }
                nrm += o[r].x * o[r].x + o[r].y * o[r].y;
            }
#pragma unroll
            for (int k = 0; k < kMaxLanczos; k++) {
                if (k <= it) {
                    load(w, k, i0);
#pragma unroll
                    for (int r = 0; r < R; r++) {
                        const double2 p = cconjmul(w[r], o[r]);
                        acc[2 * k] += p.x;
                        acc[2 * k + 1] += p.y;
                    }
                }
            }
        }
#pragma unroll
        for (int t = 0; t < kSmallSlots; t++)  // slot 2 (it + 1), by constant indices
            if (t == 2 * (it + 1)) acc[t] = nrm;
        block_sum_slots(acc, 2 * (it + 1) + 1, nwr, L.red, L.tot);
        if (threadIdx.x < 64) sil_after_reorth(st, L.tot, it, threadIdx.x);
        __syncthreads();
        if (st->stop) break;
    }
    // exp(-i T prop_dt) e_1 on wave 0, then C' = sum_k y_k w_k
    if (threadIdx.x < 64) sil_tridiag_wave(st, a.dt_re, a.dt_im, L.z, kMaxLanczos + 2, a.imagtime);
    __syncthreads();
    for (uint32_t t = threadIdx.x; t < sizeof(SilState) / sizeof(double); t += T)
        ((double*) a.st)[t] = ((const double*) st)[t];
    if (st->eig_fail) return;
    const int nd = st->iter_done;
    double2* C = L.w[0];
#pragma unroll
    for (int t = 0; t < kSmallSlots; t++) acc[t] = 0;
    fetch();
    for (uint32_t i0 = threadIdx.x; i0 < n; i0 += R * T) {
        double2 v[R], w[R];
        load(w, 0, i0);
#pragma unroll
        for (int r = 0; r < R; r++) v[r] = cmul(st->y[0], w[r]);
#pragma unroll
        for (int k = 1; k < kMaxLanczos; k++) {
            if (k < nd) {
                load(w, k, i0);
#pragma unroll
                for (int r = 0; r < R; r++) v[r] = v[r] + cmul(st->y[k], w[r]);
            }
        }
#pragma unroll
        for (int r = 0; r < R; r++) {
            if (i0 + r * T >= n) continue;
            if (a.imagtime) Ws[i0 + r * T] = v[r];
            else C[i0 + r * T] = v[r];
            acc[0] += v[r].x * v[r].x + v[r].y * v[r].y;
        }
    }
    if (a.imagtime) {  // renormalise (coefficients_integration.c:147-158)
        block_sum_slots(acc, 1, nwr, L.red, L.tot);
        const double sc = 1.0 / sqrt(L.tot[0]);
        for (uint32_t i = threadIdx.x; i < n; i += T) C[i] = cscale(Ws[i], sc);
    }
}

template <int M, int FORM>
__global__ __launch_bounds__(small_block<M>(FORM)) void k_sil_small(SmallSilCtx c, SmallSilArgs a) {
    extern __shared__ __align__(16) unsigned char smem[];
    sil_small_block<M, FORM>(smem, c, a);
}

// Packed form: one workgroup per instance.
template <int M, int FORM>
__global__ __launch_bounds__(small_block<M>(FORM)) void k_sil_small_pk(const PkSil* __restrict__ tab) {
    extern __shared__ __align__(16) unsigned char smem[];
    const PkSil& p = tab[blockIdx.x];
    sil_small_block<M, FORM>(smem, p.c, p.a);
}

template <int M> int HcTwo<M>::small(const Space* S, const double2* X, double2* psi, const SmallSilArgs& a,
                                     hipStream_t st) {
    if (!sil_small_fits(S, a.lm)) {
        set_error("space too large for the one-workgroup SIL step");
        return kInvalidArgument;
    }
    const SmallSilCtx c = small_ctx(S, X, psi);
    const int form = sil_small_form(S, a.lm), T = small_block<M>(form);
    const size_t smem = sil_small_lds(S, a.lm, form);
    switch (form) {
        case kSmallStaged: k_sil_small<M, kSmallStaged><<<1, T, smem, st>>>(c, a); break;
        case kSmallPsi: k_sil_small<M, kSmallPsi><<<1, T, smem, st>>>(c, a); break;
        default: k_sil_small<M, kSmallAll><<<1, T, smem, st>>>(c, a); break;
    }
    MCTDHB_HIP_CHECK(hipGetLastError());
    return kOk;
}

template <int M> int HcTwo<M>::small_pk(const PkSil* tab, int count, int form, size_t smem, hipStream_t st) {
    const int T = small_block<M>(form);
    switch (form) {
        case kSmallStaged: k_sil_small_pk<M, kSmallStaged><<<count, T, smem, st>>>(tab); break;
        case kSmallPsi: k_sil_small_pk<M, kSmallPsi><<<count, T, smem, st>>>(tab); break;
        default: k_sil_small_pk<M, kSmallAll><<<count, T, smem, st>>>(tab); break;
    }
    MCTDHB_HIP_CHECK(hipGetLastError());
    return kOk;
}

}  // namespace mctdhb
