// sil_device.hpp - the scalar part of the Lanczos / SIL recursion on the
// device: state initialisation, the updates after the H.C and the
// reorthogonalisation passes, the tridiagonal eigensolver and the
// exponential.  Shared by the multi-kernel step (lanczos.hip) and the
// one-workgroup step for small spaces (sil_small.hpp).
#pragma once

#include "common.hpp"
#include "sil.hpp"

namespace mctdhb {

constexpr double kBreakdownTol = 1e-14;  // reference multiconfig_lanczos.c:34

// Fresh scalars for an lm-vector recursion, by threads t of T.
__device__ inline void sil_init_state(SilState* st, int lm, int t, int T) {
    for (int k = t; k <= kMaxKrylov; k += T) {
        st->s[k] = k == 0 ? 1.0 : 0.0;
        st->beta[k] = 0;
        st->alpha[k] = make_double2(0, 0);
        st->cre[k] = make_double2(0, 0);
        st->gram[k] = make_double2(0, 0);
        st->y[k] = make_double2(0, 0);
    }
    if (t != 0) return;
    st->maxbeta = 0;
    st->nrm2 = 0;
    st->eground = 0;
    st->iter_done = lm;
    st->arrive = 0;
    st->stop = 0;
    st->eig_fail = 0;
}

// The scalar updates below run on one wave, lane k on vector k: the values a
// lane needs come in one round of loads.  (One thread looping over k waited
// for memory once per k; the launches that end in them went from 5.6 and 5.3 us to
// 4.8 and 4.6 us at N=200, M=4.)

// After the H.C pass of iteration it: alpha_it and the reorthogonalisation
// coefficients (on w_k) for the next streaming pass.
// On the last iteration only alpha is formed.  last == 2: the H.C pass
// summed <w_it, H w_it> (the half-row form), and alpha = <v_it, H v_it -
// beta v_{it-1}> = s_it^2 <w_it, H w_it> - beta conj(<v_{it-1}, v_it>).
__device__ __forceinline__ void sil_after_hc(SilState* st, const volatile double* tot, int it, int last, int k,
                                             double2* cre, bool keep) {
    if (k > it) return;
    const double2 t = make_double2(tot[2 * it], tot[2 * it + 1]), d = make_double2(tot[2 * k], tot[2 * k + 1]);
    const double nrm0 = it == 0 && !last ? tot[2] : 0.0;  // <v_0, v_0> = |C|^2
    double2 gk = st->gram[k];
    const double sk = st->s[k];
    if (it == 0) gk = make_double2(nrm0, 0);
    double2 alpha = t;
    if (last == 2) {
        const double s = st->s[it];
        alpha = make_double2(s * s * t.x, 0);
        if (it > 0) {
            const double2 gp = st->gram[it - 1];
            alpha = alpha - make_double2(st->beta[it - 1] * gp.x, -st->beta[it - 1] * gp.y);
        }
    }
    if (k == 0 && keep) {
        st->alpha[it] = alpha;
        if (it == 0) st->gram[0] = gk;
    }
    if (last) return;
    double2 ortho = d - cmul(alpha, gk);
    if (k == it) ortho = ortho + alpha;
    cre[k] = cscale(ortho, sk);
}

__device__ __forceinline__ void sil_after_hc(SilState* st, const volatile double* tot, int it, int last, int k) {
    sil_after_hc(st, tot, it, last, k, st->cre, true);
}

// After the streaming pass that produced w_{it+1}: beta_it, the breakdown
// test of the reference (beta / max beta < 1e-14 ends the recursion with
// it + 1 vectors) and the Gram column <v_k, v_{it+1}>.
__device__ __forceinline__ void sil_after_reorth(SilState* st, const volatile double* tot, int it, int k) {
    if (k > it + 1) return;
    const double nrm2 = tot[2 * (it + 1)];
    const double2 d = k <= it ? make_double2(tot[2 * k], tot[2 * k + 1]) : make_double2(nrm2, 0);
    const double sk = st->s[k], old = st->maxbeta;
    const double beta = sqrt(nrm2), maxbeta = old < beta ? beta : old;
    const bool stop = beta / maxbeta < kBreakdownTol;
    const double sn = 1.0 / beta;
    if (k == 0) {
        st->beta[it] = beta;
        st->maxbeta = maxbeta;
        if (stop) {
            st->iter_done = it + 1;
            st->stop = 1;
        } else {
            st->s[it + 1] = sn;
        }
    }
    if (!stop) st->gram[k] = k <= it ? cscale(d, sk * sn) : make_double2(nrm2 * sn * sn, 0);
}

// ------------------------------------------------ tridiagonal eigensolver
//
// Implicit-shift QL with Givens rotations (the EISPACK tql2 method) on one
// wave: lane r keeps d[r] and e[r] in registers and owns row r of the
// eigenvector matrix (in LDS), so each rotation updates all rows at once;
// the scalar recurrence runs redundantly in every lane on values broadcast
// with readlane.  n <= 64.
//
// One dependent chain of FP64 operations per rotation bounds it.  Hence one
// reciprocal square root per rotation in place of a root and a division, the
// search for a small off-diagonal entry as one comparison in all lanes and a
// ballot, and the eigenvector row carried from rotation to rotation in a
// register (one LDS read, off the chain, and one write).  With m = 8 vectors
// the launch took 36 us before, 23 us so; with m = 5 15.4 and 10.9 us.

__device__ __forceinline__ double rlane(double x, int i) {
    const int lo = __builtin_amdgcn_readlane(__double2loint(x), i);
    const int hi = __builtin_amdgcn_readlane(__double2hiint(x), i);
    return __hiloint2double(hi, lo);
}

// On return lane r holds eigenvalue d (unsorted) and zr[0..n) is row r of Z
// (eigenvector j in column j).  Returns non-zero if an eigenvalue needed
// more than 60 sweeps.
__device__ inline int tridiag_eig_wave(int n, double& d, double& e, double* zr) {
    const int lane = threadIdx.x & 63;
    for (int c = 0; c < n; c++) zr[c] = (lane == c) ? 1.0 : 0.0;
    if (lane == n - 1) e = 0.0;
    for (int l = 0; l < n - 1; l++) {
        int sweeps = 0;
        for (;;) {
            // the first m >= l whose off-diagonal entry is negligible
            const double scale = fabs(d) + fabs(__shfl_down(d, 1, 64));
            const bool small = lane >= n - 1 || fabs(e) <= 2.220446049250313e-16 * scale;
            const int m = l + __builtin_ctzll(__ballot(small) >> l);
            if (m == l) break;
            if (++sweeps > 60) return 1;
            const double dl = rlane(d, l), el = rlane(e, l);
            // |theta| <= 1 / (2 eps) after the test above and the entries
            // of T are far from overflow: plain square roots of sums of
            // squares in place of hypot
            const double theta = (rlane(d, l + 1) - dl) / (2.0 * el);
            const double rho = sqrt(theta * theta + 1.0);
            double dn = rlane(d, m);
            double g = dn - dl + el / (theta + (theta >= 0 ? rho : -rho));
            double sn = 1.0, cs = 1.0, shift = 0.0;
            double z1 = zr[m];
            bool early = false;
            for (int i = m - 1; i >= l; i--) {
                const double ei = rlane(e, i), di = rlane(d, i);
                const double z0 = zr[i];
                const double f = sn * ei, b = cs * ei;
                const double r2 = f * f + g * g;
                if (r2 == 0.0) {
                    if (lane == i + 1) {
                        e = 0.0;
                        d = dn - shift;
                    }
                    if (lane == m) e = 0.0;
                    zr[i + 1] = z1;
                    early = true;
                    break;
                }
                const double ir = rsqrt(r2);
                sn = f * ir;
                cs = g * ir;
                const double h = dn - shift;
                const double r = (di - h) * sn + 2.0 * cs * b;
                shift = sn * r;
                if (lane == i + 1) {
                    e = r2 * ir;
                    d = h + shift;
                }
                g = cs * r - b;
                dn = di;
                zr[i + 1] = sn * z0 + cs * z1;
                z1 = cs * z0 - sn * z1;
            }
            if (early) continue;
            zr[l] = z1;
            if (lane == l) {
                d = dn - shift;
                e = g;
            }
            if (lane == m) e = 0.0;
        }
    }
    return 0;
}

// exp(-i T prop_dt) e_1 from the eigen-decomposition of the real tridiagonal
// T = (Re alpha, beta), as reference coefficients_integration.c:104-145:
// y = Z exp(-i D prop_dt) Z^T e_1.  Called by one whole wave (lanes 0..63);
// z is LDS scratch of n rows of zstride doubles.
//
// renorm: the caller renormalises the result (imaginary time).  Then the
// exponentials are taken relative to the dominant one, exp((d_k - d*) b)
// with d* the eigenvalue where d b is largest: a common factor that the
// renormalisation removes, and that keeps exp(d b) from underflowing to 0
// for every k (then C' = 0 and the renormalisation would give NaN) when
// |E| dt exceeds about 745.
__device__ inline void sil_tridiag_wave(SilState* st, double dt_re, double dt_im, double* z, int zstride,
                                        int renorm) {
    const int lane = threadIdx.x;
    const int n = st->iter_done;
    double d = lane < n ? st->alpha[lane].x : 0.0;
    double e = lane < n ? st->beta[lane] : 0.0;
    double* zr = z + lane * zstride;
    if (tridiag_eig_wave(n, d, e, zr)) {
        if (lane == 0) st->eig_fail = 1;
        return;
    }
    // lane k: aux_k = Z[0][k] exp(-i d_k prop_dt); exp(-i d dt) for complex
    // dt = a + ib is exp(d b) (cos(d a) - i sin(d a))
    double shift = -INFINITY;  // max over k of d_k b
    for (int j = 0; j < n; j++) shift = fmax(shift, rlane(d, j) * dt_im);
    if (!renorm) shift = 0.0;
    double ax = 0, ay = 0;
    if (lane < n) {
        const double z0k = z[lane];  // row 0, column lane
        const double mag = exp(d * dt_im - shift);
        double sn, cs;
        sincos(-d * dt_re, &sn, &cs);
        ax = z0k * mag * cs;
        ay = z0k * mag * sn;
    }
    double yx = 0, yy = 0;
    for (int j = 0; j < n; j++) {
        const double zkj = zr[j];
        yx += rlane(ax, j) * zkj;
        yy += rlane(ay, j) * zkj;
    }
    if (lane < n) st->y[lane] = make_double2(yx * st->s[lane], yy * st->s[lane]);
}

}  // namespace mctdhb
