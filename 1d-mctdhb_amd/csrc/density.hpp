// density.hpp - rho1 / rho2 as sums over configurations.
#pragma once

#include "pairs.hpp"
#include "space.hpp"

namespace mctdhb {

enum : int { kDmFP64 = 0, kDmMixed = 1 };

// Launch plan of the pair kernel (2 <= M <= 7): nb blocks of kDmWaves waves.
struct DmPlan {
    unsigned nb;
};
constexpr int kDmWaves = 8;
constexpr int kDmThreads = 64 * kDmWaves;
DmPlan dm_plan(const Space* S);

// Scratch of density_matrices (per-block partials, totals and the arrival
// counter of the last stage, which the first one clears): one call at a time.
int dm_workspace_create(const Space* S, void** work);
// the partial sums in it
double2* dm_partials(const Space* S, void* work);

// LDS bytes of the pair kernel, or 0 where its tables exceed the budget.
size_t dm_pair_smem(const Space* S);
// Whether square roots come from a table in LDS (N + 3 <= 2048).
bool dm_root_table(const Space* S);
inline LowCtx low_ctx(const Space* S) { return LowCtx{S->d_low, S->low_dim, S->dim, S->npar}; }

// With rinv set, also the synchronisation of rho1 (eigenvalues into eig when
// set, regularisation by reg, rinv = rho1^-1), as the standalone
// density_sync_small does.
struct DmSync {
    double2* rinv;
    double* eig;
    double reg;
};
// Where the totals go.  c: the coefficients (N = 1 reads them directly).
struct DmOut {
    const void* c;
    double2* rho1;
    double2* rho2;  // may be null
    DmSync sy;
};

// Per-orbital-count kernels (dm_m<M>.hip): per-block partials of the pair
// sums, or with one block everything.
struct PkDm;
template <int M> struct DmPairs {
    // arrive: the counter to clear, where the last stage counts
    static int run(const Space* S, const void* c, int prec, double2* part, unsigned* arrive, const DmPlan& plan,
                   const DmOut& out, hipStream_t st);
    // FP64 partials of count instances (pack.hpp); max_nb: their largest plan
    static int run_pk(const PkDm* tab, int count, unsigned max_nb, size_t smem, hipStream_t st);
};

// rho1 (M x M row-major, rho1[k*M+l] = <a+_k a_l>) and, if rho2 is non-null,
// rho2 (M^4, index k + sM + qM^2 + lM^3 = <a+_k a+_s a_q a_l>), complex128.
// coef is complex128 (prec = kDmFP64) or complex64 (kDmMixed).  index is
// kIdxTables or kIdxFly; it matters for norb = 1 and norb > 7, whose generic
// kernel reads the jump tables.  work: from dm_workspace_create.
constexpr unsigned kDmFinishBlocks = 64;  // up to this many partials one block finishes
int density_matrices(const Space* S, const void* coef, double2* rho1, double2* rho2, int prec, int index,
                     void* work, hipStream_t st, const DmSync* sync = nullptr);

}  // namespace mctdhb
