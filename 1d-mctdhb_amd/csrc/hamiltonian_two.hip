// hamiltonian_two.hip - host side of the two-stage H.C: the pair matrix, the
// choice of form and the dispatch over orbital counts.
#include "hamiltonian_two.hpp"
#include "hc_coef.hpp"
#include "pack.hpp"

namespace mctdhb {

extern template struct HcTwo<2>;
extern template struct HcTwo<3>;
extern template struct HcTwo<4>;
extern template struct HcTwo<5>;
extern template struct HcTwo<6>;
extern template struct HcTwo<7>;
extern template struct HcTwoRows<6>;
extern template struct HcTwoRows<7>;

__global__ void k_pair_matrix(int M, int N, const double2* __restrict__ hob, const double2* __restrict__ hint,
                              double2* __restrict__ X) {
    pair_matrix_part(blockIdx.x * blockDim.x + threadIdx.x, gridDim.x * blockDim.x, M, N, hob, hint, X);
}

int two_matrix(const Space* S, const double2* hob, const double2* hint, double2* X, hipStream_t st) {
    const int P = pair_count(S->norb);
    k_pair_matrix<<<div_up((uint64_t) P * P, 64), 64, 0, st>>>(S->norb, S->npar, hob, hint, X);
    MCTDHB_HIP_CHECK(hipGetLastError());
    return kOk;
}

// Packed form: one block per instance.
__global__ void k_pair_matrix_pk(const PkCf* __restrict__ tab, int M) {
    const PkCf a = tab[blockIdx.x];
    pair_matrix_part(threadIdx.x, blockDim.x, M, a.npar, a.hob, a.hint, a.X);
}

int pk_pair_matrix(const PkCf* tab, int count, int M, hipStream_t st) {
    k_pair_matrix_pk<<<count, 256, 0, st>>>(tab, M);
    MCTDHB_HIP_CHECK(hipGetLastError());
    return kOk;
}

bool two_possible(const Space* S, int prec) {
    const uint64_t size = prec == kPrecFP64 ? sizeof(double2) : sizeof(float2);
    return S->d_low && S->dim * size < (1ull << 32) && kRedBytes + two_table_bytes(S) <= 64 * 1024;
}

// From M = 6 on.  The first stage's P^2 products per configuration of N - 2
// particles replace 256 (M = 6) and 504 (M = 7) gathers and products per
// configuration: FP64 product at N=37, M=6 147 -> 116 us; mixed Lanczos
// iteration at N=30, M=7 485 -> 279 us, SIL step 3.93 -> 2.21 ms; N=18, M=6
// (NC 33,649) whole step 290 -> 263 us.  No lower bound on NC: a product of the
// smallest spaces takes no longer in two launches than one-stage rows do with
// a prebuilt block (mixed, M = 6: NC 21 12.7 and 12.5 us, NC 252 12.3 and 12.0;
// M = 7: NC 28 19.7 and 26.1; FP64 is faster at every size).  At M = 5 the 15 arrays of psi go to
// memory and back (1 GB complex64 at N=100), which costs more than the 131
// gathers they replace: SIL step 1.93 -> 2.23 ms mixed, 2.82 -> 3.68 ms FP64;
// at N=200, M=4 0.67 -> 0.76 ms.
bool two_faster(const Space* S, int prec) { return S->norb >= 6 && two_possible(S, prec); }

#define ROWS(call)                                                                                          \
    switch (S->norb) {                                                                                      \
        case 6: return HcTwoRows<6>::call;                                                                   \
        case 7: return HcTwoRows<7>::call;                                                                   \
        default: set_error("the two-stage H.C covers norb 6 and 7"); return kInvalidArgument;                \
    }

int two_apply(const Space* S, const void* c, const double2* X, void* psi, void* out, int prec, hipStream_t st) {
    ROWS(plain(S, c, X, psi, out, prec, st))
}

int two_lanczos(const Space* S, const double2* X, void* psi, const LanczosHcArgs& a, int prec, hipStream_t st) {
    ROWS(lanczos(S, X, psi, a, prec, st))
}

#undef ROWS

#define DISPATCH(call)                                                                                      \
    switch (S->norb) {                                                                                      \
        case 2: return HcTwo<2>::call;                                                                       \
        case 3: return HcTwo<3>::call;                                                                       \
        case 4: return HcTwo<4>::call;                                                                       \
        case 5: return HcTwo<5>::call;                                                                       \
        case 6: return HcTwo<6>::call;                                                                       \
        case 7: return HcTwo<7>::call;                                                                       \
        default: set_error("the pair forms of H.C cover 2 <= norb <= 7"); return kInvalidArgument;           \
    }

int two_rayleigh(const Space* S, const double2* X, const LanczosHcArgs& a, int prec, hipStream_t st) {
    DISPATCH(rayleigh(S, X, a, prec, st))
}

int two_small(const Space* S, const double2* X, double2* psi, const SmallSilArgs& a, hipStream_t st) {
    DISPATCH(small(S, X, psi, a, st))
}

#undef DISPATCH

int pk_sil_small(const PkSil* tab, int count, int M, int form, size_t smem, hipStream_t st) {
    switch (M) {
        case 2: return HcTwo<2>::small_pk(tab, count, form, smem, st);
        case 3: return HcTwo<3>::small_pk(tab, count, form, smem, st);
        case 4: return HcTwo<4>::small_pk(tab, count, form, smem, st);
        case 5: return HcTwo<5>::small_pk(tab, count, form, smem, st);
        case 6: return HcTwo<6>::small_pk(tab, count, form, smem, st);
        case 7: return HcTwo<7>::small_pk(tab, count, form, smem, st);
        default: set_error("the one-workgroup SIL step covers 2 <= norb <= 7"); return kInvalidArgument;
    }
}

}  // namespace mctdhb
