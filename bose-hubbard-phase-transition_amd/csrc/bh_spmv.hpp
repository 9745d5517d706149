// bh_spmv.hpp -- launch interface of the operator kernels (shared with the Lanczos driver).
#pragma once

#include "bh_internal.hpp"

constexpr int BH_TAB_MAX = 4096;  // entries of the sqrt(code) table held in LDS (code_bits <= 12)

// J_b and U_b of a launch, passed by value: the two device arrays they replace cost a call two allocations, two copies
// and two frees (28 -> 20 us for a call on a small sector from Python)
struct SpmvCoef {
    double J[64], U[64];
};

template <typename XT>
struct SpmvArgs {
    int64_t D;
    const int32_t* row_ptr;
    const uint32_t* words;  // column << cb | code
    const float* diag;      // V (small integers and halves: exact)
    const double* table;    // sqrt(code)
    int cb;
    const double* J;        // [B] on the device, or NULL: the values of the SpmvCoef argument
    const double* U;        // [B]
    const XT* x;            // [D][B]
    XT* y;                  // [D][B]
    int xcd;                // XCD-aware tile order
};

// tuning keys of the operator pass: the caller's FP64 and mixed products, and the FP64 product of the solver's finish
constexpr int BH_KEY_FINISH = 2;

int bh_pick_lanes(const bh_ham* h, int B);
double bh_spmv_bytes(const bh_ham* h, int prec, int B);
int bh_is_pow2_le64(int B);
int bh_ham_prepare_locked(bh_ham* h, int prec);
// one product with the variant tuned for (h, key, B); key: BH_PREC_FP64, BH_PREC_MIXED or BH_KEY_FINISH
int bh_apply(bh_ctx* ctx, bh_ham* h, const SpmvArgs<double>& a, const SpmvCoef& c, int key, int B, hipStream_t s);
int bh_apply(bh_ctx* ctx, bh_ham* h, const SpmvArgs<float>& a, const SpmvCoef& c, int key, int B, hipStream_t s);
SpmvCoef bh_spmv_coef(const double* J, const double* U, int B);
// words of a wave's LDS part on the row-tile engine: the longest 64 rows could need, within BH_TILE_WORDS
int bh_tile_cap(const bh_ham* h);
