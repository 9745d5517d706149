// bh_spmv.hip -- application of H_b = J_b T + U_b V to B row-interleaved vectors.
//
// Replaces the Eigen CSC x dense product behind Spectra's SparseGenMatProd::perform_op
// (external/spectra/include/Spectra/MatOp/SparseGenMatProd.h:81-86 ->
// include/Eigen/src/SparseCore/SparseDenseProduct.h:86-107), a serial column scatter in the
// reference.  Here: CSR rows, G lanes per row and B vectors per CSR pass, FP64 accumulation.
// Both precisions read the packed words and the exact FP64 values of the table; they differ in the vectors.
// The kernel is HBM-bound: per pass it reads the matrix once (4 B per entry) plus the row pointers and the
// diagonal, and B * (x gather + y write).
#include <algorithm>
#include <cmath>
#include <mutex>

#include "bh_kernels.hpp"
#include "bh_spmv.hpp"

// the value table and the lanes' coefficients in LDS
template <typename XT, int B>
__device__ __forceinline__ void spmv_setup(const SpmvArgs<XT>& a, const SpmvCoef& c, double* tab, double* cJ, double* cU) {
    for (int i = threadIdx.x; i < (1 << a.cb); i += BH_WG) tab[i] = a.table[i];
    if (threadIdx.x < B) {
        cJ[threadIdx.x] = a.J ? a.J[threadIdx.x] : c.J[threadIdx.x];
        cU[threadIdx.x] = a.J ? a.U[threadIdx.x] : c.U[threadIdx.x];
    }
    __syncthreads();
}

SpmvCoef bh_spmv_coef(const double* J, const double* U, int B) {
    SpmvCoef c;
    for (int b = 0; b < 64; ++b) {
        c.J[b] = b < B ? J[b] : 0.0;
        c.U[b] = b < B ? U[b] : 0.0;
    }
    return c;
}

template <typename XT, int B, int G>
__global__ void __launch_bounds__(BH_WG) k_spmv(SpmvArgs<XT> a, SpmvCoef c) {
    constexpr int GB = G * B;
    constexpr int SLOTS = BH_WG / GB;
    extern __shared__ double tab[];  // (1 << cb) entries
    __shared__ double cJ[B], cU[B];
    spmv_setup<XT, B>(a, c, tab, cJ, cU);
    const int lane = threadIdx.x;
    const int slot = lane / GB;
    const int g = (lane % GB) / B;
    const int b = lane % B;
    const int64_t ntile = (a.D + SLOTS - 1) / SLOTS;
    const int64_t tile = a.xcd ? bh_xcd_tile(blockIdx.x, gridDim.x) : blockIdx.x;
    if (tile >= ntile) return;  // whole workgroup leaves together (tile is uniform)
    const int64_t r = tile * SLOTS + slot;
    double acc = 0.0;
    if (r < a.D) acc = bh_row_partial<XT, B, G>(a.row_ptr[r], a.row_ptr[r + 1], g, b, a.words, tab, a.cb, a.x);
    acc = bh_group_sum<B, G>(acc);
    if (g == 0 && r < a.D) {
        const double xr = to_d(a.x[r * B + b]);
        a.y[r * B + b] = static_cast<XT>(cJ[b] * -acc + cU[b] * static_cast<double>(a.diag[r]) * xr);
    }
}

template <typename XT, int B>
__global__ void __launch_bounds__(BH_WG) k_spmv_rb(SpmvArgs<XT> a, SpmvCoef c, const int32_t* __restrict__ rb, int64_t nblocks) {
    extern __shared__ double smem[];
    double* tab = smem;  // (1 << cb) entries
    double* prod = smem + (1 << a.cb);
    __shared__ double cJ[B], cU[B];
    spmv_setup<XT, B>(a, c, tab, cJ, cU);
    const int64_t t = a.xcd ? bh_xcd_tile(blockIdx.x, gridDim.x) : blockIdx.x;
    auto epi = [&](int64_t r, int bb, const double (&sum)[1]) {
        const double d = static_cast<double>(a.diag[r]);
        a.y[r * B + bb] = static_cast<XT>(cJ[bb] * -sum[0] + cU[bb] * d * to_d(a.x[r * B + bb]));
    };
    bh_rowblock_run<XT, B, BH_WG>(t, t + 1, rb, a.row_ptr, a.words, tab, a.cb, a.x, prod, epi);
}

// epilogue of the row-lane and row-tile engines: y for the V vectors a thread holds of a row
template <typename XT, int B, int V>
struct SpmvEpi {
    const SpmvArgs<XT>& a;
    const double *cJ, *cU;
    __device__ __forceinline__ void operator()(int64_t r, int b0, const double (&acc)[V]) const {
        const double d = static_cast<double>(a.diag[r]);
        const BhVec<XT, V> xv = bh_vload<V>(a.x + r * B + b0);
        BhVec<XT, V> yv;
#pragma unroll
        for (int v = 0; v < V; ++v)
            yv.v[v] = static_cast<XT>(cJ[b0 + v] * -acc[v] + cU[b0 + v] * d * to_d(xv.v[v]));
        *reinterpret_cast<BhVec<XT, V>*>(a.y + r * B + b0) = yv;
    }
};

template <typename XT, int B, int V>
__global__ void __launch_bounds__(BH_WG) k_spmv_rl(SpmvArgs<XT> a, SpmvCoef c, int64_t rows_per_wg) {
    extern __shared__ double tab[];
    __shared__ double cJ[B], cU[B];
    spmv_setup<XT, B>(a, c, tab, cJ, cU);
    const int64_t t = a.xcd ? bh_xcd_tile(blockIdx.x, gridDim.x) : blockIdx.x;
    const int64_t r0 = min(t * rows_per_wg, a.D), r1 = min(r0 + rows_per_wg, a.D);
    SpmvEpi<XT, B, V> epi{a, cJ, cU};
    bh_rowlane_run<XT, B, V, BH_WG, 4>(r0, r1, a.row_ptr, a.words, tab, a.cb, a.x, epi);
}

// one thread per row (V = B): the words of a wave's 64 rows go through LDS
template <typename XT, int V>
__global__ void __launch_bounds__(BH_WG) k_spmv_rt(SpmvArgs<XT> a, SpmvCoef c, int64_t rows_per_wg, int cap) {
    extern __shared__ __align__(16) double smem[];
    double* tab = smem;
    __shared__ double cJ[V], cU[V];
    spmv_setup<XT, V>(a, c, tab, cJ, cU);
    const int64_t t = a.xcd ? bh_xcd_tile(blockIdx.x, gridDim.x) : blockIdx.x;
    const int64_t r0 = min(t * rows_per_wg, a.D), r1 = min(r0 + rows_per_wg, a.D);
    SpmvEpi<XT, V, V> epi{a, cJ, cU};
    bh_rowtile_run<XT, V, BH_WG, (V == 1 ? 8 : 4)>(r0, r1, a.row_ptr, a.words, tab, a.cb, a.x,
                                                   reinterpret_cast<uint32_t*>(smem + (1 << a.cb)), cap, epi);
}

int bh_tile_cap(const bh_ham* h) {
    const int need = 64 * std::max(h->max_row, 1) + 8;
    return std::min((need + 63) / 64 * 64, BH_TILE_WORDS);
}

// row-lane engine with V vectors per thread (V * sizeof(XT) <= 16 bytes, V <= B); one thread per row: row tiles
template <typename XT>
static void launch_spmv_rl(const bh_ham* h, const SpmvArgs<XT>& a, const SpmvCoef& c, int B, int V, hipStream_t s) {
    const size_t shm = (static_cast<size_t>(1) << a.cb) * sizeof(double);
    // up to four passes of BH_WG V / B rows per workgroup, fewer while that leaves under 1024 workgroups (four per CU)
    const int64_t pass = static_cast<int64_t>(BH_WG) * V / B;
    const int64_t rows_per_wg = pass * std::max<int64_t>(1, std::min<int64_t>(4, a.D / (pass * 1024)));
    const unsigned grid = static_cast<unsigned>((a.D + rows_per_wg - 1) / rows_per_wg);
    if (B == V) {
        const int cap = bh_tile_cap(h);
        const size_t sht = shm + static_cast<size_t>(BH_WG / 64) * cap * sizeof(uint32_t);
        if (V == 1) hipLaunchKernelGGL((k_spmv_rt<XT, 1>), dim3(grid), dim3(BH_WG), sht, s, a, c, rows_per_wg, cap);
        else if (V == 2) hipLaunchKernelGGL((k_spmv_rt<XT, 2>), dim3(grid), dim3(BH_WG), sht, s, a, c, rows_per_wg, cap);
        if constexpr (sizeof(XT) == 4)
            if (V == 4) hipLaunchKernelGGL((k_spmv_rt<XT, 4>), dim3(grid), dim3(BH_WG), sht, s, a, c, rows_per_wg, cap);
        return;
    }
#define L(BB, VV)                                                                                             \
    if (B == BB && V == VV) {                                                                                 \
        hipLaunchKernelGGL((k_spmv_rl<XT, BB, VV>), dim3(grid), dim3(BH_WG), shm, s, a, c, rows_per_wg);       \
        return;                                                                                               \
    }
    L(2, 1) L(4, 1) L(8, 1) L(16, 1) L(32, 1) L(64, 1)
    L(4, 2) L(8, 2) L(16, 2) L(32, 2) L(64, 2)
    if constexpr (sizeof(XT) == 4) {
        L(8, 4) L(16, 4) L(32, 4) L(64, 4)
    }
#undef L
}

template <typename XT>
static void launch_spmv_rb(const SpmvArgs<XT>& a, const SpmvCoef& c, int B, const int32_t* rb, int64_t nb, hipStream_t s) {
    const size_t shm = ((static_cast<size_t>(1) << a.cb) + BH_STAGE_PRODUCTS) * sizeof(double);
    const unsigned grid = static_cast<unsigned>(nb);
#define L(BB)                                                                                       \
    if (B == BB) {                                                                                  \
        hipLaunchKernelGGL((k_spmv_rb<XT, BB>), dim3(grid), dim3(BH_WG), shm, s, a, c, rb, nb);     \
        return;                                                                                     \
    }
    L(1) L(2) L(4) L(8) L(16) L(32) L(64)
#undef L
}

template <typename XT>
static void launch_spmv_g(const SpmvArgs<XT>& a, const SpmvCoef& c, int B, int G, hipStream_t s) {
    const int GB = G * B;
    const int64_t slots = BH_WG / GB;
    const unsigned grid = static_cast<unsigned>((a.D + slots - 1) / slots);
    const size_t shm = (static_cast<size_t>(1) << a.cb) * sizeof(double);
#define L(BB, GG)                                                                          \
    if (B == BB && G == GG) {                                                              \
        hipLaunchKernelGGL((k_spmv<XT, BB, GG>), dim3(grid), dim3(BH_WG), shm, s, a, c);   \
        return;                                                                            \
    }
    L(1, 1) L(1, 2) L(1, 4) L(1, 8) L(1, 16) L(1, 32) L(1, 64)
    L(2, 1) L(2, 2) L(2, 4) L(2, 8) L(2, 16) L(2, 32)
    L(4, 1) L(4, 2) L(4, 4) L(4, 8) L(4, 16)
    L(8, 1) L(8, 2) L(8, 4) L(8, 8)
    L(16, 1) L(16, 2) L(16, 4)
    L(32, 1) L(32, 2)
    L(64, 1)
#undef L
}

// SpMV variants: 0 = LDS-staged row blocks; V = 1, 2, 4 = V vectors per thread, B / V threads per row (64 V / B
// rows per wavefront); 100 + G = G lanes per row (64 / (G B) rows per wavefront)
template <typename XT>
static int spmv_launch(bh_ham* h, int var, const SpmvArgs<XT>& a, const SpmvCoef& c, int B, hipStream_t s) {
    if (var == 0) {
        const int32_t* rb = nullptr;
        int64_t nb = 0;
        BH_TRY(bh_ham_rowblocks(h, B, &rb, &nb));
        launch_spmv_rb(a, c, B, rb, nb, s);
    } else if (var >= 100) {
        launch_spmv_g(a, c, B, var - 100, s);
    } else {
        launch_spmv_rl(h, a, c, B, var, s);
    }
    return BH_OK;
}

// One operator application with the variant chosen for (h, precision, B).  The first application at a
// (precision, B) runs the autotuner unless BHX_TUNE=0 or BHX_ENGINE is set: every variant that fits is
// timed with HIP events over a warm-up and three applications to the caller's own x and y (y = H x is
// idempotent), and the fastest is kept in the handle.  Under stream capture the default variant is used.
template <typename XT>
static int apply_t(bh_ctx* ctx, bh_ham* h, const SpmvArgs<XT>& a, const SpmvCoef& c, int prec, int B, hipStream_t s) {
    const int key = bh_tune_key(1, prec, B);
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    auto it = h->tuned.find(key);
    if (it != h->tuned.end()) return spmv_launch(h, it->second.variant, a, c, B, s);
    const int eng = bh_engine_choice(B, h);
    BhTuned t;
    t.variant = eng == 2 ? 1 : (eng == 1 ? 0 : 100 + bh_pick_lanes(h, B));
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    BH_HIP(ctx, hipStreamIsCapturing(s, &cs));
    if (cs != hipStreamCaptureStatusNone) return spmv_launch(h, t.variant, a, c, B, s);
    if (bh_tune_enabled() && bh_engine_env() < 0) {
        std::vector<int> cand;
        if (static_cast<int64_t>(h->max_row) * B <= BH_STAGE_PRODUCTS_HOST) cand.push_back(0);
        cand.push_back(1);
        if (B >= 2) cand.push_back(2);
        if (B >= 4 && sizeof(XT) == 4) cand.push_back(4);
        const int G = bh_pick_lanes(h, B);
        if (G > 1) cand.push_back(100 + G);
        hipEvent_t e0 = nullptr, e1 = nullptr;
        BH_HIP(ctx, hipEventCreate(&e0));
        BH_HIP(ctx, hipEventCreate(&e1));
        double best = 0.0;
        for (int var : cand) {
            BH_TRY(spmv_launch(h, var, a, c, B, s));
            BH_HIP(ctx, hipEventRecord(e0, s));
            for (int r = 0; r < 3; ++r) BH_TRY(spmv_launch(h, var, a, c, B, s));
            BH_HIP(ctx, hipEventRecord(e1, s));
            BH_HIP(ctx, hipEventSynchronize(e1));
            float ms = 0.f;
            BH_HIP(ctx, hipEventElapsedTime(&ms, e0, e1));
            const double us = 1e3 * ms / 3;
            t.cand.push_back({var, us});
            if (best == 0.0 || us < best) {
                best = us;
                t.variant = var;
            }
        }
        (void)hipEventDestroy(e0);
        (void)hipEventDestroy(e1);
    }
    h->tuned[key] = t;
    return spmv_launch(h, t.variant, a, c, B, s);
}

int bh_apply(bh_ctx* ctx, bh_ham* h, const SpmvArgs<double>& a, const SpmvCoef& c, int key, int B, hipStream_t s) {
    return apply_t(ctx, h, a, c, key, B, s);
}
int bh_apply(bh_ctx* ctx, bh_ham* h, const SpmvArgs<float>& a, const SpmvCoef& c, int key, int B, hipStream_t s) {
    return apply_t(ctx, h, a, c, key, B, s);
}

int bh_pick_lanes(const bh_ham* h, int B) {
    // lanes per row: about half the mean row length, as a power of two, G*B <= 64
    const double avg = h->D ? static_cast<double>(h->nnz) / static_cast<double>(h->D) : 1.0;
    int G = 1;
    while (G < 64 && G * 2 <= avg) G <<= 1;
    while (G * B > 64 && G > 1) G >>= 1;
    return G;
}

double bh_spmv_bytes(const bh_ham* h, int prec, int B) {
    const double D = static_cast<double>(h->D), nnz = static_cast<double>(h->nnz);
    return nnz * 4.0 + 4.0 * (D + 1) + 4.0 * D + B * 2.0 * (prec == BH_PREC_FP64 ? 8.0 : 4.0) * D;
}

int bh_is_pow2_le64(int B) { return B >= 1 && B <= 64 && (B & (B - 1)) == 0; }

// ---- the SpMV entry point that allocates nothing -------------------------------------------------------------
// The coefficients go with the launch.  Under stream capture they are staged in this file-scope array instead, whose device
// address is looked up once per device with hipGetSymbolAddress (the array's name in host code is a host-side
// stand-in, never a device address), by copies that each replay repeats from the caller's arrays.  Every captured
// call on a device shares that device's copy, so graphs that overlap on one device race.
namespace {
constexpr int SPMV_SCRATCH_LANES = 64;  // the largest batch width of the SpMV kernels
static __device__ __align__(256) double scratch[2 * SPMV_SCRATCH_LANES];
constexpr int SPMV_SCRATCH_DEVICES = 64;
std::mutex g_scratch_mu;
double* g_scratch_ptr[SPMV_SCRATCH_DEVICES] = {};

// device address of `scratch` on the context's device (the device is current), looked up on first use
int scratch_ptr(bh_ctx* ctx, double** out) {
    if (ctx->device < 0 || ctx->device >= SPMV_SCRATCH_DEVICES)
        return bh_set_error(ctx, BH_EINVAL, "spmv_noalloc: device index beyond the scratch table");
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_ptr[ctx->device]) {
        void* p = nullptr;
        BH_HIP(ctx, hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        g_scratch_ptr[ctx->device] = static_cast<double*>(p);
    }
    *out = g_scratch_ptr[ctx->device];
    return BH_OK;
}
}  // namespace

extern "C" {

int bh_spmv_noalloc(bh_ctx* ctx, bh_ham* h, int prec, int B, const double* J, const double* U, const void* x, void* y,
                    void* stream) {
    if (!ctx || !h || !J || !U || !x || !y) return BH_EINVAL;
    if (!bh_is_pow2_le64(B) || B > SPMV_SCRATCH_LANES)
        return bh_set_error(ctx, BH_EINVAL, "spmv_noalloc: B must be a power of two <= 64 (the scratch holds 64 lanes)");
    if (prec != BH_PREC_FP64 && prec != BH_PREC_MIXED) return bh_set_error(ctx, BH_EINVAL, "spmv_noalloc: prec");
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    BH_HIP(ctx, hipSetDevice(ctx->device));
    if (prec == BH_PREC_FP64 && !h->prepared64)
        return bh_set_error(ctx, BH_EINVAL, "spmv_noalloc: handle not prepared for FP64 (bh_ham_prepare first)");
    hipStream_t s = stream ? static_cast<hipStream_t>(stream) : ctx->stream;
    // under capture the coefficients are staged in the device array by copies that a replay repeats from the caller's
    // J and U; otherwise they go with the launch
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    BH_HIP(ctx, hipStreamIsCapturing(s, &cs));
    const SpmvCoef c = bh_spmv_coef(J, U, B);
    double *dJ = nullptr, *dU = nullptr;
    if (cs != hipStreamCaptureStatusNone) {
        BH_TRY(scratch_ptr(ctx, &dJ));
        dU = dJ + SPMV_SCRATCH_LANES;
        BH_HIP(ctx, hipMemcpyAsync(dJ, J, B * sizeof(double), hipMemcpyHostToDevice, s));
        BH_HIP(ctx, hipMemcpyAsync(dU, U, B * sizeof(double), hipMemcpyHostToDevice, s));
    }
    // the variant the autotuner chose for this sector (no tuning here: it times with events), else the default
    // bh_apply uses under capture; the staged engine only when its row-block table for B already exists
    const int key = bh_tune_key(1, prec, B);
    auto it = h->tuned.find(key);
    int var;
    if (it != h->tuned.end()) {
        var = it->second.variant;
    } else {
        const int eng = bh_engine_choice(B, h);
        var = eng == 2 ? 1 : (eng == 1 ? 0 : 100 + bh_pick_lanes(h, B));
    }
    if (var == 0 && h->rowblocks.find(B) == h->rowblocks.end()) var = 1;
    if (prec == BH_PREC_FP64) {
        SpmvArgs<double> a{h->D, h->row_ptr, h->words, h->diag, h->table, h->code_bits,
                           dJ, dU, static_cast<const double*>(x), static_cast<double*>(y), 1};
        BH_TRY(spmv_launch(h, var, a, c, B, s));
    } else {
        SpmvArgs<float> a{h->D, h->row_ptr, h->words, h->diag, h->table, h->code_bits,
                          dJ, dU, static_cast<const float*>(x), static_cast<float*>(y), 1};
        BH_TRY(spmv_launch(h, var, a, c, B, s));
    }
    BH_HIP(ctx, hipGetLastError());
    // outside a capture the call returns with its work done
    if (cs == hipStreamCaptureStatusNone) BH_HIP(ctx, hipStreamSynchronize(s));
    return BH_OK;
}

int bh_spmv(bh_ctx* ctx, bh_ham* h, int prec, int B, const double* J, const double* U, const void* x, void* y,
            void* stream) {
    if (!ctx || !h || !J || !U || !x || !y) return BH_EINVAL;
    if (!bh_is_pow2_le64(B)) return bh_set_error(ctx, BH_EINVAL, "spmv: B must be a power of two <= 64");
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    BH_HIP(ctx, hipSetDevice(ctx->device));
    hipStream_t s = stream ? static_cast<hipStream_t>(stream) : ctx->stream;
    BH_TRY(bh_ham_prepare_locked(h, prec));
    const SpmvCoef c = bh_spmv_coef(J, U, B);
    {
        KTimer kt(ctx, "spmv", s);
        if (prec == BH_PREC_FP64) {
            SpmvArgs<double> a{h->D, h->row_ptr, h->words, h->diag, h->table, h->code_bits,
                               nullptr, nullptr, static_cast<const double*>(x), static_cast<double*>(y), 1};
            BH_TRY(bh_apply(ctx, h, a, c, prec, B, s));
        } else {
            SpmvArgs<float> a{h->D, h->row_ptr, h->words, h->diag, h->table, h->code_bits,
                              nullptr, nullptr, static_cast<const float*>(x), static_cast<float*>(y), 1};
            BH_TRY(bh_apply(ctx, h, a, c, prec, B, s));
        }
    }
    BH_HIP(ctx, hipGetLastError());
    BH_HIP(ctx, hipStreamSynchronize(s));  // the call returns with its work done
    return BH_OK;
}

int bh_spmv_host(bh_ctx* ctx, bh_ham* h, int prec, int B, const double* J, const double* U, const double* x,
                 double* y) {
    if (!ctx || !h || !x || !y) return BH_EINVAL;
    if (!bh_is_pow2_le64(B)) return bh_set_error(ctx, BH_EINVAL, "spmv: B must be a power of two <= 64");
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    BH_HIP(ctx, hipSetDevice(ctx->device));
    hipStream_t s = ctx->stream;
    const size_t n = static_cast<size_t>(h->D) * B;
    if (prec == BH_PREC_FP64) {
        DevArray<double> dx, dy;
        BH_TRY(dx.alloc(ctx, n));
        BH_TRY(dy.alloc(ctx, n));
        BH_HIP(ctx, hipMemcpyAsync(dx.p, x, n * 8, hipMemcpyHostToDevice, s));
        BH_TRY(bh_spmv(ctx, h, prec, B, J, U, dx.p, dy.p, nullptr));
        BH_HIP(ctx, hipMemcpyAsync(y, dy.p, n * 8, hipMemcpyDeviceToHost, s));
        BH_HIP(ctx, hipStreamSynchronize(s));
    } else {
        std::vector<float> xf(n), yf(n);
        for (size_t i = 0; i < n; ++i) xf[i] = static_cast<float>(x[i]);
        DevArray<float> dx, dy;
        BH_TRY(dx.alloc(ctx, n));
        BH_TRY(dy.alloc(ctx, n));
        BH_HIP(ctx, hipMemcpyAsync(dx.p, xf.data(), n * 4, hipMemcpyHostToDevice, s));
        BH_TRY(bh_spmv(ctx, h, prec, B, J, U, dx.p, dy.p, nullptr));
        BH_HIP(ctx, hipMemcpyAsync(yf.data(), dy.p, n * 4, hipMemcpyDeviceToHost, s));
        BH_HIP(ctx, hipStreamSynchronize(s));
        for (size_t i = 0; i < n; ++i) y[i] = yf[i];
    }
    return BH_OK;
}

int bh_spmv_bench(bh_ctx* ctx, bh_ham* h, int prec, int B, int reps, double* avg_ms, double* bytes) {
    if (!ctx || !h || reps < 1) return BH_EINVAL;
    if (!bh_is_pow2_le64(B)) return bh_set_error(ctx, BH_EINVAL, "spmv: B must be a power of two <= 64");
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    BH_HIP(ctx, hipSetDevice(ctx->device));
    hipStream_t s = ctx->stream;
    BH_TRY(bh_ham_prepare_locked(h, prec));
    const size_t n = static_cast<size_t>(h->D) * B;
    const size_t es = prec == BH_PREC_FP64 ? 8 : 4;
    DevArray<uint8_t> dx, dy;
    BH_TRY(dx.alloc(ctx, n * es));
    BH_TRY(dy.alloc(ctx, n * es));
    std::vector<double> ones(B, 1.0);
    const SpmvCoef c = bh_spmv_coef(ones.data(), ones.data(), B);
    BH_HIP(ctx, hipMemsetAsync(dx.p, 0, n * es, s));
    auto launch = [&]() -> int {
        if (prec == BH_PREC_FP64) {
            SpmvArgs<double> a{h->D, h->row_ptr, h->words, h->diag, h->table, h->code_bits,
                               nullptr, nullptr, reinterpret_cast<const double*>(dx.p), reinterpret_cast<double*>(dy.p), 1};
            return bh_apply(ctx, h, a, c, prec, B, s);
        }
        SpmvArgs<float> a{h->D, h->row_ptr, h->words, h->diag, h->table, h->code_bits,
                          nullptr, nullptr, reinterpret_cast<const float*>(dx.p), reinterpret_cast<float*>(dy.p), 1};
        return bh_apply(ctx, h, a, c, prec, B, s);
    };
    BH_TRY(launch());  // warm-up (also builds the row blocks)
    hipEvent_t e0, e1;
    BH_HIP(ctx, hipEventCreate(&e0));
    BH_HIP(ctx, hipEventCreate(&e1));
    BH_HIP(ctx, hipEventRecord(e0, s));
    for (int i = 0; i < reps; ++i) BH_TRY(launch());
    BH_HIP(ctx, hipEventRecord(e1, s));
    BH_HIP(ctx, hipEventSynchronize(e1));
    float ms = 0.f;
    BH_HIP(ctx, hipEventElapsedTime(&ms, e0, e1));
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    BH_HIP(ctx, hipGetLastError());
    if (avg_ms) *avg_ms = ms / reps;
    if (bytes) *bytes = bh_spmv_bytes(h, prec, B);
    return BH_OK;
}

}  // extern "C"
