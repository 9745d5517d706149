// bh_basis.hip -- fixed-N Fock basis on the device: lexicographic unranking, exact prime-product
// keys, stable LSD radix sort, permutation / inverse permutation in the reference's order (none of the
// sorting for the lexicographic order itself).
//
// Reference: BH::init_lexicographic / next_lexicographic (src/hamiltonian.cpp:60-85) enumerate the
// states in descending lexicographic order; BH::calculate_tags (:91-106) assigns
// tag = sum n_i ln p_i; BH::sort_basis (:109-123) argsorts the tags and applies the argsort with a
// cycle-swap loop that realises the inverse permutation.  Here the ordering key is the exact integer
// prod p_i^n_i (the tag is its logarithm, so the orders agree; distinct states have distinct keys by
// unique factorisation), sorted by a radix sort.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <memory>

#include "bh_scan.hpp"

// ---- keys --------------------------------------------------------------------------------------------
//
// The sort works on the leading 32 bits of the exact key in floating form (7 bits of exponent, 25 of mantissa): the
// truncation is monotone, so equal truncations are the only places where the order is still open, and those
// are runs of a few states that the permutation kernel orders by their exact keys.  Four passes over 8 bytes a state
// replace the eight (128-bit keys: sixteen) over 12 or 20 that the exact keys take: 0.32 -> 0.13 ms at
// D = 1,352,078.

__device__ __forceinline__ uint32_t key_trunc(uint64_t lo, uint64_t hi) {
    // leading bit at position e (key >= 1), then the 25 bits below it
    const int e = hi ? 127 - __clzll(static_cast<long long>(hi)) : 63 - __clzll(static_cast<long long>(lo));
    uint64_t m;
    if (e >= 25) {
        const int sh = e - 25;  // 0 .. 102
        m = sh == 0 ? lo : (sh >= 64 ? hi >> (sh - 64) : (lo >> sh) | (hi << (64 - sh)));
    } else {
        m = lo << (25 - e);
    }
    return (static_cast<uint32_t>(e) << 25) | (static_cast<uint32_t>(m) & 0x1ffffffu);
}

// exact keys of all states by lexicographic rank (WIDE: 128-bit products); tk: their truncations, or, with count set,
// zeros for the ranks that k_basis_count adds up
template <int NW, int BITS, bool WIDE>
__global__ void __launch_bounds__(256) k_basis_keys(int64_t D, int m, int n, const uint32_t* __restrict__ gg, int gsize,
                                                     const uint64_t* __restrict__ pw_lo, const uint64_t* __restrict__ pw_hi,
                                                     uint64_t* __restrict__ klo, uint64_t* __restrict__ khi,
                                                     uint32_t* __restrict__ tk, int count) {
    extern __shared__ uint32_t g[];
    bh_stage_table(gg, gsize, g);
    const int64_t p = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (p >= D) return;
    PState<NW, BITS> s;
    bh_unrank(p, m, n, g, s);
    uint64_t lo, hi = 0;
    if constexpr (WIDE) {
        unsigned __int128 key = 1;
#pragma unroll
        for (int i = 0; i < PState<NW, BITS>::MAXM; ++i) {
            if (i < m) {
                const size_t t = static_cast<size_t>(i) * (n + 1) + s.get(i);
                key *= (static_cast<unsigned __int128>(pw_hi[t]) << 64) | pw_lo[t];
            }
        }
        lo = static_cast<uint64_t>(key);
        hi = static_cast<uint64_t>(key >> 64);
        khi[p] = hi;
    } else {
        lo = 1;
#pragma unroll
        for (int i = 0; i < PState<NW, BITS>::MAXM; ++i)
            if (i < m) lo *= pw_lo[static_cast<size_t>(i) * (n + 1) + s.get(i)];
    }
    klo[p] = lo;
    tk[p] = count ? 0u : key_trunc(lo, hi);
}

__device__ __forceinline__ bool key_less(uint64_t alo, uint64_t ahi, uint64_t blo, uint64_t bhi) {
    return ahi < bhi || (ahi == bhi && alo < blo);
}

// ---- small sectors: ranks by counting ------------------------------------------------------------------
// rank[i] = number of keys below key i, 256 states against 512 per workgroup (whole numbers added atomically: any order
// gives the same).  D^2 comparisons are one launch of a few microseconds up to BS_COUNT_MAX states (D = 16,384:
// 2,048 workgroups), where the passes of the radix sort would be a chain of a dozen.
constexpr int64_t BS_COUNT_MAX = 16384;
constexpr int BS_CHUNK = 512;

template <bool WIDE>
__global__ void __launch_bounds__(256) k_basis_count(int64_t D, const uint64_t* __restrict__ klo, const uint64_t* __restrict__ khi,
                                                      uint32_t* __restrict__ rank) {
    __shared__ uint64_t lo[BS_CHUNK], hi[WIDE ? BS_CHUNK : 1];
    const int64_t j0 = static_cast<int64_t>(blockIdx.y) * BS_CHUNK;
    const int nj = static_cast<int>(min(static_cast<int64_t>(BS_CHUNK), D - j0));
    for (int j = threadIdx.x; j < nj; j += 256) {
        lo[j] = klo[j0 + j];
        if constexpr (WIDE) hi[j] = khi[j0 + j];
    }
    __syncthreads();
    const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (i >= D) return;
    const uint64_t mlo = klo[i], mhi = WIDE ? khi[i] : 0;
    uint32_t c = 0;
    for (int j = 0; j < nj; ++j) c += WIDE ? key_less(lo[j], hi[j], mlo, mhi) : lo[j] < mlo;
    atomicAdd(rank + i, c);
}

// ---- radix sort of the truncated keys --------------------------------------------------------------------

constexpr int RS_BLOCK = 256;
constexpr int RS_ROUNDS = 16;
constexpr int RS_TILE = RS_BLOCK * RS_ROUNDS;

// per-tile digit histogram, digit-major layout hist[d * nb + tile]
__global__ void __launch_bounds__(RS_BLOCK) k_rs_hist(const uint32_t* __restrict__ key, int64_t n, int shift,
                                                      int32_t* __restrict__ hist, int nb) {
    __shared__ int32_t cnt[256];
    cnt[threadIdx.x] = 0;
    __syncthreads();
    const int64_t base = static_cast<int64_t>(blockIdx.x) * RS_TILE;
#pragma unroll
    for (int r = 0; r < RS_ROUNDS; ++r) {
        const int64_t idx = base + r * RS_BLOCK + threadIdx.x;
        if (idx < n) atomicAdd(&cnt[(key[idx] >> shift) & 0xff], 1);
    }
    __syncthreads();
    hist[static_cast<int64_t>(threadIdx.x) * nb + blockIdx.x] = cnt[threadIdx.x];
}

// one workgroup per digit: its tile counts become their exclusive prefix sums, their total goes to tot[digit]
__global__ void __launch_bounds__(RS_BLOCK) k_rs_scan(int32_t* __restrict__ hist, int nb, int32_t* __restrict__ tot) {
    __shared__ int64_t lds[RS_BLOCK / 64 + 1];
    int32_t* h = hist + static_cast<int64_t>(blockIdx.x) * nb;
    int64_t run = 0;
    for (int t0 = 0; t0 < nb; t0 += RS_BLOCK) {
        const int t = t0 + threadIdx.x;
        const int32_t v = t < nb ? h[t] : 0;
        int64_t sum = 0;
        const int64_t ex = bh_block_exclusive_scan<RS_BLOCK>(v, lds, &sum);
        if (t < nb) h[t] = static_cast<int32_t>(run + ex);
        run += sum;
    }
    if (threadIdx.x == 0) tot[blockIdx.x] = static_cast<int32_t>(run);
}

// Stable scatter.  Elements are taken in rounds of RS_BLOCK consecutive positions; inside a round the
// rank of an element among equal digits comes from a ballot match within its wave and the counts of
// the lower waves, so the output keeps input order for equal digits.  vin NULL: the value is the position.
__global__ void __launch_bounds__(RS_BLOCK) k_rs_scatter(const uint32_t* __restrict__ key, const int32_t* __restrict__ vin,
                                                         uint32_t* __restrict__ okey, int32_t* __restrict__ vout, int64_t n,
                                                         int shift, const int32_t* __restrict__ offs, int nb,
                                                         const int32_t* __restrict__ tot) {
    __shared__ int32_t run[256];
    __shared__ int32_t wcnt[RS_BLOCK / 64][256];
    __shared__ int64_t lds[RS_BLOCK / 64 + 1];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wid = tid >> 6;
    const int64_t first = bh_block_exclusive_scan<RS_BLOCK>(tot[tid], lds, nullptr);
    run[tid] = static_cast<int32_t>(first) + offs[static_cast<int64_t>(tid) * nb + blockIdx.x];
#pragma unroll
    for (int w = 0; w < RS_BLOCK / 64; ++w) wcnt[w][tid] = 0;
    const uint64_t lt_mask = (1ull << lane) - 1ull;
    const int64_t base = static_cast<int64_t>(blockIdx.x) * RS_TILE;
    uint32_t ks[RS_ROUNDS];
    int32_t vs[RS_ROUNDS];
#pragma unroll
    for (int r = 0; r < RS_ROUNDS; ++r) {
        const int64_t idx = base + r * RS_BLOCK + tid;
        ks[r] = idx < n ? key[idx] : 0;
        vs[r] = idx < n ? (vin ? vin[idx] : static_cast<int32_t>(idx)) : 0;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < RS_ROUNDS; ++r) {
        const bool active = base + r * RS_BLOCK + tid < n;
        const int d = (ks[r] >> shift) & 0xff;
        uint64_t peers = __ballot(active);
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            const bool bit = (d >> b) & 1;
            const uint64_t bb = __ballot(active && bit);
            peers &= bit ? bb : ~bb;
        }
        const int rank = __popcll(peers & lt_mask);
        if (active && rank == 0) wcnt[wid][d] = __popcll(peers);
        __syncthreads();
        if (active) {
            int pos = run[d] + rank;
            for (int w = 0; w < wid; ++w) pos += wcnt[w][d];
            okey[pos] = ks[r];
            vout[pos] = vs[r];
        }
        __syncthreads();
        int add = 0;
#pragma unroll
        for (int w = 0; w < RS_BLOCK / 64; ++w) {
            add += wcnt[w][tid];
            wcnt[w][tid] = 0;
        }
        run[tid] += add;
        __syncthreads();
    }
}

// ---- permutation -------------------------------------------------------------------------------------

// the state of lexicographic rank v is the t-th smallest by key; reference order: the state of rank t sits at position
// v (the inverse permutation); ascending order: position t holds the state of rank v
__device__ __forceinline__ void basis_place(int32_t t, int32_t v, int order, int32_t* lex_of_pos, int32_t* pos_of_lex) {
    const bool ref = order == BH_ORDER_REFERENCE;
    lex_of_pos[ref ? v : t] = ref ? t : v;
    pos_of_lex[ref ? t : v] = ref ? v : t;
}

// by counted ranks (small sectors), or the identity of the lexicographic order (rank NULL)
__global__ void k_basis_perm(int64_t D, const uint32_t* __restrict__ rank, int order, int32_t* __restrict__ lex_of_pos,
                             int32_t* __restrict__ pos_of_lex) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= D) return;
    if (rank) {
        basis_place(static_cast<int32_t>(rank[i]), static_cast<int32_t>(i), order, lex_of_pos, pos_of_lex);
    } else {
        lex_of_pos[i] = static_cast<int32_t>(i);
        pos_of_lex[i] = static_cast<int32_t>(i);
    }
}

// from the sorted truncations: a state alone with its truncation sits at its place; a run of equal truncations is ordered
// by the exact keys, each of its states counting the smaller ones
__global__ void k_basis_perm_sorted(int64_t D, const uint32_t* __restrict__ key, const int32_t* __restrict__ val,
                                    const uint64_t* __restrict__ klo, const uint64_t* __restrict__ khi, int order,
                                    int32_t* __restrict__ lex_of_pos, int32_t* __restrict__ pos_of_lex) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= D) return;
    const uint32_t k = key[i];
    const int32_t v = val[i];
    int64_t a = i, e = i + 1;
    while (a > 0 && key[a - 1] == k) --a;
    while (e < D && key[e] == k) ++e;
    int64_t t = i;
    if (e - a > 1) {
        const uint64_t lo = klo[v], hi = khi ? khi[v] : 0;
        t = a;
        for (int64_t q = a; q < e; ++q) {
            const int32_t u = val[q];
            t += key_less(klo[u], khi ? khi[u] : 0, lo, hi) ? 1 : 0;
        }
    }
    basis_place(static_cast<int32_t>(t), v, order, lex_of_pos, pos_of_lex);
}

template <int NW, int BITS>
__global__ void __launch_bounds__(256) k_basis_states(int64_t D, int m, int n, const uint32_t* __restrict__ gg, int gsize,
                                                       const int32_t* __restrict__ lex_of_pos, uint8_t* __restrict__ out) {
    extern __shared__ uint32_t g[];
    bh_stage_table(gg, gsize, g);
    const int64_t k = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (k >= D) return;
    PState<NW, BITS> s;
    bh_unrank(lex_of_pos[k], m, n, g, s);
    for (int i = 0; i < m; ++i) out[k * m + i] = static_cast<uint8_t>(s.get(i));
}

// ---- dispatch over the instantiated state layouts ---------------------------------------------------

#define BH_LAYOUT_DISPATCH(nw, bits, MACRO)               \
    do {                                                  \
        if ((nw) == 1 && (bits) == 4) MACRO(1, 4);        \
        else if ((nw) == 2 && (bits) == 4) MACRO(2, 4);   \
        else if ((nw) == 2 && (bits) == 8) MACRO(2, 8);   \
        else MACRO(4, 8);                                 \
    } while (0)

// permutations of a basis whose arrays are allocated: the identity in lexicographic order, else from the sorted keys
static int basis_fill(bh_ctx* ctx, const bh_basis* b, const std::vector<uint32_t>& g, const std::vector<uint64_t>& plo,
                      const std::vector<uint64_t>& phi, bool wide, hipStream_t s) {
    const int64_t D = b->D;
    const int m = b->m, n = b->n, gsize = static_cast<int>(g.size());
    const unsigned grid = static_cast<unsigned>((D + 255) / 256);
    BH_HIP(ctx, hipMemcpyAsync(b->rank_tab, g.data(), g.size() * sizeof(uint32_t), hipMemcpyHostToDevice, s));
    BhScratch sc;
    if (b->order == BH_ORDER_LEX) {
        hipLaunchKernelGGL(k_basis_perm, dim3(grid), dim3(256), 0, s, D, nullptr, b->order, b->lex_of_pos, b->pos_of_lex);
        BH_HIP(ctx, hipGetLastError());
        BH_HIP(ctx, hipStreamSynchronize(s));
        return BH_OK;
    }
    const bool small = D <= BS_COUNT_MAX;
    const int nb = static_cast<int>((D + RS_TILE - 1) / RS_TILE);
    const size_t n8 = BhScratch::size(D * 8), n4 = BhScratch::size(D * 4), np = BhScratch::size(plo.size() * 16);
    const size_t nh = small ? 0 : BhScratch::size(static_cast<size_t>(256) * nb * 4) + BhScratch::size(256 * 4);
    BH_TRY(sc.open(ctx, np + n8 * (wide ? 2 : 1) + n4 + (small ? 0 : 3 * n4 + nh)));
    uint64_t* pw = sc.take<uint64_t>(plo.size() * 2);
    uint64_t* klo = sc.take<uint64_t>(D);
    uint64_t* khi = wide ? sc.take<uint64_t>(D) : nullptr;
    uint32_t* ka = sc.take<uint32_t>(D);
    std::vector<uint64_t> pwh(plo);  // low words, then high words: one copy
    pwh.insert(pwh.end(), phi.begin(), phi.end());
    BH_HIP(ctx, hipMemcpyAsync(pw, pwh.data(), pwh.size() * sizeof(uint64_t), hipMemcpyHostToDevice, s));
    {
        KTimer kt(ctx, "basis_keys", s);
#define LAUNCH_KEYS(NW_, BITS_)                                                                                        \
    do {                                                                                                               \
        if (wide)                                                                                                      \
            hipLaunchKernelGGL((k_basis_keys<NW_, BITS_, true>), dim3(grid), dim3(256), gsize * 4, s, D, m, n,         \
                               b->rank_tab, gsize, pw, pw + plo.size(), klo, khi, ka, small ? 1 : 0);                  \
        else                                                                                                           \
            hipLaunchKernelGGL((k_basis_keys<NW_, BITS_, false>), dim3(grid), dim3(256), gsize * 4, s, D, m, n,        \
                               b->rank_tab, gsize, pw, nullptr, klo, nullptr, ka, small ? 1 : 0);                      \
    } while (0)
        BH_LAYOUT_DISPATCH(b->nw, b->bits, LAUNCH_KEYS);
#undef LAUNCH_KEYS
    }
    BH_HIP(ctx, hipGetLastError());
    {
        KTimer kt(ctx, "basis_sort", s);
        if (small) {
            const dim3 gc(grid, static_cast<unsigned>((D + BS_CHUNK - 1) / BS_CHUNK));
            if (wide) hipLaunchKernelGGL((k_basis_count<true>), gc, dim3(256), 0, s, D, klo, khi, ka);
            else hipLaunchKernelGGL((k_basis_count<false>), gc, dim3(256), 0, s, D, klo, khi, ka);
            hipLaunchKernelGGL(k_basis_perm, dim3(grid), dim3(256), 0, s, D, ka, b->order, b->lex_of_pos, b->pos_of_lex);
        } else {
            uint32_t* kb = sc.take<uint32_t>(D);
            int32_t* va = sc.take<int32_t>(D);
            int32_t* vb = sc.take<int32_t>(D);
            int32_t* hist = sc.take<int32_t>(static_cast<size_t>(256) * nb);
            int32_t* tot = sc.take<int32_t>(256);
            const int32_t* iv = nullptr;  // the first pass's values are the ranks themselves
            uint32_t *ik = ka, *ok = kb;
            int32_t* ov = vb;
            for (int shift = 0; shift < 32; shift += 8) {
                hipLaunchKernelGGL(k_rs_hist, dim3(nb), dim3(RS_BLOCK), 0, s, ik, D, shift, hist, nb);
                hipLaunchKernelGGL(k_rs_scan, dim3(256), dim3(RS_BLOCK), 0, s, hist, nb, tot);
                hipLaunchKernelGGL(k_rs_scatter, dim3(nb), dim3(RS_BLOCK), 0, s, ik, iv, ok, ov, D, shift, hist, nb, tot);
                std::swap(ik, ok);
                iv = ov;
                ov = ov == vb ? va : vb;
            }
            hipLaunchKernelGGL(k_basis_perm_sorted, dim3(grid), dim3(256), 0, s, D, ik, iv, klo, khi, b->order, b->lex_of_pos,
                               b->pos_of_lex);
        }
    }
    BH_HIP(ctx, hipGetLastError());
    BH_HIP(ctx, hipStreamSynchronize(s));
    return BH_OK;
}

extern "C" {

int bh_basis_build(bh_ctx* ctx, int m, int n, int order, bh_basis** out) {
    if (!ctx || !out) return BH_EINVAL;
    *out = nullptr;
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    if (m < 1 || m > BH_MAX_SITES || n < 0 || n > 255)
        return bh_set_error(ctx, BH_EINVAL, "basis: need 1 <= m <= 32 and 0 <= n <= 255");
    if (order != BH_ORDER_REFERENCE && order != BH_ORDER_ASCENDING && order != BH_ORDER_LEX)
        return bh_set_error(ctx, BH_EINVAL, "basis: unknown order");
    const int64_t D = bh_binom_host(m + n - 1, n);
    if (D <= 0 || D > INT32_MAX) return bh_set_error(ctx, BH_ERANGE, "basis: dimension exceeds the int32 range");
    const int key_bits = bh_key_bits(m, n);
    if (key_bits > 128) return bh_set_error(ctx, BH_ERANGE, "basis: ordering key prod p_i^n_i exceeds 128 bits");
    BH_HIP(ctx, hipSetDevice(ctx->device));
    hipStream_t s = ctx->stream;

    std::unique_ptr<bh_basis> bp(new bh_basis());
    bh_basis* b = bp.get();
    b->ctx = ctx;
    b->m = m;
    b->n = n;
    b->order = order;
    b->D = D;
    b->layout_id = bh_next_layout_id();
    bh_state_layout(m, n, &b->nw, &b->bits);

    // rank table g[l][R] = C(R + m-l-2, m-l-1), l in [0, m-2], R in [0, n]; values < D
    const int rows = m > 1 ? m - 1 : 1;
    std::vector<uint32_t> g(static_cast<size_t>(rows) * (n + 1), 0u);
    for (int l = 0; l + 1 < m; ++l)
        for (int R = 0; R <= n; ++R) g[static_cast<size_t>(l) * (n + 1) + R] = static_cast<uint32_t>(bh_binom_host(R + m - l - 2, m - l - 1));
    // prime powers p_i^e, e in [0, n], as 128-bit (lo, hi)
    std::vector<uint64_t> plo(static_cast<size_t>(m) * (n + 1)), phi(static_cast<size_t>(m) * (n + 1));
    for (int i = 0; i < m; ++i) {
        unsigned __int128 v = 1;
        for (int e = 0; e <= n; ++e) {
            plo[static_cast<size_t>(i) * (n + 1) + e] = static_cast<uint64_t>(v);
            phi[static_cast<size_t>(i) * (n + 1) + e] = static_cast<uint64_t>(v >> 64);
            if (e < n) {
                // p_i^e <= p_{m-1}^n < 2^128 for every e <= n, so this never wraps when used
                v *= static_cast<unsigned __int128>(bh_primes[i]);
            }
        }
    }
    const bool wide = key_bits > 64;
    const size_t gb = BhScratch::size(g.size() * sizeof(uint32_t)), pb = BhScratch::size(static_cast<size_t>(D) * sizeof(int32_t));
    void* block = nullptr;
    BH_TRY(bh_dev_alloc(ctx, &block, gb + 2 * pb));
    b->block = block;
    b->block_bytes = gb + 2 * pb;
    b->rank_tab = static_cast<uint32_t*>(block);
    b->lex_of_pos = reinterpret_cast<int32_t*>(static_cast<char*>(block) + gb);
    b->pos_of_lex = reinterpret_cast<int32_t*>(static_cast<char*>(block) + gb + pb);
    b->bytes = g.size() * sizeof(uint32_t) + 2 * static_cast<size_t>(D) * sizeof(int32_t);
    const int rc = basis_fill(ctx, b, g, plo, phi, wide, s);
    if (rc != BH_OK) {
        (void)hipStreamSynchronize(s);
        bh_dev_free(ctx, block, b->block_bytes);
        return rc;
    }
    *out = bp.release();
    return BH_OK;
}

int bh_basis_destroy(bh_basis* b) {
    if (!b) return BH_EINVAL;
    bh_ctx* ctx = b->ctx;
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    (void)hipSetDevice(ctx->device);
    bh_dev_free(ctx, b->block, b->block_bytes);
    delete b;
    return BH_OK;
}

int64_t bh_basis_dim(const bh_basis* b) { return b ? b->D : -1; }

int bh_basis_copy_states(const bh_basis* b, uint8_t* states) {
    if (!b || !states) return BH_EINVAL;
    bh_ctx* ctx = b->ctx;
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    BH_HIP(ctx, hipSetDevice(ctx->device));
    hipStream_t s = ctx->stream;
    DevArray<uint8_t> out;
    BH_TRY(out.alloc(ctx, static_cast<size_t>(b->D) * b->m));
    const unsigned grid = static_cast<unsigned>((b->D + 255) / 256);
    const int gsize = (b->m > 1 ? b->m - 1 : 1) * (b->n + 1);
#define LAUNCH_STATES(NW_, BITS_)                                                                                  \
    hipLaunchKernelGGL((k_basis_states<NW_, BITS_>), dim3(grid), dim3(256), gsize * 4, s, b->D, b->m, b->n,        \
                       b->rank_tab, gsize, b->lex_of_pos, out.p)
    BH_LAYOUT_DISPATCH(b->nw, b->bits, LAUNCH_STATES);
#undef LAUNCH_STATES
    BH_HIP(ctx, hipGetLastError());
    BH_HIP(ctx, hipMemcpyAsync(states, out.p, static_cast<size_t>(b->D) * b->m, hipMemcpyDeviceToHost, s));
    BH_HIP(ctx, hipStreamSynchronize(s));
    return BH_OK;
}

int bh_basis_copy_tags(const bh_basis* b, double* tags) {
    if (!b || !tags) return BH_EINVAL;
    std::vector<uint8_t> st(static_cast<size_t>(b->D) * b->m);
    BH_TRY(bh_basis_copy_states(b, st.data()));
    // same accumulation order as BH::calculate_tag (src/hamiltonian.cpp:91-97)
    double lp[BH_MAX_SITES];
    for (int i = 0; i < b->m; ++i) lp[i] = std::log(static_cast<double>(bh_primes[i]));
    for (int64_t k = 0; k < b->D; ++k) {
        double t = 0.0;
        for (int i = 0; i < b->m; ++i) t += static_cast<double>(st[static_cast<size_t>(k) * b->m + i]) * lp[i];
        tags[k] = t;
    }
    return BH_OK;
}

int bh_basis_copy_perm(const bh_basis* b, int32_t* lex_of_pos, int32_t* pos_of_lex) {
    if (!b) return BH_EINVAL;
    bh_ctx* ctx = b->ctx;
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    BH_HIP(ctx, hipSetDevice(ctx->device));
    if (lex_of_pos)
        BH_HIP(ctx, hipMemcpyAsync(lex_of_pos, b->lex_of_pos, static_cast<size_t>(b->D) * sizeof(int32_t),
                                   hipMemcpyDeviceToHost, ctx->stream));
    if (pos_of_lex)
        BH_HIP(ctx, hipMemcpyAsync(pos_of_lex, b->pos_of_lex, static_cast<size_t>(b->D) * sizeof(int32_t),
                                   hipMemcpyDeviceToHost, ctx->stream));
    BH_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return BH_OK;
}

}  // extern "C"
