// bh_hamiltonian.hip -- count / tile scan / fill CSR build of the hopping term T and
// the diagonal interaction V over a neighbour list, in the basis order of a bh_basis.
//
// Reference: BH::fill_hopping (src/hamiltonian.cpp:170-191) and BH::fill_interaction (:194-211),
// selected by BH::fixed_bosons_hamiltonian (:238-256).  The intended operator is built: for every
// site i and every entry j of i's neighbour list with n_j >= 1, the state a_i^+ a_j |k> receives
// -sqrt((n_i+1) n_j); repeated neighbour entries add up, as repeated triplets do in
// setFromTriplets (:190).  The target's column is found exactly: lexicographic rank of the target
// (prefix sums of binomials) -> position through the basis permutation.
//
// Storage: one 32-bit word per entry, column << code_bits | code, with code = (c w)^2 (n_i+1) n_j
// (w: multiplicity of the neighbour entry, c: 2 under BH_CONV_REF_HOP, else 1), so that the value
// -c w sqrt((n_i+1) n_j) = -sqrt(code) is read exactly from a small FP64 table.  Columns ascending per
// row, as in Eigen's compressed storage.
#include <algorithm>
#include <cmath>
#include <map>
#include <memory>

#include <cstdlib>
#include <cstring>

#include "bh_scan.hpp"
#include "bh_spmv.hpp"

constexpr int HB_BLOCK = 64;  // one wave per block: per-thread LDS row buffers stay small

struct EdgeArgs {
    int E;
    const int8_t* ei;    // target site i (gains a boson)
    const int8_t* ej;    // source site j (loses a boson)
    const uint32_t* cm;  // code multiplier (c w)^2
};

// entries a row gains per occupied site: the distinct directed bonds that leave it
struct SiteDeg {
    uint8_t d[BH_MAX_SITES];
};

constexpr int HC_BLOCK = 256;
constexpr int HC_TILE = 512;  // rows of a count tile (two per thread)

// entries of every row (cnt) and of every tile of HC_TILE rows (tile)
template <int NW, int BITS>
__global__ void __launch_bounds__(HC_BLOCK) k_ham_count(int64_t D, int m, int n, const uint32_t* __restrict__ gg, int gsize,
                                                        const int32_t* __restrict__ lex_of_pos, SiteDeg deg,
                                                        uint8_t* __restrict__ cnt, int64_t* __restrict__ tile) {
    extern __shared__ uint32_t g[];
    __shared__ int red[HC_BLOCK / 64];
    bh_stage_table(gg, gsize, g);
    int sum = 0;
#pragma unroll
    for (int u = 0; u < HC_TILE / HC_BLOCK; ++u) {
        const int64_t q = static_cast<int64_t>(blockIdx.x) * HC_TILE + u * HC_BLOCK + threadIdx.x;
        if (q >= D) continue;
        PState<NW, BITS> s;
        bh_unrank(lex_of_pos[q], m, n, g, s);
        int c = 0;
#pragma unroll
        for (int j = 0; j < PState<NW, BITS>::MAXM; ++j)
            if (j < m) c += s.get(j) >= 1 ? deg.d[j] : 0;
        cnt[q] = static_cast<uint8_t>(c);
        sum += c;
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) sum += __shfl_xor(sum, o, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = sum;
    __syncthreads();
    if (threadIdx.x == 0) tile[blockIdx.x] = red[0] + red[1] + red[2] + red[3];
}

// single workgroup: exclusive scan of the nb tile sums in place
__global__ void __launch_bounds__(1024) k_scan_tiles(int64_t* __restrict__ tile, int64_t nb) {
    __shared__ int64_t lds[1024 / 64 + 1];
    const int64_t per = (nb + 1023) / 1024;
    const int64_t b0 = static_cast<int64_t>(threadIdx.x) * per;
    int64_t s = 0;
    for (int64_t i = b0; i < b0 + per && i < nb; ++i) s += tile[i];
    int64_t run = bh_block_exclusive_scan<1024>(s, lds, nullptr);
    for (int64_t i = b0; i < b0 + per && i < nb; ++i) {
        const int64_t t = tile[i];
        tile[i] = run;
        run += t;
    }
}

// w[0 .. P-1] ascending: Batcher's odd-even merge sort, every index known at compile time (registers)
template <int P>
__device__ __forceinline__ void sort_registers(uint32_t (&w)[P]) {
#pragma unroll
    for (int p = 1; p < P; p <<= 1)
#pragma unroll
        for (int k = p; k >= 1; k >>= 1)
#pragma unroll
            for (int j = k % p; j + k < P; j += 2 * k)
#pragma unroll
                for (int i = 0; i < k; ++i)
                    if (i + j + k < P && (i + j) / (2 * p) == (i + j + k) / (2 * p)) {
                        const uint32_t a = w[i + j], b = w[i + j + k];
                        w[i + j] = min(a, b);
                        w[i + j + k] = max(a, b);
                    }
}

// Fill, one wave per 64 rows: row pointers, sorted words, diagonal, and the wave's part of the row statistics.
// A thread unranks its row's state once and keeps, for every site l, the sums over l' < l of the steps
// g[l'][R] - g[l'][R - 1] and g[l'][R + 1] - g[l'][R] (R: bosons right of l'); moving a boson from j to i changes R by one
// on the sites between, so a hop's rank is the row's plus one difference of two such sums, whatever the
// distance.  Every directed bond has a register (P >= E of them; all ones where its source is empty, which no entry
// is: the word of D = 2^k states only), so that the gathers of the positions are in flight together and the row
// is sorted by a network of min / max instead of an insertion whose 64 lanes wait for the longest (P = 32: 191 pairs).
// The 64 rows are one contiguous run of words: they are laid out in LDS and written coalesced.  D = 1,352,078 with E = 24 bonds
// in the reference's order: 280 -> 191 us, now bound by the gathers of the positions (5.4 MB, more than one L2).
// stats: longest row, largest row sum of |T|, min and max of V.
template <int NW, int BITS, int P>
__global__ void __launch_bounds__(HB_BLOCK) k_ham_fill(int64_t D, int m, int n, const uint32_t* __restrict__ g_glob, int gsize,
                                                       const int32_t* __restrict__ lex_of_pos,
                                                       const int32_t* __restrict__ pos_of_lex, EdgeArgs ed, int cb,
                                                       const double* __restrict__ table, unsigned flags,
                                                       const uint8_t* __restrict__ cntg, const int64_t* __restrict__ tile,
                                                       int64_t nnz, int32_t* __restrict__ row_ptr, uint32_t* __restrict__ words,
                                                       float* __restrict__ diag, int4* __restrict__ stats) {
    extern __shared__ uint32_t lds[];
    const int lane = threadIdx.x;
    uint32_t* g = lds;                       // gsize words
    uint32_t* dn = g + gsize;                // [m][64] prefix sums for one boson less right of the site
    uint32_t* up = dn + m * HB_BLOCK;        // [m][64] and for one more
    uint32_t* run = dn;                      // the wave's words, contiguous (dn and up are done with by then)
    for (int a = lane; a < gsize; a += HB_BLOCK) g[a] = g_glob[a];
    const int64_t q0 = static_cast<int64_t>(blockIdx.x) * HB_BLOCK, q = q0 + lane;
    const bool valid = q < D;
    const int64_t p = valid ? lex_of_pos[q] : 0;
    // first word of this row: the tile's, the tile's earlier rows', the wave's earlier lanes'
    const int64_t tq = q0 / HC_TILE;
    int before = 0;
    for (int64_t r = tq * HC_TILE + lane; r < q0; r += HB_BLOCK) before += cntg[r];
    int inc = valid ? cntg[q] : 0;
    const int cnt = inc;
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) before += __shfl_xor(before, o, 64);
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(inc, o, 64);
        if (lane >= o) inc += y;
    }
    const int64_t wave0 = tile[tq] + before;
    const int total = __shfl(inc, 63, 64), excl = inc - cnt;
    if (valid) row_ptr[q] = static_cast<int32_t>(wave0 + excl);
    if (q == D - 1) row_ptr[D] = static_cast<int32_t>(nnz);
    __syncthreads();
    PState<NW, BITS> s;
    bh_unrank(p, m, n, g, s);
    {
        int R = n;
        uint32_t d = 0, u = 0;
#pragma unroll
        for (int l = 0; l < PState<NW, BITS>::MAXM; ++l) {
            if (l < m) {
                dn[l * HB_BLOCK + lane] = d;
                up[l * HB_BLOCK + lane] = u;
                R -= s.get(l);
                if (l < m - 1) {
                    const uint32_t* gl = g + l * (n + 1);
                    const uint32_t g0 = gl[R], gm = gl[max(R - 1, 0)], gp = gl[min(R + 1, n)];
                    // R = 0 has no boson to lose, R = n none to gain: steps that no hop of this state uses
                    d += R > 0 ? g0 - gm : 0u;
                    u += R < n ? gp - g0 : 0u;
                }
            }
        }
    }
    const uint32_t mask = (1u << cb) - 1u;
    uint32_t w[P];
#pragma unroll
    for (int e = 0; e < P; ++e) {
        w[e] = 0xffffffffu;
        if (e < ed.E) {  // uniform
            const int i = ed.ei[e], j = ed.ej[e], nj = s.get(j);
            const uint32_t t = static_cast<uint32_t>(p) +
                               (i < j ? dn[i * HB_BLOCK + lane] - dn[j * HB_BLOCK + lane] : up[i * HB_BLOCK + lane] - up[j * HB_BLOCK + lane]);
            const uint32_t code = ed.cm[e] * static_cast<uint32_t>((s.get(i) + 1) * nj);
            if (valid && nj >= 1) w[e] = (t << cb) | code;
        }
    }
    if (pos_of_lex) {  // uniform: ranks to positions
#pragma unroll
        for (int e0 = 0; e0 < P; e0 += 8) {
            uint32_t c[8];
#pragma unroll
            for (int e = e0; e < e0 + 8; ++e) c[e - e0] = static_cast<uint32_t>(pos_of_lex[w[e] == 0xffffffffu ? p : w[e] >> cb]);
#pragma unroll
            for (int e = e0; e < e0 + 8; ++e) w[e] = w[e] == 0xffffffffu ? w[e] : (c[e - e0] << cb) | (w[e] & mask);
        }
    }
    sort_registers<P>(w);
    __syncthreads();  // dn, up are read no more
    double sum = 0.0;
#pragma unroll
    for (int a = 0; a < P; ++a) {
        if (a < cnt) {
            sum += table[w[a] & mask];
            run[excl + a] = w[a];
        }
    }
    __syncthreads();
    for (int a = lane; a < total; a += HB_BLOCK) words[wave0 + a] = run[a];
    float v = 0.f;
    for (int i = 0; i < m; ++i) {
        const int ni = s.get(i);
        v += (flags & BH_CONV_REF_INTERACTION) ? static_cast<float>(ni * (ni + 1)) : static_cast<float>((ni * (ni - 1)) / 2);
    }
    if (valid) diag[q] = v;
    // sums and V are not negative: their FP32 bit patterns order like the values
    int mx = valid ? cnt : 0, ms = valid ? __float_as_int(static_cast<float>(sum) * 1.0001f) : 0;
    int lo = valid ? __float_as_int(v) : 0x7f7fffff, hi = valid ? __float_as_int(v) : 0;
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
        mx = max(mx, __shfl_xor(mx, o, 64));
        ms = max(ms, __shfl_xor(ms, o, 64));
        lo = min(lo, __shfl_xor(lo, o, 64));
        hi = max(hi, __shfl_xor(hi, o, 64));
    }
    if (lane == 0) stats[blockIdx.x] = make_int4(mx, ms, lo, hi);
}

// the waves' statistics together (out starts at 0, 0, FLT_MAX, 0): one atomic a workgroup instead of four a row,
// which took 983 us at D = 1,352,078
__global__ void __launch_bounds__(256) k_ham_stats(const int4* __restrict__ stats, int64_t nb, int* __restrict__ out) {
    __shared__ int4 red[4];
    int4 a = make_int4(0, 0, 0x7f7fffff, 0);
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; i < nb; i += static_cast<int64_t>(gridDim.x) * 256) {
        const int4 x = stats[i];
        a = make_int4(max(a.x, x.x), max(a.y, x.y), min(a.z, x.z), max(a.w, x.w));
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1)
        a = make_int4(max(a.x, __shfl_xor(a.x, o, 64)), max(a.y, __shfl_xor(a.y, o, 64)), min(a.z, __shfl_xor(a.z, o, 64)),
                      max(a.w, __shfl_xor(a.w, o, 64)));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = a;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < 4; ++w)
            a = make_int4(max(a.x, red[w].x), max(a.y, red[w].y), min(a.z, red[w].z), max(a.w, red[w].w));
        atomicMax(out, a.x);
        atomicMax(out + 1, a.y);
        atomicMin(out + 2, a.z);
        atomicMax(out + 3, a.w);
    }
}

// Single-particle density matrix rho_ij = <phi| b_i^+ b_j |phi> of a real state, i <= j (the matrix is symmetric), as
// partial sums per workgroup: part[(i m + j) gridDim.x + blockIdx.x].  phi is in lexicographic order, so that
// consecutive threads hold consecutive states and a hop's targets lie close together.  A workgroup takes the rows
// i = NI blockIdx.y .. + NI - 1: a thread unranks its state once for all of them, gets the rank of b_i^+ b_j s as its own
// plus a difference of two prefix sums (as k_ham_fill does), and keeps the sums of its NI m pairs in registers over all its
// states; the wave is summed once at the end.  m = 12, n = 12: 2,290 us, when every pair of every state ranked its target site by
// site and was summed over the wave, to 362 us (387 with four rows: the sums
// then take 128 registers and two waves fit a SIMD).
template <int NW, int BITS, int NI>
__global__ void __launch_bounds__(256) k_spdm(int64_t D, int m, int n, const uint32_t* __restrict__ gg, int gsize,
                                              const double* __restrict__ phi, int nsq, double* __restrict__ part) {
    constexpr int MAXM = PState<NW, BITS>::MAXM;
    extern __shared__ __align__(16) double smem[];
    double* sq = smem;                                          // sqrt(0 .. nsq - 1)
    uint32_t* g = reinterpret_cast<uint32_t*>(smem + nsq);      // gsize words
    __shared__ double red[4][NI * (MAXM + 1)];
    for (int a = threadIdx.x; a < nsq; a += 256) sq[a] = std::sqrt(static_cast<double>(a));
    bh_stage_table(gg, gsize, g);
    const int i0 = blockIdx.y * NI;
    double acc[NI][MAXM], own[NI];
#pragma unroll
    for (int ii = 0; ii < NI; ++ii) {
        own[ii] = 0.0;
#pragma unroll
        for (int j = 0; j < MAXM; ++j) acc[ii][j] = 0.0;
    }
    for (int64_t r = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; r < D; r += static_cast<int64_t>(gridDim.x) * 256) {
        PState<NW, BITS> s;
        bh_unrank(r, m, n, g, s);
        const double pq = phi[r];
        uint32_t dn[MAXM], di[NI];
        int ni[NI];
        {
            int R = n;
            uint32_t d = 0;
#pragma unroll
            for (int ii = 0; ii < NI; ++ii) {
                di[ii] = 0;
                ni[ii] = 0;
            }
#pragma unroll
            for (int l = 0; l < MAXM; ++l) {
                dn[l] = d;
                if (l < m) {
                    const int nl = s.get(l);
#pragma unroll
                    for (int ii = 0; ii < NI; ++ii)
                        if (l == i0 + ii) {  // uniform
                            di[ii] = d;
                            ni[ii] = nl;
                        }
                    R -= nl;
                    if (l < m - 1) {
                        const uint32_t* gl = g + l * (n + 1);
                        const uint32_t g0 = gl[R], gm = gl[max(R - 1, 0)];
                        d += g0 - gm;  // 0 at R = 0
                    }
                }
            }
        }
#pragma unroll
        for (int ii = 0; ii < NI; ++ii) {
            if (i0 + ii >= m) continue;  // uniform
            own[ii] += pq * pq * ni[ii];
            double v[MAXM];
#pragma unroll
            for (int j = 0; j < MAXM; ++j)
                if (j < m && j > i0 + ii) {  // uniform; a source without a boson reads this state again, and adds nothing
                    const uint32_t t = s.get(j) >= 1 ? static_cast<uint32_t>(r) + di[ii] - dn[j] : static_cast<uint32_t>(r);
                    v[j] = phi[t];
                }
#pragma unroll
            for (int j = 0; j < MAXM; ++j)
                if (j < m && j > i0 + ii) {
                    const int c = (ni[ii] + 1) * s.get(j);
                    // no boson on j: the factor is 0, and the product of the amplitudes must not be infinite or NaN
                    // (its low word alone is finite)
                    const double pv = pq * v[j], f = __hiloint2double(s.get(j) >= 1 ? __double2hiint(pv) : 0, __double2loint(pv));
                    acc[ii][j] += f * (nsq ? sq[c] : std::sqrt(static_cast<double>(c)));
                }
        }
    }
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
    for (int ii = 0; ii < NI; ++ii) {
#pragma unroll
        for (int j = 0; j <= MAXM; ++j) {
            if (i0 + ii < m && (j == MAXM || (j < m && j > i0 + ii))) {  // uniform
                double t = j == MAXM ? own[ii] : acc[ii][j < MAXM ? j : 0];
#pragma unroll
                for (int o = 32; o >= 1; o >>= 1) t += __shfl_xor(t, o, 64);
                if (lane == 0) red[wid][ii * (MAXM + 1) + j] = t;
            }
        }
    }
    __syncthreads();
    for (int a = threadIdx.x; a < NI * (MAXM + 1); a += 256) {
        const int i = i0 + a / (MAXM + 1), q = a % (MAXM + 1), j = q == MAXM ? i : q;
        if (i < m && j < m && j >= i && (q == MAXM || q > i))
            part[static_cast<int64_t>(i * m + j) * gridDim.x + blockIdx.x] = (red[0][a] + red[1][a]) + (red[2][a] + red[3][a]);
    }
}

__global__ void __launch_bounds__(256) k_gather_f64(int64_t n, const int32_t* __restrict__ at, const double* __restrict__ x,
                                                    double* __restrict__ y) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (i < n) y[i] = x[at[i]];
}

// out[p] = sum over the nb workgroup partials of pair p = i m + j, in order (one workgroup per pair; j < i: nothing)
__global__ void __launch_bounds__(256) k_spdm_sum(const double* __restrict__ part, int nb, int m, double* __restrict__ out) {
    __shared__ double red[4];
    if (static_cast<int>(blockIdx.x) % m < static_cast<int>(blockIdx.x) / m) return;  // uniform
    double s = 0.0;
    for (int w = threadIdx.x; w < nb; w += 256) s += part[static_cast<int64_t>(blockIdx.x) * nb + w];
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) s += __shfl_xor(s, o, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) out[blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
}

#define BH_LAYOUT_DISPATCH(nw, bits, MACRO)             \
    do {                                                \
        if ((nw) == 1 && (bits) == 4) MACRO(1, 4);      \
        else if ((nw) == 2 && (bits) == 4) MACRO(2, 4); \
        else if ((nw) == 2 && (bits) == 8) MACRO(2, 8); \
        else MACRO(4, 8);                               \
    } while (0)

int bh_ham_rowblocks(bh_ham* h, int B, const int32_t** rb, int64_t* nblocks) {
    auto it = h->rowblocks.find(B);
    if (it != h->rowblocks.end()) {
        *rb = it->second.first;
        *nblocks = it->second.second;
        return BH_OK;
    }
    bh_ctx* ctx = h->ctx;
    const int64_t cap = BH_STAGE_PRODUCTS_HOST / B;
    if (static_cast<int64_t>(h->max_row) > cap) return bh_set_error(ctx, BH_ERANGE, "row longer than a staged block");
    std::vector<int32_t> rp(static_cast<size_t>(h->D + 1));
    BH_HIP(ctx, hipMemcpyAsync(rp.data(), h->row_ptr, rp.size() * 4, hipMemcpyDeviceToHost, ctx->stream));
    BH_HIP(ctx, hipStreamSynchronize(ctx->stream));
    // (first row, first entry) of every block, then (D, nnz): one load gives a block's whole extent
    std::vector<int32_t> blocks;
    auto add = [&](int64_t r) {
        blocks.push_back(static_cast<int32_t>(r));
        blocks.push_back(rp[r]);
    };
    add(0);
    int64_t start = 0;
    for (int64_t r = 0; r < h->D; ++r) {
        if (rp[r + 1] - rp[start] > cap) {
            add(r);
            start = r;
        }
    }
    add(h->D);
    DevArray<int32_t> d;
    BH_TRY(d.alloc(ctx, blocks.size()));
    BH_HIP(ctx, hipMemcpyAsync(d.p, blocks.data(), blocks.size() * 4, hipMemcpyHostToDevice, ctx->stream));
    BH_HIP(ctx, hipStreamSynchronize(ctx->stream));
    const int64_t nb = static_cast<int64_t>(blocks.size()) / 2 - 1;
    h->bytes_rb += blocks.size() * 4;
    h->rowblocks[B] = {d.release(), nb};
    *rb = h->rowblocks[B].first;
    *nblocks = nb;
    return BH_OK;
}

extern "C" int bh_ham_tuned(const bh_ham* h, int kind, int prec, int B, int* variant, int* ncand, int* cand_var,
                            double* cand_us, int cap) {
    if (!h || kind < 0 || kind > 1) return BH_EINVAL;
    std::lock_guard<std::recursive_mutex> lk(h->ctx->mu);
    auto it = h->tuned.find(bh_tune_key(kind, prec, B));
    if (it == h->tuned.end()) return bh_set_error(h->ctx, BH_EINVAL, "sector not used at this (kind, precision, width)");
    if (variant) *variant = it->second.variant;
    const int n = static_cast<int>(it->second.cand.size());
    if (ncand) *ncand = n;
    for (int i = 0; i < n && i < cap; ++i) {
        if (cand_var) cand_var[i] = it->second.cand[i].first;
        if (cand_us) cand_us[i] = it->second.cand[i].second;
    }
    return BH_OK;
}

extern "C" int bh_ham_set_tuned(bh_ham* h, int kind, int prec, int B, int variant) {
    if (!h || kind < 0 || kind > 1) return BH_EINVAL;
    if (!bh_is_pow2_le64(B) || (prec != BH_PREC_FP64 && prec != BH_PREC_MIXED))
        return bh_set_error(h->ctx, BH_EINVAL, "set_tuned: B a power of two <= 64, precision FP64 or MIXED");
    bool ok = false;
    if (variant == 0) ok = static_cast<int64_t>(h->max_row) * B <= BH_STAGE_PRODUCTS_HOST;
    else if (variant == 1 || variant == 2) ok = variant <= B;
    else if (variant == 4) ok = B >= 4 && prec == BH_PREC_MIXED;
    else if (variant == 8) ok = kind == 0 && B >= 8 && prec == BH_PREC_MIXED;
    else if (variant == 17 || variant == 33 || variant == 18 || variant == 34) ok = kind == 0 && (variant & 15) <= B && B <= 16;
    else if (variant == 20) ok = kind == 0 && B >= 4 && B <= 32 && prec == BH_PREC_MIXED;
    else if (variant > 100 && kind == 1) {
        const int G = variant - 100;
        ok = (G & (G - 1)) == 0 && G * B <= 64;
    }
    if (!ok) return bh_set_error(h->ctx, BH_EINVAL, "set_tuned: variant does not fit this sector and width");
    std::lock_guard<std::recursive_mutex> lk(h->ctx->mu);
    BhTuned t;
    t.variant = variant;
    h->tuned[bh_tune_key(kind, prec, B)] = t;
    return BH_OK;
}

int bh_engine_env() {
    static const int env = [] {
        const char* e = std::getenv("BHX_ENGINE");
        return e ? std::atoi(e) : -1;
    }();
    return env;
}

int bh_engine_choice(int B, const bh_ham* h) {
    const int env = bh_engine_env();
    const bool staged_ok = static_cast<int64_t>(h->max_row) * B <= BH_STAGE_PRODUCTS_HOST;
    if (env == 0) return 0;
    if (env == 1) return staged_ok ? 1 : 2;
    if (env == 2) return 2;
    return (B == 1 && staged_ok) ? 1 : 2;
}

static int free_ham(bh_ham* h) {
    bh_ctx* ctx = h->ctx;
    for (auto& kv : h->rowblocks) bh_dev_free(ctx, kv.second.first, static_cast<size_t>(kv.second.second + 1) * 8);
    bh_dev_free(ctx, h->block, h->block_bytes);
    bh_dev_free(ctx, h->lex_of_pos, static_cast<size_t>(h->D) * sizeof(int32_t));
    delete h;
    return BH_OK;
}

// Both precisions read the packed words, so there is nothing to build; the call is what bh_spmv_noalloc asks for.
int bh_ham_prepare_locked(bh_ham* h, int prec) {
    if (prec == BH_PREC_FP64) h->prepared64 = true;
    return BH_OK;
}

extern "C" {

int bh_hamiltonian_build(bh_ctx* ctx, const bh_basis* b, const int* nbr_off, const int* nbr_sites, unsigned flags,
                         bh_ham** out) {
    if (!ctx || !b || !nbr_off || !nbr_sites || !out) return BH_EINVAL;
    *out = nullptr;
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    const int m = b->m, n = b->n;
    const int64_t D = b->D;
    if (flags & ~(BH_CONV_REF_HOP | BH_CONV_REF_INTERACTION)) return bh_set_error(ctx, BH_EINVAL, "hamiltonian: unknown flags");
    // neighbour list: range, no self loops, symmetric as a multiset
    if (nbr_off[0] != 0) return bh_set_error(ctx, BH_EINVAL, "hamiltonian: nbr_off[0] must be 0");
    std::map<std::pair<int, int>, int> mult;  // (i <- j) -> multiplicity
    for (int i = 0; i < m; ++i) {
        if (nbr_off[i + 1] < nbr_off[i]) return bh_set_error(ctx, BH_EINVAL, "hamiltonian: nbr_off not monotone");
        for (int a = nbr_off[i]; a < nbr_off[i + 1]; ++a) {
            const int j = nbr_sites[a];
            if (j < 0 || j >= m) return bh_set_error(ctx, BH_EINVAL, "hamiltonian: neighbour site out of range");
            if (j == i) return bh_set_error(ctx, BH_EINVAL, "hamiltonian: self-loop in the neighbour list");
            mult[{i, j}] += 1;
        }
    }
    for (const auto& kv : mult) {
        auto it = mult.find({kv.first.second, kv.first.first});
        if (it == mult.end() || it->second != kv.second)
            return bh_set_error(ctx, BH_EINVAL, "hamiltonian: neighbour list is not symmetric");
    }
    const int E = static_cast<int>(mult.size());
    if (E > 128) return bh_set_error(ctx, BH_ERANGE, "hamiltonian: more than 128 directed bonds");
    const uint32_t hop = (flags & BH_CONV_REF_HOP) ? 2u : 1u;
    std::vector<int8_t> ei, ej;
    std::vector<uint32_t> cm;
    uint32_t cm_max = 1;
    for (const auto& kv : mult) {
        ei.push_back(static_cast<int8_t>(kv.first.first));
        ej.push_back(static_cast<int8_t>(kv.first.second));
        const uint32_t w = static_cast<uint32_t>(kv.second) * hop;
        cm.push_back(w * w);
        cm_max = std::max(cm_max, w * w);
    }
    // largest (n_i + 1) n_j with n_i + n_j <= n, n_j >= 1
    uint64_t qmax = 0;
    for (int nj = 1; nj <= n; ++nj) qmax = std::max<uint64_t>(qmax, static_cast<uint64_t>(n - nj + 1) * nj);
    const uint64_t code_max = std::max<uint64_t>(1, qmax * cm_max);
    int cb = 0;
    while ((code_max >> cb) != 0) ++cb;
    if (cb > 12 || (D > 1 && static_cast<uint64_t>(D - 1) >> (32 - cb)) != 0)
        return bh_set_error(ctx, BH_ERANGE, "hamiltonian: column and value code do not fit one 32-bit word");
    BH_HIP(ctx, hipSetDevice(ctx->device));
    hipStream_t s = ctx->stream;

    // every directed bond (i, j) contributes an entry per state with a boson on j
    const int64_t per_bond = n >= 1 ? bh_binom_host(m + n - 2, n - 1) : 0;
    if (per_bond < 0 || per_bond > BH_NNZ_MAX || static_cast<int64_t>(E) * per_bond > BH_NNZ_MAX)
        return bh_set_error(ctx, BH_ERANGE, "hamiltonian: number of entries exceeds the int32 index range");
    const int64_t nnz = E * per_bond;
    SiteDeg deg{};
    for (int e = 0; e < E; ++e) deg.d[ej[e]] += 1;
    // longest row possible: the busiest min(m, n) sites occupied
    std::vector<int> dsort(deg.d, deg.d + m);
    std::sort(dsort.rbegin(), dsort.rend());
    int rowcap = 0;
    for (int i = 0; i < std::min(m, n); ++i) rowcap += dsort[i];
    rowcap = std::max(rowcap, 1);
    const int gsize = (m > 1 ? m - 1 : 1) * (n + 1);
    if ((static_cast<size_t>(gsize) + static_cast<size_t>(HB_BLOCK) * (E + 1)) * sizeof(uint32_t) > 64 * 1024) return bh_set_error(ctx, BH_ERANGE, "hamiltonian: rank table too large for LDS");
    const size_t lds_bytes = (static_cast<size_t>(gsize) + static_cast<size_t>(HB_BLOCK) * std::max(rowcap, 2 * m)) * 4;

    std::unique_ptr<bh_ham> hp(new bh_ham());
    bh_ham* h = hp.get();
    h->ctx = ctx;
    h->basis = b;
    h->D = D;
    h->code_bits = cb;
    h->flags = flags;

    // one allocation: table, row pointers, diagonal, words
    const size_t tab = static_cast<size_t>(1) << cb;
    const size_t b_tab = BhScratch::size(tab * 8), b_rp = BhScratch::size(static_cast<size_t>(D + 1) * 4),
                 b_dg = BhScratch::size(static_cast<size_t>(D) * 4), b_w = BhScratch::size(static_cast<size_t>(nnz + BH_WORDS_PAD) * 4);
    DevArray<char> block;
    BH_TRY(block.alloc(ctx, b_tab + b_rp + b_dg + b_w));
    double* table = reinterpret_cast<double*>(block.p);
    int32_t* row_ptr = reinterpret_cast<int32_t*>(block.p + b_tab);
    float* diag = reinterpret_cast<float*>(block.p + b_tab + b_rp);
    uint32_t* words = reinterpret_cast<uint32_t*>(block.p + b_tab + b_rp + b_dg);
    // scratch: the small inputs (one copy), row counts, tile sums, the waves' statistics
    const int64_t ntile = (D + HC_TILE - 1) / HC_TILE;
    const unsigned grid = static_cast<unsigned>((D + HB_BLOCK - 1) / HB_BLOCK);
    const size_t b_in = 16 + static_cast<size_t>(std::max(E, 1)) * 4 + 2 * BhScratch::size(std::max(E, 1));
    BhScratch sc;
    BH_TRY(sc.open(ctx, BhScratch::size(b_in) + BhScratch::size(D) + BhScratch::size(ntile * 8) + BhScratch::size(static_cast<size_t>(grid) * 16)));
    uint8_t* in = sc.take<uint8_t>(b_in);
    uint8_t* cnt = sc.take<uint8_t>(D);
    int64_t* tile = sc.take<int64_t>(ntile);
    int4* wstats = sc.take<int4>(grid);
    std::vector<uint8_t> hin(b_in, 0);  // row statistics' start values, code multipliers, targets, sources
    int stats[4] = {0, 0, 0x7f7fffff, 0};
    const size_t o_i = 16 + static_cast<size_t>(std::max(E, 1)) * 4, o_j = o_i + std::max(E, 1);
    std::memcpy(hin.data(), stats, sizeof(stats));
    for (int e = 0; e < E; ++e) {
        std::memcpy(hin.data() + 16 + 4 * e, &cm[e], 4);
        hin[o_i + e] = static_cast<uint8_t>(ei[e]);
        hin[o_j + e] = static_cast<uint8_t>(ej[e]);
    }
    std::vector<double> htab(tab);
    for (size_t c = 0; c < tab; ++c) htab[c] = std::sqrt(static_cast<double>(c));
    BH_HIP(ctx, hipMemcpyAsync(in, hin.data(), o_j + std::max(E, 1), hipMemcpyHostToDevice, s));
    BH_HIP(ctx, hipMemcpyAsync(table, htab.data(), tab * 8, hipMemcpyHostToDevice, s));
    EdgeArgs ed{E, reinterpret_cast<int8_t*>(in + o_i), reinterpret_cast<int8_t*>(in + o_j), reinterpret_cast<uint32_t*>(in + 16)};
    {
        KTimer kt(ctx, "ham_count", s);
#define LAUNCH_COUNT(NW_, BITS_)                                                                                        \
    hipLaunchKernelGGL((k_ham_count<NW_, BITS_>), dim3(static_cast<unsigned>(ntile)), dim3(HC_BLOCK), gsize * 4, s, D,  \
                       m, n, b->rank_tab, gsize, b->lex_of_pos, deg, cnt, tile)
        BH_LAYOUT_DISPATCH(b->nw, b->bits, LAUNCH_COUNT);
#undef LAUNCH_COUNT
        hipLaunchKernelGGL(k_scan_tiles, dim3(1), dim3(1024), 0, s, tile, ntile);
    }
    BH_HIP(ctx, hipGetLastError());
    {
        KTimer kt(ctx, "ham_fill", s);
        const int32_t* pol = b->order == BH_ORDER_LEX ? nullptr : b->pos_of_lex;
#define FILL(NW_, BITS_, P_)                                                                                            \
    hipLaunchKernelGGL((k_ham_fill<NW_, BITS_, P_>), dim3(grid), dim3(HB_BLOCK), lds_bytes, s, D, m, n, b->rank_tab,    \
                       gsize, b->lex_of_pos, pol, ed, cb, table, flags, cnt, tile, nnz, row_ptr, words, diag, wstats)
#define LAUNCH_FILL(NW_, BITS_)            \
    do {                                   \
        if (E <= 8) FILL(NW_, BITS_, 8);   \
        else if (E <= 16) FILL(NW_, BITS_, 16); \
        else if (E <= 32) FILL(NW_, BITS_, 32); \
        else if (E <= 64) FILL(NW_, BITS_, 64); \
        else FILL(NW_, BITS_, 128);        \
    } while (0)
        BH_LAYOUT_DISPATCH(b->nw, b->bits, LAUNCH_FILL);
#undef LAUNCH_FILL
#undef FILL
        hipLaunchKernelGGL(k_ham_stats, dim3(std::min<unsigned>(64, (grid + 255) / 256)), dim3(256), 0, s, wstats,
                           static_cast<int64_t>(grid), reinterpret_cast<int*>(in));
    }
    BH_HIP(ctx, hipGetLastError());
    BH_HIP(ctx, hipMemcpyAsync(stats, in, sizeof(stats), hipMemcpyDeviceToHost, s));
    DevArray<int32_t> lop;
    if (bh_basis_lex_start(b)) {
        BH_TRY(lop.alloc(ctx, static_cast<size_t>(D)));
        BH_HIP(ctx, hipMemcpyAsync(lop.p, b->lex_of_pos, static_cast<size_t>(D) * sizeof(int32_t), hipMemcpyDeviceToDevice, s));
    }
    BH_HIP(ctx, hipStreamSynchronize(s));
    auto as_f = [](int v) {
        float f;
        std::memcpy(&f, &v, 4);
        return static_cast<double>(f);
    };
    h->nnz = nnz;
    h->max_row = stats[0];
    h->tmax = as_f(stats[1]);
    h->vmin = as_f(stats[2]);
    h->vmax = as_f(stats[3]);
    h->row_ptr = row_ptr;
    h->words = words;
    h->diag = diag;
    h->table = table;
    h->block_bytes = block.bytes();
    h->block = block.release();
    h->bytes = static_cast<size_t>(D + 1) * 4 + static_cast<size_t>(nnz ? nnz : 1) * 4 + static_cast<size_t>(D) * 4 +
               tab * 8;
    if (bh_basis_lex_start(b)) {
        h->lex_of_pos = lop.release();
        h->layout_id = b->layout_id;
        h->bytes += static_cast<size_t>(D) * 4;
    }
    *out = hp.release();
    return BH_OK;
}

int bh_ham_destroy(bh_ham* h) {
    if (!h) return BH_EINVAL;
    bh_ctx* ctx = h->ctx;
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    (void)hipSetDevice(ctx->device);
    (void)hipStreamSynchronize(ctx->stream);
    return free_ham(h);
}

int64_t bh_ham_dim(const bh_ham* h) { return h ? h->D : -1; }
int64_t bh_ham_nnz(const bh_ham* h) { return h ? h->nnz : -1; }
int64_t bh_ham_device_bytes(const bh_ham* h) { return h ? static_cast<int64_t>(h->bytes + h->bytes_rb) : -1; }

int bh_ham_prepare(bh_ham* h, int prec) {
    if (!h) return BH_EINVAL;
    std::lock_guard<std::recursive_mutex> lk(h->ctx->mu);
    BH_HIP(h->ctx, hipSetDevice(h->ctx->device));
    return bh_ham_prepare_locked(h, prec);
}

int bh_ham_copy_packed(const bh_ham* h, uint32_t* words, int* code_bits) {
    if (!h) return BH_EINVAL;
    bh_ctx* ctx = h->ctx;
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    BH_HIP(ctx, hipSetDevice(ctx->device));
    if (code_bits) *code_bits = h->code_bits;
    if (words && h->nnz)
        BH_HIP(ctx, hipMemcpyAsync(words, h->words, static_cast<size_t>(h->nnz) * 4, hipMemcpyDeviceToHost, ctx->stream));
    BH_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return BH_OK;
}

int bh_ham_copy_csr(const bh_ham* h, int64_t* row_ptr, int32_t* col, double* val, double* diag) {
    if (!h) return BH_EINVAL;
    bh_ctx* ctx = h->ctx;
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    BH_HIP(ctx, hipSetDevice(ctx->device));
    hipStream_t s = ctx->stream;
    if (row_ptr) {
        std::vector<int32_t> rp(static_cast<size_t>(h->D + 1));
        BH_HIP(ctx, hipMemcpyAsync(rp.data(), h->row_ptr, rp.size() * 4, hipMemcpyDeviceToHost, s));
        BH_HIP(ctx, hipStreamSynchronize(s));
        for (size_t i = 0; i < rp.size(); ++i) row_ptr[i] = rp[i];
    }
    if ((col || val) && h->nnz) {
        std::vector<uint32_t> w(static_cast<size_t>(h->nnz));
        BH_HIP(ctx, hipMemcpyAsync(w.data(), h->words, w.size() * 4, hipMemcpyDeviceToHost, s));
        BH_HIP(ctx, hipStreamSynchronize(s));
        const uint32_t mask = (1u << h->code_bits) - 1u;
        for (size_t k = 0; k < w.size(); ++k) {
            if (col) col[k] = static_cast<int32_t>(w[k] >> h->code_bits);
            if (val) val[k] = -std::sqrt(static_cast<double>(w[k] & mask));
        }
    }
    if (diag) {
        std::vector<float> d(static_cast<size_t>(h->D));
        BH_HIP(ctx, hipMemcpyAsync(d.data(), h->diag, d.size() * 4, hipMemcpyDeviceToHost, s));
        BH_HIP(ctx, hipStreamSynchronize(s));
        for (size_t i = 0; i < d.size(); ++i) diag[i] = d[i];
    }
    return BH_OK;
}

// Single-particle density matrix of one state (Analysis::SPDM / braket, src/analysis.cpp:497-512, 562-594).
int bh_spdm(bh_ctx* ctx, const bh_basis* b, const double* phi, double* rho) {
    if (!ctx || !b || !phi || !rho) return BH_EINVAL;
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    BH_HIP(ctx, hipSetDevice(ctx->device));
    hipStream_t s = ctx->stream;
    const int m = b->m, n = b->n;
    const int64_t D = b->D;
    if (m < 1) return bh_set_error(ctx, BH_EINVAL, "spdm: empty lattice");
    const int gsize = (m > 1 ? m - 1 : 1) * (n + 1);
    if (static_cast<size_t>((gsize + 1) & ~1) * 4 + static_cast<size_t>(m) * m * 8 > 64 * 1024)
        return bh_set_error(ctx, BH_ERANGE, "spdm: rank table too large for LDS");
    // amplitudes from a table while it is small (n <= 62): (n_i + 1) n_j is largest at the half filling of the pair
    const int top = ((n + 1) / 2) * (n + 1 - (n + 1) / 2) + 1;
    const int nsq = top <= 1024 ? top : 0;
    const size_t lds_bytes = static_cast<size_t>(nsq) * 8 + static_cast<size_t>(gsize) * 4;
    const int nb = static_cast<int>(std::min<int64_t>((D + 255) / 256, 768));
    const bool lex = b->order == BH_ORDER_LEX;
    const size_t vb = BhScratch::size(D * 8), sums = BhScratch::size(static_cast<size_t>(m) * m * nb * 8) + BhScratch::size(static_cast<size_t>(m) * m * 8);
    BhScratch sc;
    int rc = sc.open(ctx, vb * (lex ? 1 : 2) + sums);
    // where there is no room for a second vector the host brings phi into lexicographic order
    const bool host = rc != BH_OK && !lex;
    if (host) {
        (void)hipGetLastError();
        rc = sc.open(ctx, vb + sums);
    }
    if (rc != BH_OK) return rc;
    double* dphi = sc.take<double>(D);
    double* part = sc.take<double>(static_cast<size_t>(m) * m * nb);
    double* out = sc.take<double>(static_cast<size_t>(m) * m);
    std::vector<double> hphi;
    if (host) {
        std::vector<int32_t> pol(static_cast<size_t>(D));
        hphi.resize(static_cast<size_t>(D));
        BH_HIP(ctx, hipMemcpyAsync(pol.data(), b->pos_of_lex, pol.size() * sizeof(int32_t), hipMemcpyDeviceToHost, s));
        BH_HIP(ctx, hipStreamSynchronize(s));
        for (int64_t r = 0; r < D; ++r) hphi[r] = phi[pol[r]];
    }
    BH_HIP(ctx, hipMemcpyAsync(dphi, host ? hphi.data() : phi, static_cast<size_t>(D) * 8, hipMemcpyHostToDevice, s));
    if (!lex && !host) {
        double* pl = sc.take<double>(D);
        hipLaunchKernelGGL(k_gather_f64, dim3(static_cast<unsigned>((D + 255) / 256)), dim3(256), 0, s, D, b->pos_of_lex, dphi, pl);
        dphi = pl;
    }
#define LAUNCH_SPDM(NW_, BITS_)                                                                                       \
    do {                                                                                                              \
        constexpr int NI = PState<NW_, BITS_>::MAXM == 16 ? 2 : 1;                                                    \
        hipLaunchKernelGGL((k_spdm<NW_, BITS_, NI>), dim3(nb, (m + NI - 1) / NI), dim3(256), lds_bytes, s, D, m, n,   \
                           b->rank_tab, gsize, dphi, nsq, part);                                                      \
    } while (0)
    BH_LAYOUT_DISPATCH(b->nw, b->bits, LAUNCH_SPDM);
#undef LAUNCH_SPDM
    hipLaunchKernelGGL(k_spdm_sum, dim3(m * m), dim3(256), 0, s, part, nb, m, out);
    BH_HIP(ctx, hipGetLastError());
    BH_HIP(ctx, hipMemcpyAsync(rho, out, static_cast<size_t>(m) * m * 8, hipMemcpyDeviceToHost, s));
    BH_HIP(ctx, hipStreamSynchronize(s));
    for (int i = 0; i < m; ++i)
        for (int j = 0; j < i; ++j) rho[i * m + j] = rho[j * m + i];
    return BH_OK;
}

}  // extern "C"
