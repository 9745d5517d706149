// bh_meanfield.hip -- batched self-consistent mean-field solves of the Bose-Hubbard model (gfx950).
//
// Replaces Analysis::SCMF / Analysis::SF_density (src/analysis.cpp:95-178) and BH::h_MF
// (src/hamiltonian.cpp:290-309).  Each (mu, J) point is an independent fixed-point iteration on psi, each
// step a sequence of ground states of the tridiagonal single-site Hamiltonian h_MF on 2p+1 occupations
// (p = 1, 2, ... until the ground energy moves by at most eps).  The work is scalar FP64 with a
// data-dependent trip count per point (23 iterations on average, thousands next to the Mott-lobe boundary), so
// one thread carries one point and lanes are refilled as points finish; the points that will take longest start first
// (k_scmf).
//
// Arithmetic: every expression keeps one fixed operand order and the file's functions are compiled without
// floating-point contraction, so each result is a fixed sequence of correctly rounded IEEE operations
// (+, -, *, / and the sqrt(i) table computed on the host).  A ground state needs only a few O(2p+1) pivot
// recurrences (no eigenvector): a point's state lives in registers and one column of LDS (its diagonal).
#include <algorithm>
#include <cmath>
#include <vector>

#include "bh_internal.hpp"

namespace {

constexpr int MF_PMAX = 32;             // largest p a point may reach: h_MF on 65 occupations
constexpr int MF_NMAX = 2 * MF_PMAX + 1;
constexpr int MF_WG = 256;
constexpr int MF_NR = 9;                // diagonal entries of a lane in registers: p <= 4, most points up to mu = 4
constexpr int MF_NL = 15;               // diagonal entries a lane keeps in LDS (five workgroups a CU); p <= 7, all but rare points

__device__ __forceinline__ double mf_diag(int i, double mu, double w) {
#pragma clang fp contract(off)
    return -mu * static_cast<double>(i) + 0.5 * static_cast<double>(i) * static_cast<double>(i - 1) + w;
}

// LDL^T pivots u_i of T - x I and their x-derivatives: true when every pivot is positive (x below the lowest
// eigenvalue), with S = sum_i u_i'/u_i = d/dx ln det(T - x I).  Squared couplings e_{i-1}^2 = c^2 i (c2 = c^2).
//   u_0 = d_0 - x, u_i = (d_i - x) - e_{i-1}^2 / u_{i-1};  u_0' = -1, u_i' = -1 + e_{i-1}^2 u_{i-1}' / u_{i-1}^2
__device__ bool mf_pivots(int N, double mu, double w, double c2, double x, double& S) {
#pragma clang fp contract(off)
    double u = mf_diag(0, mu, w) - x, du = -1.0;
    if (!(u > 0.0)) return false;
    double r = 1.0 / u;
    double s = du * r;
    for (int i = 1; i < N; ++i) {
        const double ee = c2 * static_cast<double>(i);
        du = -1.0 + ee * du * r * r;
        u = (mf_diag(i, mu, w) - x) - ee * r;
        if (!(u > 0.0)) return false;
        r = 1.0 / u;
        s = s + du * r;
    }
    S = s;
    return true;
}

// 1 / u, correctly rounded, for |u| with an exponent in [-511, 512], where no intermediate value leaves the normal
// range: the hardware's estimate, two Newton steps and a residual correction by fused multiply-add (Markstein, IBM J.
// Res. Dev. 34, 111-119, 1990).  Equal to 1.0 / u bit for bit at 2.0e10 values of u over these exponents, both signs,
// mantissas next to 1 and to 2 among them.
__device__ __forceinline__ double mf_rcp(double u) {
#pragma clang fp contract(off)
    double y = __builtin_amdgcn_rcp(u);
    y = fma(y, fma(-u, y, 1.0), y);
    y = fma(y, fma(-u, y, 1.0), y);
    return fma(fma(-u, y, 1.0), y, y);
}

// Range of a pivot, by its high word less 2^29: below MF_MID, positive with an exponent in [-511, 512]; from MF_NEG
// below MF_TINY, negative; otherwise zero, tiny, huge or NaN.  The largest over a sweep tells what it met.
constexpr unsigned MF_MID = 0x40000000u, MF_NEG = 0x60000000u, MF_TINY = 0xe0000000u;
__device__ __forceinline__ unsigned mf_range(double u) { return static_cast<unsigned>(__double2hiint(u)) - 0x20000000u; }

// mf_pivots for N <= MF_NR on entries in registers, the same operations without a branch per pivot:
// 1 all pivots positive, 0 one is not (S then unused), -1 left to mf_pivots.  A sweep is one chain of dependent FP64
// operations, alone on its SIMD for most of the launch, so its length is the kernel's time: unrolled in pairs (N is
// odd), nothing but the pivots' own recurrence is left on it (a loop with the entries in LDS waits for each one).
__device__ __forceinline__ int mf_sweep_r(int N, const double (&d)[MF_NR], double c2, double x, double& S) {
#pragma clang fp contract(off)
    double u = d[0] - x, du = -1.0, r = mf_rcp(u), s = du * r;
    unsigned t = mf_range(u);
    auto step = [&](int i) {
#pragma clang fp contract(off)
        const double ee = c2 * static_cast<double>(i);
        du = -1.0 + ee * du * r * r;
        u = (d[i] - x) - ee * r;
        t = max(t, mf_range(u));
        r = mf_rcp(u);
        s = s + du * r;
    };
    step(1);
    step(2);
    if (N > 3) {
        step(3);
        step(4);
        if (N > 5) {
            step(5);
            step(6);
            if (N > 7) {
                step(7);
                step(8);
            }
        }
    }
    S = s;
    return t < MF_MID ? 1 : (t >= MF_NEG && t < MF_TINY ? 0 : -1);
}

// the same for N <= MF_NL on the entries d[0], d[MF_WG], ... of this lane in LDS
__device__ __forceinline__ int mf_sweep(int N, const double* d, double c2, double x, double& S) {
#pragma clang fp contract(off)
    double u = d[0] - x, du = -1.0, r = mf_rcp(u), s = du * r, f = 0.0;
    unsigned t = mf_range(u);
    for (int i = 1; i < N; ++i) {
        f = f + 1.0;
        const double ee = c2 * f;
        du = -1.0 + ee * du * r * r;
        u = (d[i * MF_WG] - x) - ee * r;
        t = max(t, mf_range(u));
        r = mf_rcp(u);
        s = s + du * r;
    }
    S = s;
    return t < MF_MID ? 1 : (t >= MF_NEG && t < MF_TINY ? 0 : -1);
}

// Logarithmic derivatives of det(T - x I) in x and in the coupling scale c (diagonal held fixed) at two points
// x1, x2 at once (two independent recurrences interleaved); ok1 / ok2 tell whether every pivot was positive.
// d(e_{i-1}^2)/dc = 2 c i (tc = 2c);  u_i'(c) = -(2 c i) / u_{i-1} + e_{i-1}^2 u_{i-1}'(c) / u_{i-1}^2.
__device__ void mf_logdet_deriv2(int N, double mu, double w, double c2, double tc, double x1, double x2, bool& ok1,
                                 bool& ok2, double& Sx1, double& Sc1, double& Sx2, double& Sc2) {
#pragma clang fp contract(off)
    const double d0 = mf_diag(0, mu, w);
    double u1 = d0 - x1, u2 = d0 - x2, dux1 = -1.0, dux2 = -1.0, duc1 = 0.0, duc2 = 0.0;
    ok1 = u1 > 0.0;
    ok2 = u2 > 0.0;
    double r1 = 1.0 / u1, r2 = 1.0 / u2;
    double sx1 = dux1 * r1, sx2 = dux2 * r2, sc1 = 0.0, sc2 = 0.0;
    for (int i = 1; i < N && (ok1 || ok2); ++i) {
        const double ee = c2 * static_cast<double>(i);
        const double dee = tc * static_cast<double>(i);
        const double di = mf_diag(i, mu, w);
        dux1 = -1.0 + ee * dux1 * r1 * r1;
        dux2 = -1.0 + ee * dux2 * r2 * r2;
        duc1 = -(dee * r1) + ee * duc1 * r1 * r1;
        duc2 = -(dee * r2) + ee * duc2 * r2 * r2;
        u1 = (di - x1) - ee * r1;
        u2 = (di - x2) - ee * r2;
        ok1 = ok1 && u1 > 0.0;
        ok2 = ok2 && u2 > 0.0;
        r1 = 1.0 / u1;
        r2 = 1.0 / u2;
        sx1 = sx1 + dux1 * r1;
        sx2 = sx2 + dux2 * r2;
        sc1 = sc1 + duc1 * r1;
        sc2 = sc2 + duc2 * r2;
    }
    Sx1 = sx1;
    Sc1 = sc1;
    Sx2 = sx2;
    Sc2 = sc2;
}

// mf_logdet_deriv2 for N <= MF_NR without branches: true when every pivot of both points is positive and in the range of
// mf_rcp, else left to mf_logdet_deriv2.
__device__ __forceinline__ bool mf_logdet_deriv2_r(int N, double mu, double w, double c2, double tc, double x1, double x2,
                                                   double& Sx1, double& Sc1, double& Sx2, double& Sc2) {
#pragma clang fp contract(off)
    const double d0 = mf_diag(0, mu, w);
    double u1 = d0 - x1, u2 = d0 - x2, dux1 = -1.0, dux2 = -1.0, duc1 = 0.0, duc2 = 0.0;
    unsigned t = max(mf_range(u1), mf_range(u2));
    double r1 = mf_rcp(u1), r2 = mf_rcp(u2);
    double sx1 = dux1 * r1, sx2 = dux2 * r2, sc1 = 0.0, sc2 = 0.0;
    auto step = [&](int i) {
#pragma clang fp contract(off)
        const double ee = c2 * static_cast<double>(i);
        const double dee = tc * static_cast<double>(i);
        const double di = mf_diag(i, mu, w);
        dux1 = -1.0 + ee * dux1 * r1 * r1;
        dux2 = -1.0 + ee * dux2 * r2 * r2;
        duc1 = -(dee * r1) + ee * duc1 * r1 * r1;
        duc2 = -(dee * r2) + ee * duc2 * r2 * r2;
        u1 = (di - x1) - ee * r1;
        u2 = (di - x2) - ee * r2;
        t = max(t, max(mf_range(u1), mf_range(u2)));
        r1 = mf_rcp(u1);
        r2 = mf_rcp(u2);
        sx1 = sx1 + dux1 * r1;
        sx2 = sx2 + dux2 * r2;
        sc1 = sc1 + duc1 * r1;
        sc2 = sc2 + duc2 * r2;
    };
    step(1);
    step(2);
    if (N > 3) {
        step(3);
        step(4);
        if (N > 5) {
            step(5);
            step(6);
            if (N > 7) {
                step(7);
                step(8);
            }
        }
    }
    Sx1 = sx1;
    Sc1 = sc1;
    Sx2 = sx2;
    Sc2 = sc2;
    return t < MF_MID;
}

// Ground state of h_MF(psi, p):  d_i = -mu i + i(i-1)/2 + q J psi^2,  h(i, i+1) = c sqrt(i+1), c = -q J psi.
// Returns its energy, in registers (beyond MF_NR entries the lane's LDS column d; no eigenvector is formed).
// Energy: Newton's iteration on ln det(T - x I) from below (x <- x - 1/S).  Every root is real, so each exact
// step from below the lowest root stays below it and the iterates rise monotonically to it (quadratically
// once close).  Starts at `hint` when its pivots are all positive (the previous p's eigenvalue less 1e-3
// (|lambda| + 1): more occupations only lower it), else at the Gershgorin lower bound; hi = min_i d_i, or the
// rejected hint, lies at or above the root.  An iterate without all pivots positive, or a step reaching hi,
// can only come from rounding at the root: that iterate (resp. hi) is returned, as is the last iterate when
// a step no longer moves x.
// c = 0 (diagonal h): the first smallest diagonal entry.
__device__ double mf_ground(double psi, int p, double mu, double J, int q, const double* __restrict__ sq, double hint, double* d) {
#pragma clang fp contract(off)
    const int N = 2 * p + 1;
    const double c = static_cast<double>(-q) * J * psi;
    const double w = static_cast<double>(q) * J * psi * psi;
    double lo = 0.0, hi = 0.0, top = 0.0;
    double dr[MF_NR];
    auto entry = [&](int i, double di) {
#pragma clang fp contract(off)
        const double a0 = i > 0 ? fabs(c * sq[i]) : 0.0;
        const double a1 = i < N - 1 ? fabs(c * sq[i + 1]) : 0.0;
        const double g = di - a0 - a1;
        if (i == 0 || g < lo) lo = g;
        if (i == 0 || di < hi) hi = di;
        top = fmax(top, fabs(di));
    };
#pragma unroll
    for (int i = 0; i < MF_NR; ++i) {
        dr[i] = mf_diag(i, mu, w);
        if (i < 3 || i < N) entry(i, dr[i]);
    }
    if (N > MF_NR) {
        for (int i = 0; i < N; ++i) {
            const double di = mf_diag(i, mu, w);
            if (i < MF_NL) d[i * MF_WG] = di;
            if (i >= MF_NR) entry(i, di);
        }
    }
    if (c == 0.0) return hi;
    const double c2 = c * c;
    // the sweeps without range checks on d_i - x: no pivot above 2^512 while those before it are positive
    const bool fast = N <= MF_NL && top < 0x1p400 && fabs(lo) < 0x1p400;
    auto pivots = [&](double x, double& S) -> bool {
        if (fast) {
            const int k = N <= MF_NR ? mf_sweep_r(N, dr, c2, x, S) : mf_sweep(N, d, c2, x, S);
            if (k >= 0) return k == 1;
        }
        return mf_pivots(N, mu, w, c2, x, S);
    };
    // One loop for the starts and the Newton steps, so that lanes at different p sweep together.  0: at the hint; 1: at
    // the Gershgorin bound, moved down up to 64 times if rounding put it at the eigenvalue; 2: Newton.  The
    // evaluation of a start is Newton's first.
    int phase = hint > lo && hint < hi ? 0 : 1, tries = 0, it = 0;
    double xk = phase == 0 ? hint : lo, lam = xk;
    for (;;) {
        double S = 0.0;
        if (!pivots(xk, S)) {
            if (phase == 2) break;  // a Newton iterate at the root within rounding
            if (phase == 0) {
                hi = hint;
                phase = 1;
            } else {
                lo = lo - (fabs(lo) + 1.0);
                if (++tries == 64) phase = 2;
            }
            xk = lo;
            lam = xk;
            continue;
        }
        phase = 2;
        const double xn = xk - (mf_range(fabs(S)) < MF_MID ? mf_rcp(S) : 1.0 / S);
        if (!(xn < hi)) {  // the root lies at hi within rounding
            lam = hi;
            break;
        }
        if (!(xn > xk)) break;  // no progress
        xk = xn;
        lam = xk;
        if (++it == 200) break;
    }
    return lam;
}

// <a> of the ground state with energy lam: Hellmann-Feynman, d lambda/dc = 2 sum_i sqrt(i+1) phi_i phi_{i+1} = 2 <a> and
// d lambda/dc = -(d ln det/dc) / (d ln det/dx) as x -> lambda; the ratio is taken at lambda - delta and
// lambda - 2 delta, delta = 1e-9 (|lambda| + 1), and extrapolated linearly to lambda (O(delta^2) error).
// Only the last p of an iteration needs it.  c = 0 (diagonal h): 0.
__device__ double mf_order(double psi, int p, double mu, double J, int q, double lam) {
#pragma clang fp contract(off)
    const int N = 2 * p + 1;
    const double c = static_cast<double>(-q) * J * psi;
    const double w = static_cast<double>(q) * J * psi * psi;
    if (c == 0.0) return 0.0;
    const double c2 = c * c, tc = 2.0 * c;
    double delta = 1e-9 * (fabs(lam) + 1.0);
    for (int t = 0; t < 8; ++t) {
        double sx1, sc1, sx2, sc2;
        bool ok1 = true, ok2 = true;
        if (N > MF_NR || !mf_logdet_deriv2_r(N, mu, w, c2, tc, lam - delta, lam - 2.0 * delta, sx1, sc1, sx2, sc2))
            mf_logdet_deriv2(N, mu, w, c2, tc, lam - delta, lam - 2.0 * delta, ok1, ok2, sx1, sc1, sx2, sc2);
        if (ok1 && ok2) {
            const double f1 = -0.5 * sc1 / sx1;
            const double f2 = -0.5 * sc2 / sx2;
            return 2.0 * f1 - f2;
        }
        delta = 2.0 * delta;
    }
    return 0.0;
}

// the start for p + 1 after the eigenvalue e of p
__device__ __forceinline__ double mf_hint(double e) {
#pragma clang fp contract(off)
    return e - 1e-3 * (fabs(e) + 1.0);
}

// ---- which points first ----------------------------------------------------------------------------------
// Near the lobe boundary an iteration scales psi by about J / J_c, so a point takes of the order of
// ln(1/eps) / |ln(J / J_c)| iterations; q J_c = (g - mu)(mu - g + 1)/(mu + 1), g = ceil(mu) (second-order perturbation
// theory of the unit cell).  Points are counted into classes of the power of two of |J / J_c - 1|, nearest first.
// Only the order of the work depends on this.
constexpr int MF_CLASSES = 16;

__device__ __forceinline__ int mf_class(double mu, double J, int q) {
    const double g = fmax(ceil(mu), 0.0);
    const double jc = (g - mu) * (mu - g + 1.0) / (mu + 1.0);
    const double d = fabs(static_cast<double>(q) * J / jc - 1.0);
    if (!(d < 1.0)) return MF_CLASSES - 1;
    const int e = static_cast<int>((static_cast<unsigned>(__double2hiint(d)) >> 20) & 0x7ff) - 1023;  // 2^e <= d < 2^(e + 1)
    return max(e, -(MF_CLASSES - 1)) + MF_CLASSES - 1;
}

// count[c]: points of class c
__global__ void __launch_bounds__(256) k_scmf_count(int64_t npts, const double* __restrict__ mu, const double* __restrict__ J, int q,
                                                    unsigned* __restrict__ count) {
    __shared__ unsigned cnt[MF_CLASSES];
    if (threadIdx.x < MF_CLASSES) cnt[threadIdx.x] = 0;
    __syncthreads();
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; i < npts; i += static_cast<int64_t>(gridDim.x) * 256)
        atomicAdd(&cnt[mf_class(mu[i], J[i], q)], 1u);
    __syncthreads();
    if (threadIdx.x < MF_CLASSES && cnt[threadIdx.x]) atomicAdd(count + threadIdx.x, cnt[threadIdx.x]);
}

// ord: the points class by class, in any order within one (taken[c]: places of class c given out)
__global__ void __launch_bounds__(256) k_scmf_order(int64_t npts, const double* __restrict__ mu, const double* __restrict__ J, int q,
                                                    const unsigned* __restrict__ count, unsigned* __restrict__ taken,
                                                    uint32_t* __restrict__ ord) {
    __shared__ unsigned cnt[MF_CLASSES], base[MF_CLASSES];
    if (threadIdx.x < MF_CLASSES) cnt[threadIdx.x] = 0;
    __syncthreads();
    const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    int c = 0;
    unsigned r = 0;
    if (i < npts) {
        c = mf_class(mu[i], J[i], q);
        r = atomicAdd(&cnt[c], 1u);
    }
    __syncthreads();
    if (threadIdx.x < MF_CLASSES) {
        unsigned b = 0;
        for (int t = 0; t < static_cast<int>(threadIdx.x); ++t) b += count[t];
        base[threadIdx.x] = b + (cnt[threadIdx.x] ? atomicAdd(taken + threadIdx.x, cnt[threadIdx.x]) : 0u);
    }
    __syncthreads();
    if (i < npts) ord[base[c] + r] = static_cast<uint32_t>(i);
}

constexpr int MF_NEXT = 1 + MF_CLASSES;  // 64-bit words: the claim counter, then count and taken of the classes

// How the points are dealt out at the start: wavefronts below w1 take c1 points each, those below w2 c2, the others c3;
// the points after these `first` are claimed from a counter.
struct MfDeal {
    int w1, w2, c1, c2, c3;
    int64_t first;
};

// Analysis::SCMF with its two stopping rules (ground energy over p, psi over the self-consistency loop),
// U = 1, as a per-lane state machine: every pass of the loop is one ground state per lane, after which the
// lane either moves to the next p, starts the next self-consistency iteration, or finishes its point (status
// 0 converged, 1 max_outer iterations reached with psi the last iterate, 2 p would exceed pmax) and takes the
// next unclaimed point in wavefront batches from *next (zero at launch).  A wavefront leaves the loop when none of its
// lanes holds a point.
// A pass lasts as long as its slowest lane's, and the launch as long as the slowest point's chain of passes (some 2,200
// iterations on the reference's 1000 x 1000 grid, 26 to 31 ms alone: about 18 sweeps and 108 pivots an iteration, a
// pivot some 25 instructions of 5 cycles).  So the points nearest to the lobe boundary start first,
// one to a wavefront and ahead of the others in the SIMD's arbitration, the next ones a few to a wavefront; such a
// wavefront takes full loads once its first points are done.  The grid is what is resident at a time, four wavefronts
// per SIMD (128 VGPRs).  1000 x 1000: 64 ms in the order of the grid with half of the workgroups waiting for the end of
// the others, 53 so, 40 with the sweeps in registers.
__global__ void __launch_bounds__(MF_WG) __attribute__((amdgpu_waves_per_eu(4))) k_scmf(int64_t npts, const double* __restrict__ mu_in,
                                                const double* __restrict__ J_in, const double* __restrict__ psi0,
                                                const uint32_t* __restrict__ ord, MfDeal deal, int q, double eps, int max_outer,
                                                int pmax, const double* __restrict__ sq_in, double* __restrict__ psi_out,
                                                int32_t* __restrict__ status_out, int32_t* __restrict__ iters_out,
                                                int32_t* __restrict__ p_out, unsigned long long* __restrict__ next) {
#pragma clang fp contract(off)
    __shared__ double sq[MF_NMAX + 1];
    __shared__ double dl[MF_NL * MF_WG];
    for (int i = threadIdx.x; i <= MF_NMAX; i += MF_WG) sq[i] = sq_in[i];
    __syncthreads();
    double* d = dl + threadIdx.x;
    const int lane = static_cast<int>(__lane_id());
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(blockIdx.x) * (MF_WG / 64) + static_cast<int>(threadIdx.x >> 6));
    // lanes of this wavefront that take points, and its first place in the order
    int cap = wave < deal.w1 ? deal.c1 : (wave < deal.w2 ? deal.c2 : deal.c3);
    int64_t slot = static_cast<int64_t>(min(wave, deal.w1)) * deal.c1 +
                   static_cast<int64_t>(max(min(wave, deal.w2) - deal.w1, 0)) * deal.c2 +
                   static_cast<int64_t>(max(wave - deal.w2, 0)) * deal.c3 + lane;
    if (wave < deal.w1) __builtin_amdgcn_s_setprio(3);
    else if (wave < deal.w2) __builtin_amdgcn_s_setprio(2);
    int64_t k = 0;
    double mu = 0.0, J = 0.0, psi = 0.0, e0 = 0.0;
    int p = 1, outer = 1;
    bool have = lane < cap && slot < npts, exhausted = false;
    if (have) {
        k = ord ? static_cast<int64_t>(ord[slot]) : slot;
        mu = mu_in[k];
        J = J_in[k];
        psi = psi0[k];
    }
    for (;;) {
        if (have) {
            const double e = mf_ground(psi, p, mu, J, q, sq, p == 1 ? -INFINITY : mf_hint(e0), d);
            int status = -1;
            if (p == 1) {
                e0 = e;
                p = 2;
            } else {
                const double tmp = fabs(e0 - e);
                e0 = e;
                if (tmp > eps) {
                    if (p + 1 > pmax)
                        status = 2;
                    else
                        ++p;
                } else {
                    const double sf = mf_order(psi, p, mu, J, q, e);
                    const double dpsi = fabs(sf - psi);
                    psi = sf;
                    if (dpsi <= eps) {
                        status = 0;
                    } else if (outer >= max_outer) {
                        status = 1;
                    } else {
                        ++outer;
                        p = 1;
                    }
                }
            }
            if (status >= 0) {
                psi_out[k] = psi;
                status_out[k] = status;
                iters_out[k] = outer;
                p_out[k] = p;
                have = false;
            }
        }
        if (cap < 64 && !__ballot(have)) {  // the first points are done: a wavefront like the others
            cap = 64;
            __builtin_amdgcn_s_setprio(0);
        }
        // refill: the lanes without a point claim consecutive points with one atomic per wavefront
        const bool want = cap == 64 && !have && !exhausted;
        const unsigned long long need = __ballot(want);
        if (need) {
            const int cnt = __popcll(need);
            const int leader = __ffsll(static_cast<long long>(need)) - 1;
            unsigned long long base = 0;
            if (lane == leader) base = atomicAdd(next, static_cast<unsigned long long>(cnt));
            base = __shfl(base, leader);
            if (want) {
                const int rank = __popcll(need & ((1ull << lane) - 1ull));
                slot = deal.first + static_cast<int64_t>(base) + rank;
                if (slot < npts) {
                    have = true;
                    k = ord ? static_cast<int64_t>(ord[slot]) : slot;
                    mu = mu_in[k];
                    J = J_in[k];
                    psi = psi0[k];
                    p = 1;
                    outer = 1;
                } else {
                    exhausted = true;
                }
            }
        }
        if (!__ballot(have)) break;
    }
}

}  // namespace

extern "C" {

int bh_mean_field(bh_ctx* ctx, int64_t npts, const double* mu, const double* J, const double* psi0, int q,
                  double eps, int max_outer, int pmax, double* psi, int32_t* status, int32_t* iters,
                  int32_t* p_last) {
    if (!ctx) return BH_EINVAL;
    if (npts < 0 || (npts > 0 && (!mu || !J || !psi0 || !psi)))
        return bh_set_error(ctx, BH_EINVAL, "mean_field: need npts >= 0 and the mu, J, psi0, psi arrays");
    if (pmax < 2 || pmax > MF_PMAX)
        return bh_set_error(ctx, BH_EINVAL, "mean_field: need 2 <= pmax <= " + std::to_string(MF_PMAX));
    if (max_outer < 1) return bh_set_error(ctx, BH_EINVAL, "mean_field: need max_outer >= 1");
    if (!(eps >= 0.0) || std::isinf(eps)) return bh_set_error(ctx, BH_EINVAL, "mean_field: need finite eps >= 0");
    if (npts > (static_cast<int64_t>(1) << 31) * MF_WG / 2)
        return bh_set_error(ctx, BH_ERANGE, "mean_field: too many points for one launch");
    if (npts == 0) return BH_OK;
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    BH_HIP(ctx, hipSetDevice(ctx->device));
    hipStream_t s = ctx->stream;
    const size_t n = static_cast<size_t>(npts);
    std::vector<double> sqh(MF_NMAX + 1);
    for (int i = 0; i <= MF_NMAX; ++i) sqh[i] = std::sqrt(static_cast<double>(i));
    DevArray<double> dmu, dJ, dpsi0, dpsi, dsq;
    DevArray<int32_t> dst, dit, dp;
    DevArray<unsigned long long> dnext;
    BH_TRY(dmu.alloc(ctx, n));
    BH_TRY(dJ.alloc(ctx, n));
    BH_TRY(dpsi0.alloc(ctx, n));
    BH_TRY(dpsi.alloc(ctx, n));
    BH_TRY(dsq.alloc(ctx, MF_NMAX + 1));
    BH_TRY(dst.alloc(ctx, n));
    BH_TRY(dit.alloc(ctx, n));
    BH_TRY(dp.alloc(ctx, n));
    BH_TRY(dnext.alloc(ctx, MF_NEXT));
    BH_HIP(ctx, hipMemcpyAsync(dmu.p, mu, n * 8, hipMemcpyHostToDevice, s));
    BH_HIP(ctx, hipMemcpyAsync(dJ.p, J, n * 8, hipMemcpyHostToDevice, s));
    BH_HIP(ctx, hipMemcpyAsync(dpsi0.p, psi0, n * 8, hipMemcpyHostToDevice, s));
    BH_HIP(ctx, hipMemcpyAsync(dsq.p, sqh.data(), sqh.size() * 8, hipMemcpyHostToDevice, s));
    BH_HIP(ctx, hipMemsetAsync(dnext.p, 0, MF_NEXT * sizeof(unsigned long long), s));
    // The wavefronts that fit at a time.  Up to one point for each: one point to a wavefront.  More: half of
    // the wavefronts (two per SIMD) begin with one point, a quarter with four, the others with what is left, in the order
    // of the classes (1000 x 1000: 40 ms; a quarter and a quarter 43, an eighth each 48, no such wavefronts 48); where there is no room for the order (4 bytes a point), or its indices don't fit, in the given one.
    int wgs = 0, cus = 0;
    BH_HIP(ctx, hipOccupancyMaxActiveBlocksPerMultiprocessor(&wgs, k_scmf, MF_WG, 0));
    BH_HIP(ctx, hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, ctx->device));
    constexpr int WPG = MF_WG / 64;
    const int64_t waves = static_cast<int64_t>(std::max(wgs, 1)) * std::max(cus, 1) * WPG;
    const unsigned nb = static_cast<unsigned>((std::min(npts, waves) + WPG - 1) / WPG);
    MfDeal deal{static_cast<int>(nb) * WPG, static_cast<int>(nb) * WPG, 1, 1, 1, 0};
    DevArray<uint32_t> ord;
    if (npts > waves) {
        deal.w1 = static_cast<int>(waves / 2);
        deal.w2 = deal.w1 + static_cast<int>(waves / 4);
        deal.c2 = 4;
        const int64_t rest = npts - deal.w1 - static_cast<int64_t>(deal.w2 - deal.w1) * deal.c2, full = waves - deal.w2;
        deal.c3 = static_cast<int>(std::max<int64_t>(1, std::min<int64_t>(64, (rest + full - 1) / full)));
        if (npts <= INT32_MAX && ord.alloc(ctx, n) != BH_OK) (void)hipGetLastError();
    }
    deal.first = static_cast<int64_t>(deal.w1) * deal.c1 + static_cast<int64_t>(deal.w2 - deal.w1) * deal.c2 +
                 (static_cast<int64_t>(nb) * WPG - deal.w2) * deal.c3;
    {
        KTimer kt(ctx, "scmf", s);
        if (ord.p) {
            unsigned* count = reinterpret_cast<unsigned*>(dnext.p + 1);
            const unsigned g = static_cast<unsigned>((npts + 255) / 256);
            hipLaunchKernelGGL(k_scmf_count, dim3(std::min(g, 1024u)), dim3(256), 0, s, npts, dmu.p, dJ.p, q, count);
            hipLaunchKernelGGL(k_scmf_order, dim3(g), dim3(256), 0, s, npts, dmu.p, dJ.p, q, count, count + MF_CLASSES, ord.p);
        }
        hipLaunchKernelGGL(k_scmf, dim3(nb), dim3(MF_WG), 0, s, npts, dmu.p, dJ.p, dpsi0.p, ord.p, deal, q, eps, max_outer, pmax,
                           dsq.p, dpsi.p, dst.p, dit.p, dp.p, dnext.p);
    }
    BH_HIP(ctx, hipGetLastError());
    BH_HIP(ctx, hipMemcpyAsync(psi, dpsi.p, n * 8, hipMemcpyDeviceToHost, s));
    if (status) BH_HIP(ctx, hipMemcpyAsync(status, dst.p, n * 4, hipMemcpyDeviceToHost, s));
    if (iters) BH_HIP(ctx, hipMemcpyAsync(iters, dit.p, n * 4, hipMemcpyDeviceToHost, s));
    if (p_last) BH_HIP(ctx, hipMemcpyAsync(p_last, dp.p, n * 4, hipMemcpyDeviceToHost, s));
    BH_HIP(ctx, hipStreamSynchronize(s));
    return BH_OK;
}

}  // extern "C"
