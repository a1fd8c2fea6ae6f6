// A whole FP64 solve with DIAG or NONE (LEQ_BICGS0, model/leq_bicgs.f:316-466)
// in one launch, for systems small enough that every cell's row and vectors
// stay in the registers of one thread.
//
// As launches, an iteration of such a system is eight kernels of 3-5 us each,
// of which the work is a fraction: 32^3 ran 31 us an iteration.  Here the
// blocks (256 cells each, all resident: a cooperative launch) iterate by
// themselves and meet three times an iteration, at its three reductions:
//   v = A P/D, <Rtilde,v>            -> alpha
//   t = A S/D, <t,S>, <t,t>, ||S||^2 -> omega
//   x, r, ||r||^2, <Rtilde,r>        -> beta, convergence
// Only r and v cross between blocks.  A thread keeps P at its cell and at the
// six neighbours and updates all seven from r and v (and S likewise), the
// values the neighbours themselves form, so the operands of the two stencil
// rows never travel.
//
// The exchange goes through memory at agent scope (stores written through,
// loads past the XCD's own L2), without cache write-backs or invalidations.  A
// block's r or v stores are complete (vmcnt 0 in every wave) before its partial
// sums are stored; block 0 collects the partial sums and publishes the totals,
// and every block applies the scalar logic to its own copy of the state.  A
// value is its own arrival flag: its slot holds a signalling NaN, which no
// arithmetic gives, until it is stored.  Slots are used in three sets in turn;
// their owner clears those of the next reduction when a phase begins, by which
// time they have been read (their readers have taken part in the reduction in
// between), and the clears are complete before it takes part in this one.  (All
// blocks reading all partial sums instead took 6.5 us a reduction with 154 blocks
// against 4.1.)
// Measured, an iteration with launches -> here: 16^3 27.8 -> 9.6 us, 32^3 25.5
// -> 10.1, 40^3 27.1 -> 11.9, 48^3 27.9 -> 13.1 (488 blocks); with R exchanged
// through its own array, which the set-up's kernels leave in the L2s, 11.6, 12.1,
// 14.1 and 15.2.  What is left is three round trips of about 3 us.
//
// The arithmetic and the order of every sum are those of the launched kernels
// (leq_phases.h) and of the one-block finish (finish_sum, fin_apply), so the
// solve gives the same bits.
#pragma once
#include "leq_phases.h"

namespace mfix {

constexpr int kResidentBlock = 256;
constexpr int kResidentPerCu = 2;  // blocks a CU holds (200 VGPRs)
constexpr int kResidentBlocks = kResidentPerCu * kNumCus;
constexpr unsigned long long kNoSum = 0x7ff4a5a5a5a5a5a5ull;
constexpr int kResidentSpins = 1 << 23;  // tries of a wait (about a microsecond each) before the launch gives up

// The launch gives up when a wait runs out (another stream or process holds the
// CUs).  Nothing that a launched solve starts from is touched before all blocks
// have ended, so that one can follow: R stays, its exchange goes through T; the
// solution and the final state wait in S and in the partial sums' array for
// k_resident_end, which takes them over unless a block gave up.

// Slots of the partial sums, one 128-byte line per set and block, in the
// solve's P array, 48 of the 256 values of a block (a system of one block that
// has fewer goes on into S, which is written when no slot is read any more);
// and in the partial sums' array the totals, one line per set and XCD, the two
// flags and the final state.
constexpr int kSlotLine = 16;
__host__ __device__ inline int64_t resident_slots(int64_t nblk) { return 3 * nblk * kSlotLine; }
constexpr int kResidentTotals = 3 * kNumXcd * kSlotLine;
struct ResidentEnd {
    int gone;   // a block gave up waiting for another
    int ended;  // the iteration ran, to `st`
    SolverState st;
};
__device__ __forceinline__ auto resident_end(double *partials) {
    return to_global((ResidentEnd *)(partials + kResidentTotals));
}
static_assert(sizeof(double) * kResidentTotals + sizeof(ResidentEnd) <= sizeof(double) * kUpdateBlocks, "in the partial sums");

static __global__ void __launch_bounds__(256) k_resident_slots(const Sys<double> *__restrict__ sys) {
    const int64_t n = resident_slots(sys->P.nblk);
    const gptr<unsigned long long> q = to_global((unsigned long long *)sys->p);
    const gptr<unsigned long long> tot = to_global((unsigned long long *)sys->partials);
    const int64_t k0 = (int64_t)blockIdx.x * 256 + threadIdx.x;
    for (int64_t k = k0; k < n; k += (int64_t)gridDim.x * 256) q[k] = kNoSum;
    if (k0 < kResidentTotals) tot[k0] = kNoSum;
    if (k0 + 256 < kResidentTotals && blockIdx.x == 0) tot[k0 + 256] = kNoSum;
    if (k0 == 0) resident_end(sys->partials)->gone = resident_end(sys->partials)->ended = 0;
}
static_assert(kResidentTotals <= 512, "cleared by the first block");

__device__ __forceinline__ void store_agent(gptr<double> p, double v) {
    __hip_atomic_store((gptr<double>)p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

struct ResidentShared {
    double pair[2][kResidentBlock / 2];  // the update passes' threads take two cells: their sums
    double w[3][16];
    int gone;
    SolverState st;
};

// Waits for a slot's value, up to `most` tries in all.
__device__ __forceinline__ double await_agent(gptr<double> p, int &spins, int most) {
    double x = load_agent(p);
    while ((unsigned long long)__double_as_longlong(x) == kNoSum && ++spins < most) x = load_agent(p);
    return x;
}

// Clears this block's slots of reduction red + 1 at the start of the phase that
// leads to reduction red (complete with the phase's other stores).
__device__ __forceinline__ void resident_clear(gptr<double> slots, gptr<double> totals, int64_t nblk, int64_t blk,
                                               int red) {
    const int set = (red + 1) % 3, t = threadIdx.x;
    const double none = __longlong_as_double((long long)kNoSum);
    if (t < 3) store_agent(slots + (set * nblk + blk) * kSlotLine + t, none);
    if (blk == 0 && t >= 64 && t < 64 + 4 * kNumXcd && (t & 3) < 3)
        store_agent(totals + (set * kNumXcd + ((t - 64) >> 2)) * kSlotLine + (t & 3), none);
}

// Grid-wide sums of NV values in reduction number `red`, in v of thread 0.
// Values PAIR0 .. PAIR0+NPAIR-1 are summed like the update passes' (two cells
// per thread, 128 threads a block), the others like the stencil passes' (one
// cell per thread).  sh.gone is set when
// a wait was given up.
template <int NV, int PAIR0, int NPAIR>
__device__ __forceinline__ void resident_sum(double (&v)[NV], gptr<double> slots, gptr<double> totals, int64_t nblk,
                                             int64_t blk, int red, int most, ResidentShared &sh) {
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int set = red % 3;
    if (NPAIR > 0) {
#pragma unroll
        for (int q = 0; q < NPAIR; ++q) {
            const double odd = __shfl_down(v[PAIR0 + q], 1, 64);
            if (!(t & 1)) sh.pair[q][t >> 1] = (0.0 + v[PAIR0 + q]) + odd;
        }
    }
#pragma unroll
    for (int q = 0; q < NV; ++q)
        if (q < PAIR0 || q >= PAIR0 + NPAIR) {
            const double s = wave_sum(0.0 + v[q]);
            if (lane == 0) sh.w[q][wave] = s;
        }
    if (NPAIR > 0) {
        __syncthreads();
        if (wave < 2) {
#pragma unroll
            for (int q = 0; q < NPAIR; ++q) {
                const double s = wave_sum(sh.pair[q][t]);
                if (lane == 0) sh.w[PAIR0 + q][wave] = s;
            }
        }
    }
    // this wave's stores of r or v are complete before the block arrives
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    int spins = 0;
    if (t == 0) {
        const gptr<double> mine = slots + (set * nblk + blk) * kSlotLine;
#pragma unroll
        for (int q = 0; q < NV; ++q) {
            const int nw = q >= PAIR0 && q < PAIR0 + NPAIR ? 2 : 4;
            double s = sh.w[q][0];
            for (int u = 1; u < nw; ++u) s += sh.w[q][u];
            store_agent(mine + q, s);
        }
    }
    if (blk == 0) {
        // every block's sums, one per virtual thread of the 1,024-thread finish
        double s[NV][kResidentPerCu];
#pragma unroll
        for (int j = 0; j < kResidentPerCu; ++j) {
            const int64_t b = t + 256 * j;
#pragma unroll
            for (int q = 0; q < NV; ++q) {
                s[q][j] = 0.0;
                if (b < nblk) s[q][j] = 0.0 + await_agent(slots + (set * nblk + b) * kSlotLine + q, spins, most);
            }
        }
        __syncthreads();  // (the waves' sums above were read)
#pragma unroll
        for (int q = 0; q < NV; ++q)
#pragma unroll
            for (int j = 0; j < kResidentPerCu; ++j) {
                double x = 0.0;
                if (256 * j < nblk) x = wave_sum(s[q][j]);
                if (lane == 0) sh.w[q][wave + 4 * j] = x;
            }
        __syncthreads();
        if (t == 0) {
#pragma unroll
            for (int q = 0; q < NV; ++q) {
                double x = sh.w[q][0];
                for (int u = 1; u < 4 * kResidentPerCu; ++u) x += sh.w[q][u];  // (the other waves' sums are 0)
                v[q] = x;
            }
#pragma unroll
            for (int k = 0; k < kNumXcd; ++k)
#pragma unroll
                for (int q = 0; q < NV; ++q) store_agent(totals + (set * kNumXcd + k) * kSlotLine + q, v[q]);
        }
    } else if (t == 0) {
        const gptr<double> mine = totals + (set * kNumXcd + (int)(blockIdx.x % kNumXcd)) * kSlotLine;
#pragma unroll
        for (int q = 0; q < NV; ++q) v[q] = await_agent(mine + q, spins, most);
    }
    if (spins >= most) sh.gone = 1;
}

template <int OP>
__global__ void __launch_bounds__(kResidentBlock, kResidentPerCu) k_resident(const Sys<double> *__restrict__ sys, int most) {
    __shared__ ResidentShared sh;
    const Sys<double> &S = *sys;
    const DGrid &g = S.g;
    const int64_t nblk = S.P.nblk, n3 = g.n3, blk = xcd_block(nblk);
    {
        const gptr<const double> src = to_global((const double *)S.st);
        for (int k = threadIdx.x; k < (int)(sizeof(SolverState) / 8); k += kResidentBlock) ((double *)&sh.st)[k] = src[k];
        if (threadIdx.x == 0) sh.gone = 0;
    }
    __syncthreads();
    if (sh.st.done) return;
    // a thread past the last cell follows cell n3-1 and counts for nothing
    const int64_t cell = blk * kResidentBlock + threadIdx.x;
    const bool mine = cell < n3;
    const int64_t c = mine ? cell : n3 - 1;
    const Nb n = neighbours_fast(g, c);
    const uint32_t nb[6] = {(uint32_t)n.km, (uint32_t)n.im, (uint32_t)n.jm, (uint32_t)n.jp, (uint32_t)n.ip, (uint32_t)n.kp};
    const bool dots = mine && (g.dot_all || n.interior);
    const bool dots1 = mine && ((g.dot_all && !sh.st.minimize) || n.interior);  // (the second pass's domain)
    const gptr<const double> a = to_global(S.a);
    const gptr<const double> r0 = to_global((const double *)S.r);
    const gptr<double> gr = to_global(S.t), gv = to_global(S.v), slots = to_global(S.p), totals = to_global(S.partials);
    double A[7], D[6];
#pragma unroll
    for (int p = 0; p < 7; ++p) A[p] = a[p * n3 + c];
#pragma unroll
    for (int k = 0; k < 6; ++k) D[k] = OP == OP_DIAG ? a[3 * n3 + nb[k]] : 1.0;
    double r = r0[c], x = to_global(S.x)[c], p = 0.0, v = 0.0;
    const double rt = to_global(S.rt)[c];
    double rn[6], pn[6], vn[6];
#pragma unroll
    for (int k = 0; k < 6; ++k) {
        rn[k] = r0[nb[k]];
        pn[k] = vn[k] = 0.0;
    }
    auto pre = [&](double z, double d) { return OP == OP_DIAG ? diag_apply(z, d) : z; };
    auto row = [&](const double (&z)[6], double zc) {
        return stencil_combine<double>(g.do_k, A[0], A[1], A[2], A[3], A[4], A[5], A[6], pre(z[0], D[0]), pre(z[1], D[1]),
                                       pre(z[2], D[2]), zc, pre(z[3], D[3]), pre(z[4], D[4]), pre(z[5], D[5]));
    };
    for (int red = 0;; red += 3) {
        resident_clear(slots, totals, nblk, blk, red);
        // P = R, or P = R + beta*(P - omega*V) (leq_bicgs.f:334-343)
        const bool first = sh.st.i == 1;
        const double beta = sh.st.beta, om = sh.st.omega;
        p = first ? r : r + beta * (p - om * v);
#pragma unroll
        for (int k = 0; k < 6; ++k) pn[k] = first ? rn[k] : rn[k] + beta * (pn[k] - om * vn[k]);
        const double ph = pre(p, A[3]);
        v = row(pn, ph);
        if (mine) store_agent(gv + c, v);
        double s1[1] = {dots ? rt * v : 0.0};
        resident_sum<1, 0, 0>(s1, slots, totals, nblk, blk, red, most, sh);
        if (threadIdx.x == 0) fin_apply<FIN_ALPHA, 1>(&sh.st, s1, nullptr);
        __syncthreads();
        if (sh.gone) break;
        resident_clear(slots, totals, nblk, blk, red + 1);
        // S = R - alpha*V (:365-367) and T = A*Shat
        const double alpha = sh.st.alpha;
#pragma unroll
        for (int k = 0; k < 6; ++k) vn[k] = load_agent(gv + nb[k]);
        const double s = r - alpha * v;
        double sn[6];
#pragma unroll
        for (int k = 0; k < 6; ++k) sn[k] = rn[k] - alpha * vn[k];
        const double shv = pre(s, A[3]);
        const double tt = row(sn, shv);
        double s3[3] = {dots1 ? tt * s : 0.0, dots1 ? tt * tt : 0.0, dots ? s * s : 0.0};
        resident_sum<3, 2, 1>(s3, slots, totals, nblk, blk, red + 1, most, sh);
        if (threadIdx.x == 0) fin_apply<FIN_OMEGA, 3>(&sh.st, s3, nullptr);
        __syncthreads();
        if (sh.gone) break;
        resident_clear(slots, totals, nblk, blk, red + 2);
        // Var += alpha*Phat + omega*Shat; R = S - omega*T (:432-436)
        const double omega = sh.st.omega;
        double s2[2] = {0.0, 0.0};
        if (sh.st.s_exit) {
            x = x + alpha * ph;
        } else {
            x = x + alpha * ph + omega * shv;
            r = s - omega * tt;
            if (mine) store_agent(gr + c, r);
            if (dots) {
                s2[0] = r * r;
                s2[1] = rt * r;
            }
        }
        resident_sum<2, 0, 2>(s2, slots, totals, nblk, blk, red + 2, most, sh);
        if (threadIdx.x == 0) fin_apply<FIN_XR, 2>(&sh.st, s2, nullptr);
        __syncthreads();
        if (sh.gone) break;
        if (sh.st.done) break;
#pragma unroll
        for (int k = 0; k < 6; ++k) rn[k] = load_agent(gr + nb[k]);
    }
    const auto end = resident_end(S.partials);
    if (sh.gone) {
        if (threadIdx.x == 0) end->gone = 1;
        return;
    }
    if (mine) to_global(S.s)[c] = x;
    if (blk == 0) {
        __syncthreads();
        const gptr<double> dst = (gptr<double>)&end->st;
        for (int k = threadIdx.x; k < (int)(sizeof(SolverState) / 8); k += kResidentBlock) dst[k] = ((double *)&sh.st)[k];
        if (threadIdx.x == 0) end->ended = 1;
    }
}

// The solution and the state of a launch that ended (one that had nothing to do
// leaves them as they are).
static __global__ void __launch_bounds__(kResidentBlock) k_resident_end(const Sys<double> *__restrict__ sys) {
    const Sys<double> &S = *sys;
    const auto end = resident_end(S.partials);
    if (end->gone || !end->ended) return;
    const int64_t c = (int64_t)blockIdx.x * kResidentBlock + threadIdx.x;
    if (c < S.g.n3) to_global(S.x)[c] = to_global((const double *)S.s)[c];
    if (blockIdx.x == 0) {
        const gptr<double> dst = to_global((double *)S.st);
        const gptr<const double> src = (gptr<const double>)&end->st;
        for (int k = threadIdx.x; k < (int)(sizeof(SolverState) / 8); k += kResidentBlock) dst[k] = src[k];
    }
}

}  // namespace mfix
