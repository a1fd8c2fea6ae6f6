// Red-black J-line phases of the LINE preconditioner (LEQ_MSOLVE,
// model/leqsol_mod.f:286-598; LEQ_IKSWEEP :851-921; DGTSV
// model/DGTSV.f:107-246), whole lines in LDS.
//
// A block of 256 threads takes S.lpb lines of one colour and holds their
// rows in LDS: all threads load them (consecutive lanes take consecutive rows
// of a line, every load of a thread issued before its first use) and form the
// right-hand side, one lane per line runs the tridiagonal solve in LDS, and
// all threads store the solution.  One memory round trip and six barriers a
// block; blocks of a CU overlap each other's loads and chains.
//
// What bounds a phase is the serial chain of a line where few blocks share a
// CU, and where many do the time a line holds its LDS (chain, load and store)
// against the bytes.  The chain is shortened by factoring once per solve: the
// multipliers and the eliminated diagonal of DGTSV depend on A_M alone, which
// does not change during a solve, so k_line_factor runs the elimination of
// every line at set-up (DGTSV's operations in its order) and the phases read
// its results in the places of DL and A0.  A phase's chain is then b_i -=
// fact_i b_{i-1} forward (a product and a difference) and x_i = (b_i - u_i
// x_{i+1})/d_i back, the division done with the refined reciprocal of d_i
// (Newton-Raphson, then Markstein's quotient correction: q = n r, q += (n - q
// d) r): five dependent operations where a division alone takes about ten.
// Blocks with a row interchange carry it through both passes.  Every value is
// the one DGTSV's own operations give, bit for bit (but for the sign of a
// zero), as long as no operand leaves the range in which the correction is
// exact; a block whose solution holds a value outside the range divides instead
// (whole_back_exact), and one with a pivot outside it or zero (marked by
// k_line_factor) runs DGTSV itself in LDS.
//
// Measured (events of the dispatches, LINE solve, colour phase; before, one
// DGTSV lane per line over 16-row tiles with the finished rows in global
// scratch): 64^3 28.4 -> 10.3 us, 128^3 56.2 -> 29.4 us, 158^3 70.9 -> 50.5
// us, 256^3 409 -> 234 us.
#pragma once
#include <cmath>

#include "leq_phases.h"

namespace mfix {

constexpr int kWholeThreads = 256;
// Rows a thread loads at most (their diagonals stay in its registers through
// the forward pass); longer lines take k_line_color_sys.
constexpr int kWholeElems = 6, kWholeRows = kWholeThreads * kWholeElems;
// LDS of a block beside its lines (WholeLines, DGTSV's INFO, block sums), and what
// is left for them where four blocks fit on a CU (as the launch bound allows).
constexpr int kWholeFixed = 2048, kWholePerCu = 4, kWholeLdsTarget = 160 * 1024 / kWholePerCu - kWholeFixed;
constexpr int kWholeLines = 64;  // one lane of the solving wave per line

// k_line_stream: two blocks per CU, one wave of each solving, the other
// threads holding rows.
constexpr int kStreamThreads = 512, kStreamLoaders = kStreamThreads - 64, kStreamElems = 5,
              kStreamRows = kStreamLoaders * kStreamElems, kStreamBlocks = 2 * kNumCus,
              kStreamLdsTarget = 160 * 1024 / 2 - 3072;
constexpr int kStreamMost = 1024;  // entries of a block, a bit each in k_line_stream

// A line holds whole_rows rows (its own and up to three identity rows, so that
// the chains take four rows a step) and lines sit an odd number of 16-byte
// units apart: the solving lanes (one line each, the same two rows) and the
// loading lanes (one line, consecutive rows) both spread over the banks.
__host__ __device__ constexpr int whole_rows(int n) { return (n + 3) & ~3; }
__host__ __device__ constexpr int whole_stride(int n) { return whole_rows(n) + 2; }
__host__ inline bool whole_fits(int n) { return n <= kWholeRows; }
// Elements kept free before the first array and behind the last, for the
// chains' reads past a line's ends.
constexpr int kWholeFront = 16, kWholeTail = 16;
// Lines of k_line_stream, and of blocks of up to eight, hold rows in eights
// (whole_forward_swap8).
__host__ __device__ constexpr int stream_rows(int n) { return (n + 7) & ~7; }
__host__ __device__ constexpr int stream_stride(int n) { return stream_rows(n) + 2; }
__host__ __device__ constexpr int stream_elems(int n, int lpb) {
    return kWholeFront + 4 * lpb * stream_stride(n) + kWholeTail;
}
__host__ __device__ constexpr bool whole_few(int lpb) { return lpb <= 8; }
// LDS elements of a block of lpb lines: four arrays.
__host__ __device__ constexpr int whole_elems(int n, int lpb) {
    return whole_few(lpb) ? stream_elems(n, lpb) : kWholeFront + 4 * lpb * whole_stride(n) + kWholeTail;
}

// Lines whose LDS leaves room for four blocks on a CU (one line of more than
// 1,200 rows leaves room for three).
__host__ inline int whole_most(int n, size_t elem) {
    int most = (kWholeLdsTarget / (int)elem - kWholeFront - kWholeTail) / (4 * whole_stride(n));
    while (most > 1 && whole_elems(n, most) * elem > kWholeLdsTarget) --most;
    return most > 1 ? most : 1;
}
// Lines whose LDS the device holds at once.
__host__ inline double whole_at_once(int n, size_t elem) {
    return (double)kNumCus * kWholePerCu * whole_most(n, elem);
}

// Lines per block.  `table` is the part of the device that all lines of one
// colour of every system of the launch take together.  Where they fit in one
// round, blocks are sized for two per CU: fewer would leave CUs with one more
// block than others, more only share them (64^3 10.2 us a phase with five lines a
// block, 13.2 with three).  Else the blocks' shares are even over the fewest
// rounds that hold them: a round more costs a whole load, chain and store (nine
// 64^3 systems 45 us a phase with five lines a block, four rounds, 34 us with
// ten, two rounds).  pin: mfix_leq_set_line_block's value, 0 = none.
__host__ inline int whole_lpb(int n, double table, size_t elem, int pin) {
    const double rounds = std::ceil(table), blocks = kNumCus * (rounds > 1.0 ? rounds * kWholePerCu : 2.0);
    // (a share that is a whole number of lines stays it)
    int64_t lpb = (int64_t)std::ceil(table * whole_at_once(n, elem) / blocks - 1e-6);
    if (lpb > whole_most(n, elem)) lpb = whole_most(n, elem);
    if (pin > 0) lpb = pin;
    if (lpb > kWholeRows / n) lpb = kWholeRows / n;
    if (lpb > kWholeLines) lpb = kWholeLines;
    return lpb < 1 ? 1 : (int)lpb;
}

// Entries of a colour of `lines` lines then: the fewest a block, of lines that
// it holds.
__host__ inline int64_t stream_most(int n) {
    int64_t most = (kStreamLdsTarget / 8 - kWholeFront - kWholeTail) / (4 * stream_stride(n));
    if (most > kStreamRows / n) most = kStreamRows / n;
    if (most > kWholeLines) most = kWholeLines;
    return most;
}
__host__ inline int64_t stream_entries(int n, int64_t lines) {
    const int64_t most = stream_most(n);
    return (lines + kStreamBlocks * most - 1) / (kStreamBlocks * most) * kStreamBlocks;
}
// Whether a colour's lines are better in k_line_color_sys, 64 a block in no more
// LDS than one or two take here: lines of more than 746 rows, one or two an
// entry, from the eighth entry a block on (one line an entry: the seventh).
// Colour phase, in whole lines and there: 1,002 rows, 6,272 lines (seven
// entries) 411 and 429 us, 8,450 (nine) 520 and 457; 1,502 rows, 2,738 lines
// (six) 518 and 579, 3,362 (seven) 598 and 591, 11,552 (23) 1,897 and 742.
__host__ inline bool long_lines(int n, int64_t lines) {
    const int64_t most = stream_most(n);
    return most <= 2 && stream_entries(n, lines) > (5 + most) * kStreamBlocks;
}
// Whether the lines of a system stream: their LDS is more than one round of
// k_line_whole's blocks.  Colour phase of whole lines and of streamed ones:
// 7,320 lines of 146 rows (seven a block) 32.2 and 26.1 us; but 800 of 1,502 rows,
// two rounds at three blocks a CU, 163 and 183, and 72,962 of 10 rows, which the
// 64 lanes of a block hold before its LDS is full, 21 and 24.
__host__ inline bool line_streams(int n, int64_t lines, int64_t cells) {
    return n <= kWholeRows && (double)lines > whole_at_once(n, sizeof(double)) && cells < (1ll << 29) &&
           stream_entries(n, lines) <= (int64_t)kStreamBlocks * kStreamMost;
}
// Lines of entry j of a colour: [first(j), first(j + 1)), where first(j) = j
// step / 2^32.  step = lines / entries, rounded up, shares them evenly (the last
// entry's end is the last line: entries < 2^32); a whole number of lines is exact.
__host__ inline uint64_t entry_step(int64_t lines, int64_t entries) {
    const unsigned __int128 l = (unsigned __int128)lines << 32;
    return (uint64_t)((l + (uint64_t)entries - 1) / (uint64_t)entries);
}
__host__ __device__ __forceinline__ int64_t entry_first(uint64_t step, int j) {
    return (int64_t)(((unsigned __int128)step * (uint64_t)j) >> 32);
}

// The ranges in which the corrected quotient is the correctly rounded one: no
// intermediate of it is subnormal or overflows (the remainder's last place is
// at least 2^-106 of the numerator, |x d| >= 2^-960).
__device__ __forceinline__ bool factor_in_range(double d) {
    const double m = fabs(d);
    return m >= 0x1p-60 && m <= 0x1p60;  // (NaN: false)
}
__device__ __forceinline__ bool solution_in_range(double x) {
    const double m = fabs(x);
    return x == 0.0 || (m >= 0x1p-900 && m <= 0x1p900);
}

// 1/d to the last place but for ties: two Newton-Raphson steps on the
// hardware's estimate.
__device__ __forceinline__ double refined_rcp(double d) {
    double r = __builtin_amdgcn_rcp(d);
    r = __builtin_fma(__builtin_fma(-d, r, 1.0), r, r);
    return __builtin_fma(__builtin_fma(-d, r, 1.0), r, r);
}
// n/d from r = refined_rcp(d).
__device__ __forceinline__ double corrected_quotient(double n, double d, double r) {
    const double q = n * r;
    return __builtin_fma(__builtin_fma(-q, d, n), r, q);
}

// Start cell and I/K neighbour offsets of the block's lines, constant along a
// J-line (set_increments.f:72-112); the lines past the colour's last are
// missing from the end.
struct WholeLines {
    uint32_t c0[kWholeLines], im[kWholeLines], ip[kWholeLines], km[kWholeLines], kp[kWholeLines];
    int n;
    int odd, own;  // (k_line_whole: a right-hand side is out of range; the block's mark is kOwnDgtsv)
};
__device__ __forceinline__ void whole_lines(const DGrid &g, uint64_t step, int j, int param, WholeLines &w) {
    const int l = threadIdx.x;
    if (l < 64) {
        int u = 0, v = 0;
        const int64_t first = entry_first(step, j);
        const bool ok = l < entry_first(step, j + 1) - first &&
                        color_line(g.ni, g.nk, g.do_k ? 1 : 0, param, first + l, u, v);
        const uint32_t c1 = (uint32_t)g.c1, c2 = (uint32_t)g.c2;
        if (ok) {
            w.c0[l] = (uint32_t)u * c1 + (uint32_t)v * c2;
            w.im[l] = (uint32_t)(nb_minus(u, g.ni, g.cyc_x) - u) * c1;
            w.ip[l] = (uint32_t)(nb_plus(u, g.ni, g.cyc_x) - u) * c1;
            w.km[l] = g.do_k ? (uint32_t)(nb_minus(v, g.nk, g.cyc_z) - v) * c2 : 0u;
            w.kp[l] = g.do_k ? (uint32_t)(nb_plus(v, g.nk, g.cyc_z) - v) * c2 : 0u;
        }
        const uint64_t have = __ballot(ok);
        if (l == 0) {
            w.n = __popcll(have);
            w.odd = w.own = 0;
        }
    }
    __syncthreads();
}

// A multiplier of an interchanged row is stored times 2^600: DGTSV's
// multipliers are at most 1 in size, so the factor marks the row and comes off
// exactly.
constexpr double kSwapUp = 0x1p600, kSwapDown = 0x1p-600;
__device__ __forceinline__ bool swapped(double f) { return fabs(f) > 2.0; }
// A block's mark, in the place of its first row's multiplier (which has none):
// kSwapUp where it has an interchanged row, this where it has a pivot of zero or
// out of range.  By block, so that one such line does not cost the others: with
// DGTSV in every block of a system that has one 150x201x180 took 208 us a phase
// and 256^3 690, now 94 and 228 (109 and 399 with k_line_color_sys).
constexpr double kOwnDgtsv = 0x1p620;
__device__ __forceinline__ bool own_dgtsv(double mark) { return fabs(mark) > 0x1p610; }

// The elimination of one line without row interchanges and the two passes on
// its factored rows, in the lane that solves the line, over whole_rows(n)
// rows.  A pass is bound by its LDS instructions (each
// costs what all 64 lanes of it would, 10-25 cycles) more than by the
// arithmetic (a dependent FP64 operation takes about five): two rows move per
// instruction, read one register set ahead of the chain at fixed offsets from
// running pointers, and the scheduler keeps the order written here.  The last
// reads run past the line's end (forward) or before its first row (back),
// inside the block's LDS, and are not used.  Measured alone: 35 and 61 cycles
// a row.
typedef double pair2 __attribute__((ext_vector_type(2)));

// (the divisions by the running diagonal are the chain: rows in and out are
// the last of it).  Whether the multipliers and the diagonal are DGTSV's is for
// the caller to look at: |F| <= 1 (no interchange) and both in range.
__device__ __forceinline__ void whole_eliminate(double *__restrict__ pf, double *__restrict__ pd,
                                                const double *__restrict__ pu, int rows) {
    constexpr int R = 4;
    struct Rows {
        pair2 f[R / 2], d[R / 2], u[R / 2];
    } s0, s1;
    auto get = [&](Rows &w, int at) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < R / 2; ++k) {
            w.f[k] = *(const pair2 *)&pf[at + 2 * k];
            w.d[k] = *(const pair2 *)&pd[at + 2 * k];
            w.u[k] = *(const pair2 *)&pu[at + 2 * k];
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    double d = 1.0, u = 0.0;  // (row 0's lower coupling is 0)
    auto one = [&](double &f, double &dr, double ur) __attribute__((always_inline)) {
        f = corrected_quotient(f, d, refined_rcp(d));
        d = dr - f * u;
        dr = d;
        u = ur;
    };
    auto run = [&](Rows &w, int at) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < R / 2; ++k) {
            double f0 = w.f[k].x, f1 = w.f[k].y, d0 = w.d[k].x, d1 = w.d[k].y;
            one(f0, d0, w.u[k].x);
            one(f1, d1, w.u[k].y);
            *(pair2 *)&pf[at + 2 * k] = pair2{f0, f1};
            *(pair2 *)&pd[at + 2 * k] = pair2{d0, d1};
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    get(s0, 0);
    for (; rows >= 2 * R; rows -= 2 * R, pf += 2 * R, pd += 2 * R, pu += 2 * R) {
        get(s1, R);
        run(s0, 0);
        get(s0, 2 * R);
        run(s1, R);
    }
    if (rows > 0) run(s0, 0);
}

__device__ __forceinline__ void whole_forward(const double *__restrict__ pf, double *__restrict__ pb, int rows) {
    constexpr int R = 8;
    struct Rows {
        pair2 f[R / 2], b[R / 2];
    } s0, s1;
    auto get = [&](Rows &w, int at) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < R / 2; ++k) {
            w.f[k] = *(const pair2 *)&pf[at + 2 * k];
            w.b[k] = *(const pair2 *)&pb[at + 2 * k];
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    double b = 0.0;  // (row 0's multiplier is 0)
    auto run = [&](const Rows &w, int at, int cnt) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < cnt / 2; ++k) {
            pair2 o;
            b = w.b[k].x - w.f[k].x * b;
            o.x = b;
            b = w.b[k].y - w.f[k].y * b;
            o.y = b;
            *(pair2 *)&pb[at + 2 * k] = o;
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    get(s0, 0);
    for (; rows >= 2 * R; rows -= 2 * R, pf += 2 * R, pb += 2 * R) {
        get(s1, R);
        run(s0, 0, R);
        get(s0, 2 * R);
        run(s1, R, R);
    }
    if (rows >= R) {
        get(s1, R);
        run(s0, 0, R);
        if (rows > R) run(s1, R, R / 2);
    } else if (rows > 0) {
        run(s0, 0, R / 2);
    }
}

__device__ __forceinline__ void whole_back(double *__restrict__ pb, const double *__restrict__ pu,
                                           const double *__restrict__ pd, const double *__restrict__ pr, int rows) {
    constexpr int R = 4;
    struct Rows {
        pair2 b[R / 2], u[R / 2], d[R / 2], r[R / 2];
    } s0, s1;
    pb += rows - 2;
    pu += rows - 2;
    pd += rows - 2;
    pr += rows - 2;
    double x = 0.0;  // (the last row's upper coupling is 0)
    auto get = [&](Rows &w, int at) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < R / 2; ++k) {
            w.b[k] = *(const pair2 *)&pb[-at - 2 * k];
            w.u[k] = *(const pair2 *)&pu[-at - 2 * k];
            w.d[k] = *(const pair2 *)&pd[-at - 2 * k];
            w.r[k] = *(const pair2 *)&pr[-at - 2 * k];
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    auto run = [&](const Rows &w, int at) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < R / 2; ++k) {
            pair2 o;
            x = corrected_quotient(w.b[k].y - w.u[k].y * x, w.d[k].y, w.r[k].y);
            o.y = x;
            x = corrected_quotient(w.b[k].x - w.u[k].x * x, w.d[k].x, w.r[k].x);
            o.x = x;
            *(pair2 *)&pb[-at - 2 * k] = o;
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    get(s0, 0);
    for (; rows >= 2 * R; rows -= 2 * R, pb -= 2 * R, pu -= 2 * R, pd -= 2 * R, pr -= 2 * R) {
        get(s1, R);
        run(s0, 0);
        get(s0, 2 * R);
        run(s1, R);
    }
    if (rows > 0) run(s0, 0);
}

// The same two passes where some line of the block interchanges rows: the
// right-hand sides trade places with them, and the second super-diagonal (in
// V, the reciprocals' place: they are formed in the chain here) comes in.
__device__ __forceinline__ void whole_forward_swap(const double *__restrict__ pf, double *__restrict__ pb, int rows) {
    constexpr int R = 4;
    struct Rows {
        pair2 f[R / 2], b[R / 2];
    } s0, s1;
    auto get = [&](Rows &w, int at) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < R / 2; ++k) {
            w.f[k] = *(const pair2 *)&pf[at + 2 * k];
            w.b[k] = *(const pair2 *)&pb[at + 2 * k];
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    double b = 0.0;
    // row q's multiplier and right-hand side; returns row q-1's after the interchange
    auto one = [&](double f, double r) __attribute__((always_inline)) {
        const bool s = swapped(f);
        const double fact = s ? f * kSwapDown : f;
        const double top = s ? r : b;
        b = (s ? b : r) - fact * top;
        return top;
    };
    auto run = [&](const Rows &w, int at) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < R / 2; ++k) {  // (row 0 writes in front of the line, an element that is not used)
            pb[at + 2 * k - 1] = one(w.f[k].x, w.b[k].x);
            pb[at + 2 * k] = one(w.f[k].y, w.b[k].y);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    get(s0, 0);
    for (; rows >= 2 * R; rows -= 2 * R, pf += 2 * R, pb += 2 * R) {
        get(s1, R);
        run(s0, 0);
        get(s0, 2 * R);
        run(s1, R);
    }
    if (rows > 0) {
        run(s0, 0);
        pb += R;
    }
    pb[-1] = b;
}

// EXACT: by DGTSV's own operations, the division and (V false) the product with
// a second super-diagonal of 0 included, from the rows after on (x1, x2).
template <bool EXACT = false, bool V = true>
__device__ __forceinline__ void whole_back_swap(double *__restrict__ pb, const double *__restrict__ pu,
                                                const double *__restrict__ pv, const double *__restrict__ pd, int rows,
                                                double x1 = 0.0, double x2 = 0.0) {
    constexpr int R = 4;
    struct Rows {
        pair2 b[R / 2], u[R / 2], v[R / 2], d[R / 2];
    } s0, s1;
    pb += rows - 2;
    pu += rows - 2;
    pv += rows - 2;
    pd += rows - 2;
    auto get = [&](Rows &w, int at) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < R / 2; ++k) {
            w.b[k] = *(const pair2 *)&pb[-at - 2 * k];
            w.u[k] = *(const pair2 *)&pu[-at - 2 * k];
            w.v[k] = V ? *(const pair2 *)&pv[-at - 2 * k] : pair2{0.0, 0.0};
            w.d[k] = *(const pair2 *)&pd[-at - 2 * k];
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    auto one = [&](double b, double u, double v, double d) __attribute__((always_inline)) {
        const double num = b - u * x1 - v * x2, x = EXACT ? num / d : corrected_quotient(num, d, refined_rcp(d));
        x2 = x1;
        x1 = x;
        return x;
    };
    auto run = [&](const Rows &w, int at) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < R / 2; ++k) {
            pair2 o;
            o.y = one(w.b[k].y, w.u[k].y, w.v[k].y, w.d[k].y);
            o.x = one(w.b[k].x, w.u[k].x, w.v[k].x, w.d[k].x);
            *(pair2 *)&pb[-at - 2 * k] = o;
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    get(s0, 0);
    for (; rows >= 2 * R; rows -= 2 * R, pb -= 2 * R, pu -= 2 * R, pv -= 2 * R, pd -= 2 * R) {
        get(s1, R);
        run(s0, 0);
        get(s0, 2 * R);
        run(s1, R);
    }
    if (rows > 0) run(s0, 0);
}

// The back pass by DGTSV's own operations: for values out of range, infinities
// and NaN (the forward passes are DGTSV's as they are; the identity rows behind
// the line, which may hold a NaN then, are left out).  A solution that decays
// along its line leaves the range, so such blocks must not cost much more than
// others: with every value out of range a colour phase takes 12.8 us at 64^3
// (10.4 in range), 85 at 150x201x180 (68) and 248 at 256^3 (196), where DGTSV
// itself, its elimination included, took 32, 253 and 847.  Looking at the
// right-hand sides first costs 1-2 % of a phase.
template <bool V>
__device__ __forceinline__ void whole_back_exact(double *__restrict__ pb, const double *__restrict__ pu,
                                                 const double *__restrict__ pv, const double *__restrict__ pd, int n) {
    double x1 = 0.0, x2 = 0.0;
    for (int q = n - 1; q >= (n & ~3); --q) {  // (the last row's couplings are 0)
        const double x = (pb[q] - pu[q] * x1 - (V ? pv[q] : 0.0) * x2) / pd[q];
        pb[q] = x;
        x2 = x1;
        x1 = x;
    }
    whole_back_swap<true, V>(pb, pu, pv, pd, n & ~3, x1, x2);
}

// These two passes by eight lanes a line (j = lane % 8), rows in eights, for a
// wave of up to eight lines: lane j holds row j of a group of eight, and a step
// forms every lane's row from its neighbour's, passed by a lane shift, so row j
// is right after j + 1 steps and stays (its operands do not change), and eight
// steps solve the group.  The row next to the group before (lane 0 forward,
// lane 7 back) takes that group's values first and is then held by zero
// couplings.  What does not depend on the neighbour, the marked multipliers and
// the reciprocal, is formed for eight rows at once; in one lane a line it is
// most of the instructions (256^3: 261 -> 228 us a phase; with more lines a
// wave takes two turns: 11 lines a block, 150x201x180, 91 -> 121 us; without
// interchanges there is little of it: 203 -> 205).
__device__ __forceinline__ void whole_forward_swap8(const double *__restrict__ pf, double *__restrict__ pb, int rows,
                                                    int j) {
    double f = pf[j], b = pb[j], v = 0.0;
    for (int at = j; at < rows; at += 8) {
        const double nf = pf[at + 8], nb = pb[at + 8];
        const double c = row_down<7>(v);
        const bool s = swapped(f);
        const double fact = s ? f * kSwapDown : f, m = fact * b;
        v = s ? c - m : b - fact * c;  // (lane 0's, the others' below)
        const bool s1 = s && j != 0;
        const double f1 = j == 0 ? 0.0 : fact, b1 = j == 0 ? v : b;
#pragma unroll
        for (int k = 1; k < 8; ++k) {
            const double p = row_up<1>(v), keep = b1 - f1 * p, trade = p - m;
            v = s1 ? trade : keep;
        }
        const double p = row_up<1>(v);
        pb[at - 1] = s ? b : j == 0 ? c : p;  // (row 0 writes in front of the line, an element that is not used)
        f = nf;
        b = nb;
    }
    if (j == 7) pb[rows - 1] = v;
}

__device__ __forceinline__ void whole_back_swap8(double *__restrict__ pb, const double *__restrict__ pu,
                                                 const double *__restrict__ pv, const double *__restrict__ pd,
                                                 int rows, int j) {
    int at = rows - 8 + j;
    double b = pb[at], u = pu[at], v = pv[at], d = pd[at], x = 0.0;
    for (; at >= 0; at -= 8) {
        const double nb = pb[at - 8], nu = pu[at - 8], nv = pv[at - 8], nd = pd[at - 8], r = refined_rcp(d);
        // the group after's first row in lane 7; its first two in lanes 6 and 7
        const double c1 = row_up<7>(x), c2 = row_up<6>(x);
        b = j == 7 ? b - u * c1 - v * c2 : b;
        u = j == 7 ? 0.0 : u;
        v = j == 7 ? 0.0 : v;
        x = corrected_quotient(b, d, r);
#pragma unroll
        for (int k = 1; k < 8; ++k) {
            const double two = row_down<2>(x);
            x = corrected_quotient(b - u * row_down<1>(x) - v * (j >= 6 ? c2 : two), d, r);
        }
        pb[at] = x;
        b = nb;
        u = nu;
        v = nv;
        d = nd;
    }
}

// DGTSV's elimination of every line of the listed FP64 systems, both colours
// (blockIdx.y = colour), in cell order: the multipliers (row 0: 0) to S.lf and
// the eliminated diagonal to S.ld, and, for a block of lines with a row
// interchange, the eliminated first and second super-diagonals to S.lu and
// S.lu2 (else they are A_M's upper coupling and 0).
static __global__ void __launch_bounds__(kWholeThreads) k_line_factor(const Sys<double> *__restrict__ sys,
                                                                      const int2 *__restrict__ map) {
    extern __shared__ __align__(16) char whole_lds[];
    __shared__ WholeLines w;
    const int2 e = map[blockIdx.x];
    if (e.x < 0) return;
    const Sys<double> &S = sys[e.x];
    auto *__restrict__ st = to_global(S.st);
    if (st->done) return;
    const DGrid &g = S.g;
    const int n = g.nj, ls = whole_stride(n);
    whole_lines(g, S.lstep, e.y, (int)blockIdx.y, w);
    const int nl = w.n, tot = nl * n;
    double *__restrict__ F = (double *)whole_lds + kWholeFront, *__restrict__ D = F + S.lpb * ls,
                         *__restrict__ U = D + S.lpb * ls, *__restrict__ V = U + S.lpb * ls;
    const int64_t n3 = g.n3;
    const gptr<const double> a = to_global(S.a);
    auto load = [&]() {
        for (int xs = threadIdx.x; xs < tot; xs += 3 * kWholeThreads) {
            double dl[3], d[3], du[3];
            int o[3];
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const int x0 = xs + k * kWholeThreads;
                const int x = x0 < tot ? x0 : tot - 1;  // (past the end: the last row again)
                const int l = (int)div_by((uint32_t)x, g.mnj, g.snj), q = x - l * n;
                const uint32_t c = w.c0[l] + (uint32_t)q;
                o[k] = l * ls + q;
                dl[k] = q > 0 ? a[1 * n3 + c] : 0.0;
                d[k] = a[3 * n3 + c];
                du[k] = q < n - 1 ? a[5 * n3 + c] : 0.0;
            }
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                F[o[k]] = dl[k];
                D[o[k]] = d[k];
                U[o[k]] = du[k];
            }
        }
        for (int x = threadIdx.x; x < 4 * nl; x += kWholeThreads) {
            const int q = n + (x & 3), at = (x >> 2) * ls + q;
            if (q < whole_rows(n)) {  // identity rows
                F[at] = U[at] = 0.0;
                D[at] = 1.0;
            }
        }
        __syncthreads();
    };
    const gptr<double> lf = to_global(S.lf), ld = to_global(S.ld), lu = to_global(S.lu), lu2 = to_global(S.lu2);
    // without interchanges first; all threads look at the result
    load();
    if ((int)threadIdx.x < nl) {
        const int o = threadIdx.x * ls;
        whole_eliminate(F + o, D + o, U + o, whole_rows(n));
    }
    __syncthreads();
    int bad = 0;
    for (int x = threadIdx.x; x < tot; x += kWholeThreads) {
        const int l = (int)div_by((uint32_t)x, g.mnj, g.snj), at = l * ls + x - l * n;
        bad |= !(fabs(F[at]) <= 1.0 && solution_in_range(F[at]) && factor_in_range(D[at]));
    }
    if (!__syncthreads_or(bad)) {
        for (int x = threadIdx.x; x < tot; x += kWholeThreads) {
            const int l = (int)div_by((uint32_t)x, g.mnj, g.snj), q = x - l * n, at = l * ls + q;
            const uint32_t c = w.c0[l] + (uint32_t)q;
            lf[c] = F[at];
            ld[c] = D[at];
        }
        return;
    }
    load();
    int any = 0;
    bool ok = true;
    if ((int)threadIdx.x < nl) {
        const int o = threadIdx.x * ls;
        double d = D[o], u = U[o];
        double dl1 = F[o + 1], d1 = D[o + 1], u1 = U[o + 1];  // (a line has at least three rows)
        for (int i = 0; i < n - 1; ++i) {
            const int nx = i + 2 < n ? i + 2 : n - 1;  // the next row is read ahead of this one's division
            const double dl2 = F[o + nx], d2 = D[o + nx], u2 = U[o + nx];
            double fd = d, fu = u, fv = 0.0, f, dn, un = u1;
            if (fabs(d) >= fabs(dl1)) {
                f = dl1 / d;  // (DGTSV.f:111-122)
                dn = d1 - f * u;
            } else {
                // interchange rows i and i+1 (DGTSV.f:123-136, :148-158)
                const double fact = d / dl1;
                fd = dl1;
                fu = d1;
                dn = u - fact * d1;
                if (i < n - 2) {
                    fv = u1;
                    un = -fact * u1;
                }
                f = fact * kSwapUp;
                ok = ok && swapped(f);
                any = 1;
            }
            ok = ok && factor_in_range(fd);
            F[o + i + 1] = f;
            D[o + i] = fd;
            U[o + i] = fu;
            V[o + i] = fv;
            d = dn;
            u = un;
            dl1 = dl2;
            d1 = d2;
            u1 = u2;
        }
        D[o + n - 1] = d;
        U[o + n - 1] = 0.0;
        V[o + n - 1] = 0.0;
        ok = ok && factor_in_range(d);
    }
    any = __syncthreads_or(any);
    const int own = __syncthreads_or(!ok);
    for (int x = threadIdx.x; x < tot; x += kWholeThreads) {
        const int l = (int)div_by((uint32_t)x, g.mnj, g.snj), q = x - l * n, at = l * ls + q;
        const uint32_t c = w.c0[l] + (uint32_t)q;
        lf[c] = x > 0 || !(any || own) ? F[at] : own ? kOwnDgtsv : kSwapUp;
        ld[c] = D[at];
        if (any) {
            lu[c] = U[at];
            lu2[c] = V[at];
        }
    }
}

// DGTSV.f:107-163, :233-246 of one line in place: row i's diagonal, first and
// second super-diagonal and right-hand side stay in slot i of D, U, F, B
// (DL(i) was consumed one step before).  Returns INFO.
template <typename T>
__device__ __forceinline__ int whole_dgtsv(T *__restrict__ F, T *__restrict__ B, T *__restrict__ U,
                                           T *__restrict__ D, int n) {
    T d0 = D[0], u0 = U[0], b0 = B[0];
    int info = 0;
    for (int i = 0; i < n - 1; ++i) {
        const T dl1 = F[i + 1], d1 = D[i + 1], u1 = U[i + 1], b1 = B[i + 1];
        const bool keep = fabs((double)d0) >= fabs((double)dl1);  // no interchange
        if (keep && d0 == (T)0 && !info) info = i + 1;
        const T fact = (keep ? dl1 : d0) / (keep ? d0 : dl1);
        const T pm = keep ? u0 : d1;  // row i's DU after the interchange
        const T pb = keep ? b0 : b1;  // row i's B after the interchange
        const bool sh = !keep && i < n - 2;
        D[i] = keep ? d0 : dl1;
        U[i] = pm;
        F[i] = sh ? u1 : (T)0;
        B[i] = pb;
        d0 = (keep ? d1 : u0) - fact * pm;
        u0 = sh ? -fact * u1 : u1;
        b0 = (keep ? b1 : b0) - fact * pb;
    }
    if (!info && d0 == (T)0) info = n;  // DGTSV.f:160-163
    T x1 = b0 / d0, x2 = (T)0;
    B[n - 1] = x1;
    for (int q = n - 2; q >= 0; --q) {  // (row n-2 has F = 0 and x2 = 0)
        const T x = (B[q] - U[q] * x1 - F[q] * x2) / D[q];
        x2 = x1;
        x1 = x;
        B[q] = x;
    }
    return info;
}

// Row inputs of one element of a colour phase: B minus the I/K neighbour terms
// in LEQ_IKSWEEP's order (leqsol_mod.f:891-902), the coupling to the row
// above, and two planes' values at the row (the multiplier and the eliminated
// diagonal, or DL and A0).
template <typename T>
struct WholeArrays {
    gptr<const T> im, ip, km, kp, jp, bm, f, d;
    gptr<T> var;
};
template <typename T>
struct WholeRow {
    T b, im, ip, km, kp, vim, vip, vkm, vkp, f, d, u;
    __device__ __forceinline__ void load(const WholeArrays<T> &A, const WholeLines &w, int l, uint32_t c) {
        b = A.bm[c];
        im = A.im[c];
        ip = A.ip[c];
        vim = A.var[c + w.im[l]];
        vip = A.var[c + w.ip[l]];
        km = A.km[c];  // (in 2-D the K offsets are 0: in bounds, not used)
        kp = A.kp[c];
        vkm = A.var[c + w.km[l]];
        vkp = A.var[c + w.kp[l]];
        f = A.f[c];
        d = A.d[c];
        u = A.jp[c];
    }
    __device__ __forceinline__ T rhs(int do_k) const {
        const T two = b - im * vim - ip * vip;
        return do_k ? two - km * vkm - kp * vkp : two;
    }
};

// DGTSV itself on the block's lines.
template <typename T>
__device__ __forceinline__ WholeArrays<T> whole_arrays(const Sys<T> &S, int which) {
    const gptr<const T> a = to_global(S.a);
    const int64_t n3 = S.g.n3;
    WholeArrays<T> A;
    A.km = a;
    A.im = a + 2 * n3;
    A.ip = a + 4 * n3;
    A.jp = a + 5 * n3;
    A.kp = a + 6 * n3;
    A.bm = to_global((const T *)(which == 0 ? S.p : S.s));
    A.var = to_global(which == 0 ? S.phat : S.shat);
    A.f = a + n3;
    A.d = a + (int64_t)DiagPlane<T>::value * n3;
    return A;
}
template <typename T, int NT>
__device__ void whole_general(const Sys<T> &S, const WholeLines &w, int *linfo, int which) {
    extern __shared__ __align__(16) char whole_lds[];
    const DGrid &g = S.g;
    const int n = g.nj, ls = whole_stride(n), nl = w.n, tot = nl * n, do_k = g.do_k;
    T *__restrict__ F = (T *)whole_lds + kWholeFront, *__restrict__ B = F + S.lpb * ls, *__restrict__ U = B + S.lpb * ls,
                    *__restrict__ D = U + S.lpb * ls;
    const WholeArrays<T> A = whole_arrays(S, which);
    auto line_of = [&](int x) { return (int)div_by((uint32_t)x, g.mnj, g.snj); };
    __syncthreads();
    for (int x = threadIdx.x; x < tot; x += NT) {
        const int l = line_of(x), q = x - l * n, at = l * ls + q;
        WholeRow<T> r;
        r.load(A, w, l, w.c0[l] + (uint32_t)q);
        F[at] = q > 0 ? r.f : (T)0;
        B[at] = r.rhs(do_k);
        U[at] = q < n - 1 ? r.u : (T)0;
        D[at] = r.d;
    }
    __syncthreads();
    if ((int)threadIdx.x < nl) {
        const int ol = threadIdx.x * ls;
        linfo[threadIdx.x] = whole_dgtsv(F + ol, B + ol, U + ol, D + ol, n);
    }
    __syncthreads();
    for (int x = threadIdx.x; x < tot; x += NT) {
        const int l = line_of(x), q = x - l * n;
        // a line whose elimination hit a zero pivot keeps its values (leqsol_mod.f:910-914)
        if (!linfo[l]) A.var[w.c0[l] + (uint32_t)q] = B[l * ls + q];
    }
}

// The block's lines on their factored rows by DGTSV's own operations.
template <int NT>
__device__ void whole_exact(const Sys<double> &S, const WholeLines &w, int which, bool swaps) {
    extern __shared__ __align__(16) char whole_lds[];
    const DGrid &g = S.g;
    const int n = g.nj, ls = whole_stride(n), nl = w.n, tot = nl * n, do_k = g.do_k;
    double *F = (double *)whole_lds + kWholeFront, *B = F + S.lpb * ls, *U = B + S.lpb * ls, *D = U + S.lpb * ls;
    WholeArrays<double> A = whole_arrays(S, which);
    A.f = to_global((const double *)S.lf);
    if (swaps) A.jp = to_global((const double *)S.lu);
    const gptr<const double> ld = to_global((const double *)S.ld), lu2 = to_global((const double *)S.lu2);
    auto line_of = [&](int x) { return (int)div_by((uint32_t)x, g.mnj, g.snj); };
    const int ol = threadIdx.x * ls;
    __syncthreads();
    for (int x = threadIdx.x; x < tot; x += NT) {
        const int l = line_of(x), q = x - l * n, at = l * ls + q;
        const uint32_t c = w.c0[l] + (uint32_t)q;
        WholeRow<double> r;
        r.load(A, w, l, c);
        F[at] = q > 0 ? r.f : 0.0;
        B[at] = r.rhs(do_k);
        U[at] = q < n - 1 ? r.u : 0.0;
        D[at] = swaps ? lu2[c] : 0.0;
    }
    for (int x = threadIdx.x; x < 4 * nl; x += NT) {
        const int q = n + (x & 3);
        if (q < whole_rows(n)) F[(x >> 2) * ls + q] = 0.0;  // (no interchange behind the line)
    }
    __syncthreads();
    if ((int)threadIdx.x < nl) {
        if (swaps) whole_forward_swap(F + ol, B + ol, whole_rows(n));
        else whole_forward(F + ol, B + ol, whole_rows(n));
    }
    __syncthreads();
    for (int x = threadIdx.x; x < tot; x += NT) {
        const int l = line_of(x), q = x - l * n;
        F[l * ls + q] = ld[w.c0[l] + (uint32_t)q];
    }
    __syncthreads();
    if ((int)threadIdx.x < nl) whole_back_exact<true>(B + ol, U + ol, D + ol, F + ol, n);
    __syncthreads();
    for (int x = threadIdx.x; x < tot; x += NT) {
        const int l = line_of(x), q = x - l * n;
        A.var[w.c0[l] + (uint32_t)q] = B[l * ls + q];
    }
}

// One colour phase: block e takes lines [e.y*S.lpb, +S.lpb) of colour
// `param` (color_line).  which = 0 preconditions P into Phat, 1 S into Shat.
// FP32 tables (lines longer than the k_line_pcr_sys variants hold) always run
// DGTSV in LDS.
template <typename T>
__global__ void __launch_bounds__(kWholeThreads, 4) k_line_whole(const Sys<T> *__restrict__ sys,
                                                              const int2 *__restrict__ map, int param, int which) {
    extern __shared__ __align__(16) char whole_lds[];
    __shared__ WholeLines w;
    __shared__ int linfo[kWholeLines];  // DGTSV INFO per line
    const int2 e = map[blockIdx.x];
    if (e.x < 0) return;
    const Sys<T> &S = sys[e.x];
    auto *__restrict__ st = to_global(S.st);
    if (st->done || (which == 1 && st->s_exit)) return;
    if (e.y == 0 && threadIdx.x == 0) st->line_launches += 1;  // (timing: working launches)
    const DGrid &g = S.g;
    const bool few = whole_few(S.lpb);
    const int n = g.nj, ls = few ? stream_stride(n) : whole_stride(n), do_k = g.do_k;
    const int rows = whole_rows(n), held = few ? stream_rows(n) : rows;
    whole_lines(g, S.lstep, e.y, param, w);
    const int nl = w.n, tot = nl * n;
    // right-hand side (then the solution), upper coupling, and: multipliers
    // (then the eliminated diagonal) and its reciprocals, or DL (then the
    // second super-diagonal) and A0
    T *__restrict__ F = (T *)whole_lds + kWholeFront, *__restrict__ B = F + S.lpb * ls, *__restrict__ U = B + S.lpb * ls,
                    *__restrict__ D = U + S.lpb * ls;
    WholeArrays<T> A = whole_arrays(S, which);
    // (a line's rows are consecutive elements: element x is row x % n of line x / n)
    auto line_of = [&](int x) { return (int)div_by((uint32_t)x, g.mnj, g.snj); };
    if constexpr (sizeof(T) == sizeof(double)) {
        A.f = to_global((const T *)S.lf);
        A.d = to_global((const T *)S.ld);
        constexpr int K = 3;  // rows in flight per thread
        T td[kWholeElems];    // the diagonals wait for the multipliers' place
        int o[kWholeElems], any = 0, out = 0, own = 0;
#pragma unroll
        for (int k0 = 0; k0 < kWholeElems; k0 += K) {
            if (k0 * kWholeThreads >= tot) break;
            WholeRow<T> r[K];
            bool first[K], last[K];
#pragma unroll
            for (int k = 0; k < K; ++k) {
                const int x0 = (int)threadIdx.x + (k0 + k) * kWholeThreads;
                const int x = x0 < tot ? x0 : tot - 1;  // (past the end: the last row again)
                const int l = line_of(x), q = x - l * n;
                o[k0 + k] = l * ls + q;
                r[k].load(A, w, l, w.c0[l] + (uint32_t)q);
                first[k] = q == 0;
                last[k] = q == n - 1;
            }
#pragma unroll
            for (int k = 0; k < K; ++k) {
                F[o[k0 + k]] = first[k] ? (T)0 : r[k].f;
                any |= swapped(r[k].f);
                own |= own_dgtsv(r[k].f);
                const T b = r[k].rhs(do_k);
                out |= !solution_in_range((double)b);
                B[o[k0 + k]] = b;
                U[o[k0 + k]] = last[k] ? (T)0 : r[k].u;
                D[o[k0 + k]] = (T)refined_rcp(r[k].d);
                td[k0 + k] = r[k].d;
            }
        }
        if (out) w.odd = 1;
        if (own) w.own = 1;
        for (int x = threadIdx.x; x < 8 * nl; x += kWholeThreads) {
            const int q = n + (x & 7), at = (x >> 3) * ls + q;
            if (q < held) {  // identity rows
                F[at] = B[at] = U[at] = 0.0;
                D[at] = 1.0;
            }
        }
        const bool swaps = __syncthreads_or(any);
        if (swaps) {  // (or the block's mark is kOwnDgtsv, and the planes hold nothing)
            const gptr<const double> lu = to_global((const double *)S.lu), lu2 = to_global((const double *)S.lu2);
            for (int x = threadIdx.x; x < tot; x += kWholeThreads) {
                const int l = line_of(x), q = x - l * n;
                const uint32_t c = w.c0[l] + (uint32_t)q;
                U[l * ls + q] = lu[c];
                D[l * ls + q] = lu2[c];
            }
        }
        if (!swaps || !w.own) {
            // the solving wave: another one in each of the blocks that share a
            // CU (every 256th), so that they do not share a SIMD
            const int solver = (int)threadIdx.x - 64 * ((blockIdx.x >> 8) & 3);
            const bool mine = solver >= 0 && solver < nl;
            const int ol = solver * ls;
            // with interchanges eight lanes a line where they are few (past the
            // last line: it again, the same values): 30x90x3 13.5 -> 11.4 us, 64^3
            // 13.7 -> 12.0, 40x200x40 30 -> 21
            const bool eight = swaps && few && nl > 0 && solver >= 0 && solver < 64 && !w.odd;
            const int o8 = (solver >> 3 < nl ? solver >> 3 : nl - 1) * ls;
            if (eight) {
                whole_forward_swap8(F + o8, B + o8, held, threadIdx.x & 7);
            } else if (mine) {
                if (swaps) whole_forward_swap(F + ol, B + ol, rows);
                else whole_forward(F + ol, B + ol, rows);
            }
            __syncthreads();
#pragma unroll
            for (int k = 0; k < kWholeElems; ++k)
                if (k / K * K * kWholeThreads < tot) F[o[k]] = td[k];
            for (int x = threadIdx.x; x < 8 * nl; x += kWholeThreads) {
                const int q = n + (x & 7);
                if (q < held) F[(x >> 3) * ls + q] = 1.0;
            }
            // a right-hand side out of range, and its solution most likely is:
            // DGTSV's own operations at once
            const bool exact = __builtin_amdgcn_readfirstlane(w.odd);
            __syncthreads();
            if (eight) {
                whole_back_swap8(B + o8, U + o8, D + o8, F + o8, held, threadIdx.x & 7);
            } else if (mine) {
                if (exact && swaps) whole_back_exact<true>(B + ol, U + ol, D + ol, F + ol, n);
                else if (exact) whole_back_exact<false>(B + ol, U + ol, U + ol, F + ol, n);
                else if (swaps) whole_back_swap(B + ol, U + ol, D + ol, F + ol, rows);
                else whole_back(B + ol, U + ol, F + ol, D + ol, rows);
            }
            __syncthreads();
            int bad = 0;
            for (int x = threadIdx.x; x < tot; x += kWholeThreads) {
                const int l = line_of(x);
                bad |= !exact && !solution_in_range((double)B[l * ls + (x - l * n)]);
            }
            if (__syncthreads_or(bad)) {
                whole_exact<kWholeThreads>(S, w, which, swaps);
                return;
            }
            for (int x = threadIdx.x; x < tot; x += kWholeThreads) {
                const int l = line_of(x), q = x - l * n;
                A.var[w.c0[l] + (uint32_t)q] = B[l * ls + q];
            }
            return;
        }
    }
    whole_general<T, kWholeThreads>(S, w, linfo, which);
}

// The same phase of a system of more than one round of blocks, its lines
// streamed through kStreamBlocks blocks: block b takes the map entries b,
// b + gridDim.x, ...  One wave solves; the others read the next entry's rows
// into registers meanwhile (right-hand side, multiplier, upper coupling,
// diagonal, and the second super-diagonal where rows were interchanged).
// What bounded k_line_whole there was not the bytes: an LDS instruction costs a
// CU about 11 cycles whatever its active lanes, so four solving waves a CU of
// four lines each took twice as long over their chains as one does alone, and
// a block's loads, chain and store came one after the other.  With two solving
// waves of eight lines the chains fit beside the loads, and a phase moves what
// it moves (a fifth more than the arrays: the other colour's values twice) at
// 4.2 of the 5.1 TB/s of a copy: 256^3 233 -> 196 us, 170^3 71 -> 59 us,
// 150x201x180 76 -> 68 us.  Non-temporal loads of the arrays read once: 195 us
// at 256^3, but 48 for 42 us at 200x100x200, whose arrays the last-level cache
// holds.  An entry with a pivot or a value of its solution out of range
// is left for the end; with a right-hand side out of range it divides at once.

// Start cell and I/K neighbour offsets of line `lane` of a block, in every wave.
struct StreamLines {
    uint32_t c0, im, ip, km, kp;
    int n;
    int ends;  // some line is on a clamped end of I or K: its own neighbour
    __device__ __forceinline__ void set(const DGrid &g, uint64_t step, int j, int param, int lane) {
        int u = 0, v = 0;
        const int64_t first = entry_first(step, j);
        const bool ok = lane < entry_first(step, j + 1) - first &&
                        color_line(g.ni, g.nk, g.do_k ? 1 : 0, param, first + lane, u, v);
        const uint32_t c1 = (uint32_t)g.c1, c2 = (uint32_t)g.c2;
        c0 = ok ? (uint32_t)u * c1 + (uint32_t)v * c2 : 0u;
        im = (uint32_t)(nb_minus(u, g.ni, g.cyc_x) - u) * c1;
        ip = (uint32_t)(nb_plus(u, g.ni, g.cyc_x) - u) * c1;
        km = g.do_k ? (uint32_t)(nb_minus(v, g.nk, g.cyc_z) - v) * c2 : 0u;
        kp = g.do_k ? (uint32_t)(nb_plus(v, g.nk, g.cyc_z) - v) * c2 : 0u;
        n = __popcll(__ballot(ok));
        ends = __any(ok && (im == 0 || ip == 0 || (g.do_k && (km == 0 || kp == 0))));
    }
    static __device__ __forceinline__ uint32_t of(uint32_t v, int l) { return (uint32_t)__shfl((int)v, l, 64); }
};

static __global__ void __launch_bounds__(kStreamThreads, 4) k_line_stream(const Sys<double> *__restrict__ sys,
                                                                         const int2 *__restrict__ map, int nmap,
                                                                         int param, int which) {
    extern __shared__ __align__(16) char whole_lds[];
    __shared__ WholeLines w;
    __shared__ int linfo[kWholeLines];
    __shared__ int tiny;                          // the entry has a right-hand side out of range
    __shared__ int odd;                           // the entry has a pivot or a value of its solution out of range
    __shared__ uint32_t again[kStreamMost / 32];  // this block's entries that are left for the end
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    // another solving wave in each of the blocks that share a CU (every 256th)
    const int solver = (blockIdx.x >> 8) & 1;
    const int lt = (wave < solver ? wave : wave - 1) * 64 + lane;
    const int step = (int)gridDim.x;
    int it = blockIdx.x;
    int2 e = map[it];
    if (e.x < 0) return;
    const int id = e.x;
    const Sys<double> &S = sys[id];
    auto *__restrict__ st = to_global(S.st);
    if (st->done || (which == 1 && st->s_exit)) return;
    if (e.y == 0 && threadIdx.x == 0) st->line_launches += 1;  // (timing: working launches)
    if (threadIdx.x == 0) odd = tiny = 0;
    if (threadIdx.x < kStreamMost / 32) again[threadIdx.x] = 0;
    __syncthreads();
    const DGrid &g = S.g;
    const int n = g.nj, ls = stream_stride(n), do_k = g.do_k, rows = stream_rows(n), lpb = S.lpb;
    double *__restrict__ F = (double *)whole_lds + kWholeFront, *__restrict__ B = F + lpb * ls,
                         *__restrict__ U = B + lpb * ls, *__restrict__ D = U + lpb * ls;
    WholeArrays<double> A = whole_arrays(S, which);
    A.f = to_global((const double *)S.lf);
    A.d = to_global((const double *)S.ld);
    const gptr<const double> lu = to_global((const double *)S.lu), lu2 = to_global((const double *)S.lu2);
    // rows lt + k kStreamLoaders of the block's: row q of line l
    double b[kStreamElems], f[kStreamElems], u[kStreamElems], v[kStreamElems], d[kStreamElems];
    int lq[kStreamElems];
#pragma unroll
    for (int k = 0; k < kStreamElems; ++k) {
        const int x0 = lt + k * kStreamLoaders, x = x0 < lpb * n ? x0 : lpb * n - 1;
        const int l = (int)div_by((uint32_t)x, g.mnj, g.snj);
        lq[k] = l << 16 | (x - l * n);
    }
    StreamLines L;
    int tot = 0, out = 0;  // out: a right-hand side of the next entry is out of range
    // (opaque: what is formed from lq is formed again in each step and
    // not held in registers over the loop)
    auto fresh = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < kStreamElems; ++k) asm volatile("" : "+v"(lq[k]));
    };
    auto at = [&](int k) __attribute__((always_inline)) { return (lq[k] >> 16) * ls + (lq[k] & 0xffff); };
    auto here = [&](int k) __attribute__((always_inline)) { return lt + k * kStreamLoaders < tot; };
    // byte offset of its cell (a row past the entry's last: a row of
    // line 0, not used)
    auto cell = [&](int k) __attribute__((always_inline)) {
        const int l = lq[k] >> 16;
        return 8u * (StreamLines::of(L.c0, l < L.n ? l : 0) + (uint32_t)(lq[k] & 0xffff));
    };
    auto ld = [](gptr<const double> p, uint32_t o) __attribute__((always_inline)) {
        return *(gptr<const double>)((gptr<const char>)p + o);
    };
    auto rhs2 = [&](int k0) __attribute__((always_inline)) {
        if (k0 * kStreamLoaders >= L.n * n) return;
        double bb[2], m[2][4], y[2][4];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            if (k0 + k >= kStreamElems) break;
            const int l0 = lq[k0 + k] >> 16, l = l0 < L.n ? l0 : 0;
            const uint32_t c = cell(k0 + k);
            bb[k] = ld(A.bm, c);
            m[k][0] = ld(A.im, c);
            m[k][1] = ld(A.ip, c);
            m[k][2] = ld(A.km, c);  // (in 2-D the K offsets are 0: in bounds, not used)
            m[k][3] = ld(A.kp, c);
            y[k][0] = ld(A.var, c + 8u * StreamLines::of(L.im, l));
            y[k][1] = ld(A.var, c + 8u * StreamLines::of(L.ip, l));
            y[k][2] = ld(A.var, c + 8u * StreamLines::of(L.km, l));
            y[k][3] = ld(A.var, c + 8u * StreamLines::of(L.kp, l));
        }
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            if (k0 + k >= kStreamElems) break;
            const double two = bb[k] - m[k][0] * y[k][0] - m[k][1] * y[k][1];
            b[k0 + k] = do_k ? two - m[k][2] * y[k][2] - m[k][3] * y[k][3] : two;
            out |= !solution_in_range(b[k0 + k]);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    auto factors = [&](int sw) __attribute__((always_inline)) {
        const gptr<const double> up = sw ? lu : A.jp;
#pragma unroll
        for (int k = 0; k < kStreamElems; ++k) {
            if (k * kStreamLoaders >= L.n * n) break;
            const uint32_t c = cell(k);
            f[k] = ld(A.f, c);
            d[k] = ld(A.d, c);
            u[k] = ld(up, c);
            if (sw) v[k] = ld(lu2, c);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    auto mark = [&]() __attribute__((always_inline)) { return ld(A.f, 8u * StreamLines::of(L.c0, 0)); };  // (in every wave alike)
    // 1: rows interchanged, 2: DGTSV itself
    auto marked = [](double f) __attribute__((always_inline)) {
        return __builtin_amdgcn_readfirstlane((int)swapped(f) + (int)own_dgtsv(f));
    };
    // (both loops below take the same entries and meet at the same four
    // or five barriers an entry; apart, the solving wave's chains and the others'
    // rows do not share registers)
    auto next = [&]() __attribute__((always_inline)) {
        return it + step < nmap ? map[it + step] : make_int2(-1, 0);
    };
    int2 en = next();
    L.set(g, S.lstep, e.y, param, lane);
    double mk = mark();
    if (wave == solver) {
        for (;;) {
            const int nl = L.n, ends = L.ends;
            const bool more = en.x == id, mine = lane < nl;
            const int swp = marked(mk), ol = lane * ls;
            // (eight lanes a line; past the last line: it again, the same values)
            const int o8 = (lane >> 3 < nl ? lane >> 3 : nl - 1) * ls;
            if (more) L.set(g, S.lstep, en.y, param, lane);
            it += step;
            e = en;
            if (more) en = next();
            if (more) mk = mark();
            __syncthreads();  // the rows are there
            if (lane == 0) odd = 0;
            const bool exact = tiny, eight = swp && nl > 0 && nl <= 8 && !exact;
            if (eight) {
                whole_forward_swap8(F + o8, B + o8, rows, lane & 7);
            } else if (mine) {
                if (swp) whole_forward_swap(F + ol, B + ol, whole_rows(n));
                else whole_forward(F + ol, B + ol, whole_rows(n));
            }
            __syncthreads();  // forward pass done
            __syncthreads();  // the diagonals are there
            if (eight) {
                whole_back_swap8(B + o8, U + o8, D + o8, F + o8, rows, lane & 7);
            } else if (mine) {
                if (exact && swp) whole_back_exact<true>(B + ol, U + ol, D + ol, F + ol, n);
                else if (exact) whole_back_exact<false>(B + ol, U + ol, U + ol, D + ol, n);
                else if (swp) whole_back_swap(B + ol, U + ol, D + ol, F + ol, whole_rows(n));
                else whole_back(B + ol, U + ol, D + ol, F + ol, whole_rows(n));
            }
            __syncthreads();  // solved
            if (ends) __syncthreads();  // looked at
            if (!more) break;
        }
    } else {
        int swn = marked(mk);
        factors(swn);
#pragma unroll
        for (int k0 = 0; k0 < kStreamElems; k0 += 2) rhs2(k0);
        for (int nth = 0;; ++nth) {
            const bool more = en.x == id;
            const int nl = L.n, ends = L.ends, swp = swn;
            const uint32_t c0 = L.c0;  // start cells of the entry being solved
            tot = nl * n;
            fresh();
#pragma unroll
            for (int k = 0; k < kStreamElems; ++k) {
                if (k * kStreamLoaders >= tot) break;
                if (!here(k)) continue;
                const int o = at(k), q = lq[k] & 0xffff;
                F[o] = q > 0 ? f[k] : 0.0;
                B[o] = b[k];
                U[o] = q < n - 1 ? u[k] : 0.0;
                D[o] = swp ? v[k] : d[k];
            }
            if (out) tiny = 1;
            out = 0;
            for (int x = lt; x < 8 * nl; x += kStreamLoaders) {
                const int q = n + (x & 7), o = (x >> 3) * ls + q;
                if (q < rows) {  // identity rows
                    F[o] = B[o] = U[o] = 0.0;
                    D[o] = 1.0;
                }
            }
            if (more) L.set(g, S.lstep, en.y, param, lane);
            it += step;
            e = en;
            if (more) en = next();
            __syncthreads();  // the rows are there
            const int exact = tiny;
            if (more) mk = mark();
            if (!swp) {
#pragma unroll
                for (int k = 0; k < kStreamElems; ++k) d[k] = refined_rcp(d[k]);
            }
            if (more) {
                fresh();
                rhs2(0);
                fresh();
                rhs2(2);
                swn = marked(mk);
            }
            __syncthreads();  // forward pass done
            if (lt == 0) tiny = 0;
            fresh();
#pragma unroll
            for (int k = 0; k < kStreamElems; ++k) {
                if (k * kStreamLoaders >= tot) break;
                if (here(k)) F[at(k)] = d[k];
            }
            for (int x = lt; x < 8 * nl; x += kStreamLoaders) {
                const int q = n + (x & 7);
                if (q < rows) F[(x >> 3) * ls + q] = 1.0;
            }
            __syncthreads();  // the diagonals are there
            if (more) {
                fresh();
                factors(swn);
                fresh();
                rhs2(4);
            }
            fresh();
            uint32_t c[kStreamElems];
#pragma unroll
            for (int k = 0; k < kStreamElems; ++k)
                c[k] = 8u * (StreamLines::of(c0, lq[k] >> 16) + (uint32_t)(lq[k] & 0xffff));
            __syncthreads();  // solved
            fresh();
            // An entry out of range is left for the end.  Where a line is its
            // own neighbour, nothing of it may be stored before all of it has
            // been looked at.  (A barrier for every entry: 200x100x200 40.8 ->
            // 42.0 us.)
            int bad = swp == 2;
            if (ends) {
#pragma unroll
                for (int k = 0; k < kStreamElems; ++k) {
                    if (k * kStreamLoaders >= tot) break;
                    if (here(k)) bad |= !exact && !solution_in_range(B[at(k)]);
                }
                if (bad) odd = 1;
                __syncthreads();  // looked at
                bad = odd;
                fresh();
            }
            const bool keep = ends ? !bad : swp != 2;
#pragma unroll
            for (int k = 0; k < kStreamElems; ++k) {
                if (k * kStreamLoaders >= tot) break;
                if (!here(k) || !keep) continue;
                const double x = B[at(k)];
                bad |= !exact && !solution_in_range(x);
                *(gptr<double>)((gptr<char>)A.var + c[k]) = x;
            }
            if (bad) again[nth >> 5] |= 1u << (nth & 31);
            if (!more) break;
        }
    }
    __syncthreads();
    // the entries left (their inputs are as they were: the other colour's values
    // and, on clamped ends, their own, which were not stored)
    for (int k = 0, at = blockIdx.x; at < nmap && map[at].x == id; ++k, at += step) {
        if (!(again[k >> 5] >> (k & 31) & 1u)) continue;
        __syncthreads();
        whole_lines(g, S.lstep, map[at].y, param, w);
        const double m = w.n > 0 ? (double)to_global((const double *)S.lf)[w.c0[0]] : 0.0;
        if (own_dgtsv(m)) whole_general<double, kStreamThreads>(S, w, linfo, which);
        else whole_exact<kStreamThreads>(S, w, which, swapped(m));
    }
}

}  // namespace mfix
