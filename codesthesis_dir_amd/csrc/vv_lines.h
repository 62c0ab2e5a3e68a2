// vv_lines.h -- the reference's line recurrences, split into chunks with
// proven entries (device code; included by the .hip files only).
//
// tdma and ptdma are chains of one multiply-subtract per row going forward
// and one division per row coming back, and the parity bar is their bits, so
// the rows cannot be reassociated.  But both chains forget: with the settled
// pivots of the 1-4-1 rows a row's value depends on the one w rows before it
// by 0.268^w only, so a chain started anywhere meets the true one bit for
// bit after about 30 rows (measured on random and smooth lines: 8 % of the
// chains still differ after 30 rows, 0.035 % after 34, none of 20000 after
// 36).  P lanes of one wavefront therefore share a line: each starts LWARM
// rows before its own rows, and at the end compares the value it entered its
// own rows with against the one its predecessor left them with.  Equal bits
// in every lane prove the whole chain, by induction from the first lane,
// which starts exactly.  Per lane that is 2 (LWARM + 8 mb) rows in place of
// twice the line.
//
// Where a lane differs, the chain is run again from that lane to its end by
// one lane (line_fwd_again, line_back_again), out of the same LDS.  That takes
// a chain that needs more rows to meet: one through rows whose right-hand
// sides vanish (or fall off faster than 0.268 a row) behind a disturbance,
// where all the chain holds is the disturbance's tail, which lasts 565 rows
// until it underflows.  Wall layers before a core that is constant to the last
// bit are such fields, a tank started from a uniform temperature without noise
// among them.
//
// A line's N rows fill whole blocks of 8 from the back: row q is at place
// p = q + shift, the places before row 0 hold zeros.  LDS keeps one word of
// padding per block (lrow), so that lanes 8 mb rows apart read different
// banks.  The rows are overwritten in place: the lanes run in lockstep, and
// a lane that only warms up over a row reads it at least mb blocks before
// the row's owner writes it.
//
// One wavefront issues an instruction every 5 to 8 cycles here, so what
// bounds a chain is its instructions per row (2 forward, 4 or 5 back, and
// the LDS accesses two rows at a time), not the arithmetic's latency: no
// per-row selects, no table reads for settled rows, stores by one lane where
// all lanes hold the same value (the stores of many lanes to one word go one
// by one).
#pragma once

#include <hip/hip_runtime.h>

#include <vector>

namespace vv {

constexpr int LU = 8;                 // rows per block
constexpr int LWB = 5;                // warm-up blocks
constexpr int LWARM = LWB * LU;       // warm-up rows
constexpr int LHEAD = 24;             // places of the head: rows before the settled ones (16) and the shift

// The settled rows of the 1-4-1 elimination: factor 1/b, pivot b (the fixed
// point of b = 4 - 1/b in double precision, reached within 16 rows).
constexpr double LB = 0x1.ddb3d742c2655p+1, LF = 0x1.126145e9ecd56p-2;
// 1/LB - LF, rounded.  x/LB = RN(x LF + RN(x LFL)) for every x without
// underflow: the sum is within 2^-106.3 of the quotient, and a quotient that
// near a rounding boundary N/2^k (k = 53, 54) needs |X 2^k - N B| <= 1 for
// its 53-bit significands; the 137 significands X with a residue up to 64
// were enumerated and all round right (tests/test_lines_cpu.py).
constexpr double LFL = 0x1.49c290bb649bfp-56;

__host__ __device__ inline int lrow(int p) { return p + (p >> 3); }
// whole blocks of N rows, the places before row 0, LDS words of the blocks
__host__ __device__ inline int lblocks(int N) { return (N + LU - 1) / LU; }
__host__ __device__ inline int lshift(int N) { return lblocks(N) * LU - N; }
__host__ __device__ inline int lwords(int N) { return lblocks(N) * (LU + 1); }
// words of a line with its nx closing words, odd: lines side by side start
// in different banks
__host__ __device__ inline int lpitch(int N, int nx) { return (lwords(N) + nx) | 1; }
// blocks of the head, blocks behind it
__host__ __device__ inline int lheadb(int N) { return lblocks(N) < LHEAD / LU ? lblocks(N) : LHEAD / LU; }

// nb blocks on P lanes: blocks per lane beyond the warm-up
__host__ __device__ inline int line_mb(int nb, int P)
{
    const int m = (nb - LWB + P - 1) / P;
    return m < 1 ? 1 : m;
}

// x / b for b > 0 with rb = RN(1/b), correctly rounded (Markstein's
// correction: q0 is within an ulp, the remainder is exact in one FMA; -t
// keeps the sign of a zero quotient)
__device__ __forceinline__ double line_div(double x, double b, double rb)
{
    const double q0 = x * rb;
    const double t = __builtin_fma(b, q0, -x);
    return __builtin_fma(-t, rb, q0);
}
// x / LB, correctly rounded, two operations; x LFL underflows for quotients
// that are tiny(), which the chunks leave to line_div
__device__ __forceinline__ double line_div_settled(double x) { return __builtin_fma(x, LF, x * LFL); }

__device__ __forceinline__ bool tiny(double y) { return y != 0.0 && fabs(y) < 0x1p-960; }

__device__ __forceinline__ bool same_bits(double a, double b)
{
    return __double_as_longlong(a) == __double_as_longlong(b);
}

// orders this wavefront's LDS accesses (the hardware keeps them in order;
// this keeps the compiler from moving them)
__device__ __forceinline__ void wave_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Every place in LDS below is a word of S, the kernel's dynamic LDS, and not
// a pointer: a pointer that goes through a struct or a choice would make the
// accesses generic (flat) ones.

// What a lane's chunk ends with: whether its entry is proven, the value its
// last row leaves.
struct LaneEnd {
    bool ok;
    double exit;
};

// the first of a line's P lanes whose entry is not proven; P if there is none
__device__ __forceinline__ int line_first_bad(bool ok, int P)
{
    unsigned long long m = __ballot(!ok) >> ((threadIdx.x & 63) & ~(P - 1));
    if (P < 64) m &= (1ull << P) - 1;
    return m ? __ffsll(m) - 1 : P;
}

// Forward r_p = r_p - f_p r_{p-1} over one block at word q, all lanes of the
// line alike; TAB: factors at word tf, settled ones otherwise.
template <bool TAB>
__device__ __forceinline__ double block_fwd(double *S, int q, int tf, bool store, double rp)
{
    double r[LU], f[LU];
#pragma unroll
    for (int u = 0; u < LU; ++u) {
        r[u] = S[q + u];
        if (TAB) f[u] = S[tf + u];
    }
    wave_fence();
#pragma unroll
    for (int u = 0; u < LU; ++u) {
        rp = r[u] - (TAB ? f[u] : LF) * rp;
        r[u] = rp;
    }
    if (store) {
#pragma unroll
        for (int u = 0; u < LU; ++u) S[q + u] = r[u];
    }
    wave_fence();
    return rp;
}

// Back y_p = (r_p - c_p y_{p+1} [- a_p yn]) / b_p over one block; TAB: b at
// word tb, 1/b at tr and (CYC false) c at tc; CYC: a at ta.  Settled rows
// and all rows of CYC have c = 1.
template <bool TAB, bool CYC>
__device__ __forceinline__ double block_back(double *S, int q, int tb, int tr, int tc, int ta, bool store, double yn, double y)
{
    double r[LU], b[LU], e[LU], g[LU], s[LU];
#pragma unroll
    for (int u = 0; u < LU; ++u) {
        r[u] = S[q + u];
        if (TAB) {
            b[u] = S[tb + u];
            e[u] = S[tr + u];
            if (!CYC) g[u] = S[tc + u];
        }
        if (CYC) s[u] = S[ta + u];
    }
    wave_fence();
    if (CYC) {
#pragma unroll
        for (int u = 0; u < LU; ++u) s[u] = s[u] * yn;
    }
#pragma unroll
    for (int u = LU - 1; u >= 0; --u) {
        double x = r[u] - ((TAB && !CYC) ? g[u] * y : y);
        if (CYC) x = x - s[u];
        y = TAB ? line_div(x, b[u], e[u]) : line_div_settled(x);
        r[u] = y;
    }
    if (store) {
#pragma unroll
        for (int u = 0; u < LU; ++u) S[q + u] = r[u];
    }
    wave_fence();
    return y;
}

// Rows forward over the nb > 0 blocks at q0 (block 0 first) from rp, the row
// before block 0 (exact), on the P lanes of the line, this one c; every lane
// runs LWB + mb blocks (past the last block it reads that one and stores
// nothing).  TAB: factors at word tf, laid out as the rows; settled ones
// otherwise.  MAX: mx gathers |r| of the rows behind the first LWB blocks.
template <bool TAB, bool MAX>
__device__ __forceinline__ LaneEnd line_fwd(double *S, int q0, int nb, int c, int mb, int P, int tf, double rp, double &mx)
{
    const int b0 = c * mb;
    if (c) rp = 0.0;
#pragma unroll 1
    for (int t = 0; t < LWB; ++t) {
        const int b = b0 + t, o = (b < nb ? b : nb - 1) * (LU + 1);
        rp = block_fwd<TAB>(S, q0 + o, tf + o, c == 0 && b < nb, rp);
    }
    const double ent = rp;
#pragma unroll 1
    for (int b = b0 + LWB; b < b0 + LWB + mb; ++b) {
        const int o = (b < nb ? b : nb - 1) * (LU + 1), q = q0 + o;
        rp = block_fwd<TAB>(S, q, tf + o, b < nb, rp);
        if (MAX && b < nb) {
#pragma unroll
            for (int u = 0; u < LU; ++u) mx = fmax(mx, fabs(S[q + u]));
        }
    }
    const double prev = __shfl_up(rp, 1, P);
    return {c == 0 || b0 + LWB >= nb || same_bits(prev, ent), rp};
}

// Rows back over the same blocks from the last, from y, the row after them
// (exact).  TAB: b, 1/b and c at words tb, tr, tc, laid out as the rows;
// settled ones otherwise, and a lane that enters or leaves its rows with a
// tiny() value is not proven, nor is the first so if it starts from one.  CYC:
// a's words at ta, zeros from word taw on (a block of zeros is there).
template <bool TAB, bool CYC>
__device__ __forceinline__ LaneEnd line_back(double *S, int q0, int nb, int c, int mb, int P, double y, int tb, int tr, int tc,
                                             int ta, int taw, double yn)
{
    const int b0 = c * mb;
    if (c) y = 0.0;
    bool small = !TAB && tiny(y);
    auto block = [&](int b, bool own) {
        const int o = (b < nb ? nb - 1 - b : 0) * (LU + 1);
        y = block_back<TAB, CYC>(S, q0 + o, tb + o, tr + o, tc + o, ta + (o < taw ? o : taw), own && b < nb, yn, y);
    };
#pragma unroll 1
    for (int b = b0; b < b0 + LWB; ++b) block(b, c == 0);
    const double ent = y;
    if (!TAB) small |= tiny(y);
#pragma unroll 1
    for (int b = b0 + LWB; b < b0 + LWB + mb; ++b) block(b, true);
    if (!TAB) small |= tiny(y);
    const double prev = __shfl_up(y, 1, P);
    return {c == 0 ? !small : b0 + LWB >= nb || (same_bits(prev, ent) && !small), y};
}

// The rows of a line whose entries were not proven, once more, from the first
// such lane `bad` to the end: put(b0, b1) restores the right-hand sides of
// blocks b0..b1-1 (all lanes of the line), then one lane runs the chain with
// the next block's rows already on their way, which leaves it the chain's own
// latency: 2 dependent operations a row forward, 4 back (with the full
// division, as the tails end in tiny() values; the two-operation one where it
// holds made no difference).  The 2D lines of a step (two launches) on wall
// layers before a flat core, beside noise: 85 and 38 us at 513x257, 214 and
// 66 at 1025x513, 1160 and 265 at 2049x2049.  One lane a line takes 81, 292
// and 3490 us on any field; the redo from tables in memory and over the whole
// line took 272, 830 and 5050.
template <bool TAB, bool MAX, class Put>
__device__ __forceinline__ void line_fwd_again(double *S, int q0, int nb, int c, int mb, int P, int bad, int tf, double exit,
                                               double &mx, Put put)
{
    const int k0 = bad * mb + LWB;
    double rp = __shfl(exit, bad - 1, P);
    wave_fence();
    put(k0, nb);
    wave_fence();
    if (c) return;
    double r[2][LU], f[2][LU];
    auto load = [&](int k, int s) {
        const int o = min(k, nb - 1) * (LU + 1);
#pragma unroll
        for (int u = 0; u < LU; ++u) {
            r[s][u] = S[q0 + o + u];
            if (TAB) f[s][u] = S[tf + o + u];
        }
    };
    auto run = [&](int k, int s) {
#pragma unroll
        for (int u = 0; u < LU; ++u) {
            rp = r[s][u] - (TAB ? f[s][u] : LF) * rp;
            S[q0 + k * (LU + 1) + u] = rp;
            if (MAX) mx = fmax(mx, fabs(rp));
        }
    };
    load(k0, 0);
#pragma unroll 1
    for (int k = k0; k < nb; k += 2) {
        load(k + 1, 1);
        run(k, 0);
        load(k + 2, 0);
        if (k + 1 < nb) run(k + 1, 1);
    }
}

// Back, from y for the first lane: the eliminated rows that the chain from
// `bad` on overwrote come first, every lane's own from the row before them
// (rpre), which the lane read before.
template <bool TAB, bool CYC, class Put>
__device__ __forceinline__ void line_back_again(double *S, int q0, int nb, int c, int mb, int P, int bad, int tf, double rpre,
                                                double y, double exit, int tb, int tr, int tc, int ta, int taw, double yn, Put put)
{
    const int k0 = nb - 1 - (bad ? bad * mb + LWB : 0);
    const double prev = __shfl(exit, max(bad - 1, 0), P);
    if (bad) y = prev;
    wave_fence();
    put(0, k0 + 1);
    wave_fence();
    if (c >= bad)
#pragma unroll 1
        for (int k = max(0, nb - (c + 1) * mb - LWB); k <= nb - 1 - (c ? c * mb + LWB : 0); ++k)
            rpre = block_fwd<TAB>(S, q0 + k * (LU + 1), tf + k * (LU + 1), true, rpre);
    wave_fence();
    if (c) return;
    double r[2][LU], b[2][LU], e[2][LU], g[2][LU];
    auto load = [&](int k, int s) {
        const int o = max(k, 0) * (LU + 1), oa = ta + (o < taw ? o : taw);
#pragma unroll
        for (int u = 0; u < LU; ++u) {
            r[s][u] = S[q0 + o + u];
            if (TAB) {
                b[s][u] = S[tb + o + u];
                e[s][u] = S[tr + o + u];
            }
            if (TAB || CYC) g[s][u] = S[(CYC ? oa : tc + o) + u];
        }
    };
    auto run = [&](int k, int s) {
#pragma unroll
        for (int u = LU - 1; u >= 0; --u) {
            double x = r[s][u] - ((TAB && !CYC) ? g[s][u] * y : y);
            if (CYC) x = x - g[s][u] * yn;
            y = TAB ? line_div(x, b[s][u], e[s][u]) : line_div(x, LB, LF);
            S[q0 + k * (LU + 1) + u] = y;
        }
    };
    load(k0, 0);
#pragma unroll 1
    for (int k = k0; k >= 0; k -= 2) {
        load(k - 1, 1);
        run(k, 0);
        load(k - 2, 0);
        if (k > 0) run(k - 1, 1);
    }
}

// The eliminated row before the rows that lane c takes back; exists: whether
// there is a row before block 0 at q0.
__device__ __forceinline__ double line_row_before(const double *S, int q0, int nb, int c, int mb, bool exists)
{
    const int k = max(0, nb - (c + 1) * mb - LWB);
    return (k > 0 || exists) ? S[q0 + k * (LU + 1) - 2] : 0.0;
}

// How lines are split: P lanes a line (mb blocks each beyond the warm-up), T
// lines a workgroup.
struct LineTile {
    int P, lgP, T, mb;
};

// Words of the tables in LDS: LTC closing words, then over the head's places
// f | b | 1/b | c (tdma) or f | b | 1/b (ptdma, CYC), and for CYC a over all
// places (zeros left out, a block of zeros behind) and the factors of rn,
// g_p = f2 of the next place, in whole blocks.
constexpr int LTC = 8;
struct LineTab {
    int hw;                 // places of the head
    int Ta, Tg, taw, nf;    // CYC: words of a and g, words of a before its zeros, blocks of g
};

// Place of row q in a line's LDS: the N rows' places, the closing rows behind
// them.
__device__ __forceinline__ int line_pos(int q, int N) { return q < N ? lrow(q + lshift(N)) : lwords(N) + (q - N); }

// One line of the constant 1-4-1 rows, N rows at word Q and the closing row
// (tdma: one; ptdma: two) behind them, its tables from word 0 on: the settled
// rows by the line's P lanes as chunks with proven entries, the head's places
// and the closing rows by all of them alike.  rhs(q): the right-hand side of
// row q, for settled rows that are done again (none of them an end row of the
// line: those are in the head or close it).  Bound by the chain's
// instructions: 2 (40 + 8 mb) + 48 rows a lane, where one lane a line ran 2 n.
// Measured, the whole 2D kernel, one lane a line against this: 12.7 -> 12.8 us
// at 65x33, 41 -> 14.5 at 97x337, 42 -> 19 at 513x257, 154 -> 33 at 1025x513,
// 3265 -> 237 at 2049x2049 (where the tables had left LDS as well).
template <bool CYC, class Rhs>
__device__ __forceinline__ void line_solve(double *S, int Q, int N, int c, const LineTile &L, const LineTab &t, Rhs rhs)
{
    const int hb = t.hw / LU, nb = lblocks(N) - hb;   // blocks of the head, settled blocks
    const int X = Q + lwords(N), Q0 = Q + hb * (LU + 1), Th = LTC;
    double rp = 0.0, mx = 0.0;
#pragma unroll 1
    for (int b = 0; b < hb; ++b) rp = block_fwd<true>(S, Q + b * (LU + 1), Th + b * LU, c == 0, rp);
    auto put = [&](int b0, int b1) {
        const int at = hb * LU + b0 * LU - lshift(N), n = (b1 - b0) * LU;
#pragma unroll 4
        for (int e = c; e < n; e += L.P) S[Q0 + b0 * (LU + 1) + lrow(e)] = rhs(at + e);
    };
    if (nb > 0) {
        const LaneEnd l = line_fwd<false, CYC>(S, Q0, nb, c, L.mb, L.P, 0, rp, mx);
        const int bad = line_first_bad(l.ok, L.P);
        if (bad < L.P) line_fwd_again<false, CYC>(S, Q0, nb, c, L.mb, L.P, bad, 0, l.exit, mx, put);
        wave_fence();
        rp = S[X - 2];   // the last place
    }
    // closing rows
    double y, yn = 0.0;
    if (CYC) {
        // rn takes f2_j r_{j-1} of every row in the reference's order;
        // |f2_j+1| = |f2_j| / b_j falls off as 0.268^j, so once the rest
        // cannot move rn's last bit (|f2| max|r| below 2^-57 |rn|) it is
        // left out
        if (nb > LWB) atomicMax(reinterpret_cast<unsigned long long *>(S) + X + 2, (unsigned long long)__double_as_longlong(mx));
        wave_fence();
        double rn = S[X + 1];
        const double m = S[X + 2];
        const int free = hb + LWB;   // blocks that m does not cover
#pragma unroll 1
        for (int b = 0; b < t.nf; ++b) {
            double g[LU], r[LU];
#pragma unroll
            for (int u = 0; u < LU; ++u) {
                g[u] = S[t.Tg + b * LU + u];
                r[u] = S[Q + b * (LU + 1) + u];
            }
            if (b >= free && fabs(g[0]) * m <= 0x1p-57 * fabs(rn)) break;
#pragma unroll
            for (int u = 0; u < LU; ++u) rn = rn - g[u] * r[u];
        }
        const double rn1 = S[X] - S[0] * rp;
        rn = rn - S[1] * rp;
        rn = rn - S[2] * rn1;
        yn = line_div(rn, S[3], S[4]);
        y = line_div(rn1 - S[5] * yn, S[6], S[7]);
        wave_fence();
        if (c == 0) {
            S[X + 1] = yn;
            S[X] = y;
        }
    } else {
        rp = S[X] - S[0] * rp;
        y = line_div(rp, S[1], S[2]);
        wave_fence();
        if (c == 0) S[X] = y;
    }
    if (nb > 0) {
        const int o = hb * (LU + 1);
        const double rpre = line_row_before(S, Q0, nb, c, L.mb, true);
        wave_fence();
        const LaneEnd l = line_back<false, CYC>(S, Q0, nb, c, L.mb, L.P, y, 0, 0, 0, t.Ta + o, t.taw - o, yn);
        const int bad = line_first_bad(l.ok, L.P);
        if (bad < L.P)
            line_back_again<false, CYC>(S, Q0, nb, c, L.mb, L.P, bad, 0, rpre, y, l.exit, 0, 0, 0, t.Ta + o, t.taw - o, yn, put);
        wave_fence();
        y = S[Q0];
    }
#pragma unroll 1
    for (int b = hb - 1; b >= 0; --b)
        y = block_back<true, CYC>(S, Q + b * (LU + 1), Th + t.hw + b * LU, Th + 2 * t.hw + b * LU, Th + 3 * t.hw + b * LU,
                                  t.Ta + b * (LU + 1), c == 0, yn, y);
}

// Host side: the closing words (at most LTC) and the head's tables in that
// order, the places before row 0 neutral (f = 0, b = 1).  Returns whether
// every row from the 17th on has the settled factor and pivot and c = 1, as
// the chunks take them.
inline bool line_pack_head(std::vector<double> &t, const double *f, const double *b, const double *c, int N, bool with_c,
                           const std::vector<double> &close)
{
    const int sh = lshift(N), hw = lheadb(N) * LU;
    t = close;
    t.resize(LTC, 0.0);
    for (int p = 0; p < hw; ++p) t.push_back(p < sh ? 0.0 : f[p - sh]);
    for (int p = 0; p < hw; ++p) t.push_back(p < sh ? 1.0 : b[p - sh]);
    for (int p = 0; p < hw; ++p) t.push_back(p < sh ? 1.0 : 1.0 / b[p - sh]);
    bool ok = true;
    if (with_c)
        for (int p = 0; p < hw; ++p) t.push_back(p < sh ? 1.0 : c[p - sh]);
    for (int q = 0; q < N; ++q) {
        if (!with_c || q + sh >= hw) ok = ok && c[q] == 1.0;
        if (q + sh >= hw) ok = ok && f[q] == LF && b[q] == LB;
    }
    return ok;
}

}  // namespace vv
