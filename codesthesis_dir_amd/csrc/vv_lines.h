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
// which starts exactly; a line with a lane that differs (a chain that needs
// more rows to meet, as behind a single disturbance in a field of zeros) is
// done again row by row by the caller.  Per lane that is 2 (LWARM + 8 mb)
// rows in place of twice the line.
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
// its 53-bit significands; the 119 significands X with a residue up to 64
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
// x / LB, correctly rounded, two operations
__device__ __forceinline__ double line_div_settled(double x) { return __builtin_fma(x, LF, x * LFL); }

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
// Returns whether the lane's entry is proven.
template <bool TAB, bool MAX>
__device__ __forceinline__ bool line_fwd(double *S, int q0, int nb, int c, int mb, int P, int tf, double rp, double &mx)
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
    return c == 0 || b0 + LWB >= nb || same_bits(prev, ent);
}

// Rows back over the same blocks from the last, from y, the row after them
// (exact).  TAB: b, 1/b and c at words tb, tr, tc, laid out as the rows.  CYC:
// a's words at ta, zeros from word taw on (a block of zeros is there).
template <bool TAB, bool CYC>
__device__ __forceinline__ bool line_back(double *S, int q0, int nb, int c, int mb, int P, double y, int tb, int tr, int tc,
                                          int ta, int taw, double yn)
{
    const int b0 = c * mb;
    if (c) y = 0.0;
    auto block = [&](int b, bool own) {
        const int o = (b < nb ? nb - 1 - b : 0) * (LU + 1);
        y = block_back<TAB, CYC>(S, q0 + o, tb + o, tr + o, tc + o, ta + (o < taw ? o : taw), own && b < nb, yn, y);
    };
#pragma unroll 1
    for (int b = b0; b < b0 + LWB; ++b) block(b, c == 0);
    const double ent = y;
#pragma unroll 1
    for (int b = b0 + LWB; b < b0 + LWB + mb; ++b) block(b, true);
    const double prev = __shfl_up(y, 1, P);
    return c == 0 || b0 + LWB >= nb || same_bits(prev, ent);
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

// One line of the constant 1-4-1 rows, N rows at word Q and the closing row
// (tdma: one; ptdma: two) behind them, its tables from word 0 on: the settled
// rows by the line's P lanes as chunks with proven entries, the head's places
// and the closing rows by all of them alike.  Bound by the chain's
// instructions: 2 (40 + 8 mb) + 48 rows a lane, where one lane a line ran 2 n.
// Measured, the whole 2D kernel, one lane a line against this: 12.7 -> 12.8 us
// at 65x33, 41 -> 14.5 at 97x337, 42 -> 19 at 513x257, 154 -> 38 at 1025x513,
// 3265 -> 262 at 2049x2049 (where the tables had left LDS as well).  Returns
// whether every entry was proven.
template <bool CYC>
__device__ __forceinline__ bool line_solve(double *S, int Q, int N, int c, const LineTile &L, const LineTab &t)
{
    const int hb = t.hw / LU, nb = lblocks(N) - hb;   // blocks of the head, settled blocks
    const int X = Q + lwords(N), Q0 = Q + hb * (LU + 1), Th = LTC;
    double rp = 0.0, mx = 0.0;
#pragma unroll 1
    for (int b = 0; b < hb; ++b) rp = block_fwd<true>(S, Q + b * (LU + 1), Th + b * LU, c == 0, rp);
    bool ok = true;
    if (nb > 0) {
        ok = line_fwd<false, CYC>(S, Q0, nb, c, L.mb, L.P, 0, rp, mx);
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
        ok = line_back<false, CYC>(S, Q0, nb, c, L.mb, L.P, y, 0, 0, 0, t.Ta + o, t.taw - o, yn) && ok;
        y = S[Q0];
    }
#pragma unroll 1
    for (int b = hb - 1; b >= 0; --b)
        y = block_back<true, CYC>(S, Q + b * (LU + 1), Th + t.hw + b * LU, Th + 2 * t.hw + b * LU, Th + 3 * t.hw + b * LU,
                                  t.Ta + b * (LU + 1), c == 0, yn, y);
    return ok;
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
