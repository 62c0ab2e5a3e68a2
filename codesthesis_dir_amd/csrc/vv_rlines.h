// The last stage of the 3D direct Poisson solves: per (y or phi mode q, z
// eigenvalue l) a tridiagonal system along the n = i1 rows,
//
//   sub_i x_{i-1} + (dia_i + mu_q w_i + lam_l) x_i + sup_i x_{i+1} = y_i,
//
// whose first and last rows may have a coefficient two points inward (e1,
// en), removed with their neighbour rows.  The operators do not change during
// a run, so the reciprocal pivots r_i of the elimination are tabulated once
// (k_rline_pivots) and both sweeps are first-order recurrences,
//
//   y_i <- r_i y_i - (sub_i r_i) y_{i-1},   x_i = y_i - (sup_i r_i) x_{i+1},
//
// without a division, which chunks of rows can run side by side: a chunk is
// an affine map of the value entering it.
#pragma once
#include "vv_xcd.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>

namespace vv {

struct RLines {
    const double *rt;    // sub | dia | sup | w, i1 each
    const double *lz, *lq;
    double *piv;         // [q][i][l]: the reciprocal pivots
    int i1, j1, nq;
    int half;            // >0: mode q in (0, half) has a second right-hand side, at row half + q of T
    int w;               // 0: w = 1 throughout (rt has no fourth part)
    double e1, en;
};

__device__ __forceinline__ double rline_diag(const RLines &L, int i, double mu, double lam)
{
    return L.w ? L.rt[L.i1 + i] + mu * L.rt[3 * L.i1 + i] + lam : L.rt[L.i1 + i] + mu + lam;
}

// the two end rows with their outer coefficient removed: the neighbour row's
// weight, the diagonal and the coupling inward
struct REnd { double f, d, b; };

__device__ __forceinline__ REnd rline_first(const RLines &L, double mu, double lam)
{
    const double *sub = L.rt, *sup = L.rt + 2 * L.i1;
    REnd h{0.0, rline_diag(L, 0, mu, lam), sup[0]};
    if (L.e1 != 0.0) {
        h.f = L.e1 / sup[1];
        h.d -= h.f * sub[1];
        h.b -= h.f * rline_diag(L, 1, mu, lam);
    }
    return h;
}

__device__ __forceinline__ REnd rline_last(const RLines &L, double mu, double lam)
{
    const int n = L.i1;
    const double *sub = L.rt, *sup = L.rt + 2 * n;
    REnd h{0.0, rline_diag(L, n - 1, mu, lam), sub[n - 1]};
    if (L.en != 0.0) {
        h.f = L.en / sub[n - 2];
        h.d -= h.f * sup[n - 2];
        h.b -= h.f * rline_diag(L, n - 2, mu, lam);
    }
    return h;
}

static __global__ void __launch_bounds__(64) k_rline_pivots(RLines L)
{
    const int n = L.i1, line = blockIdx.x * 64 + threadIdx.x;
    if (line >= L.nq * L.j1) return;
    const int q = line / L.j1, l = line - q * L.j1;
    const double mu = L.lq[q], lam = L.lz[l];
    const REnd hd = rline_first(L, mu, lam), tl = rline_last(L, mu, lam);
    double *p = L.piv + (size_t)q * n * L.j1 + l;
    double c = 0.0;
    for (int i = 0; i < n; ++i) {
        const double a = i < n - 1 ? L.rt[i] : tl.b, d = i == 0 ? hd.d : i < n - 1 ? rline_diag(L, i, mu, lam) : tl.d;
        const double r = 1.0 / (i ? d - a * c : d);
        p[(size_t)i * L.j1] = r;
        c = (i ? L.rt[2 * n + i] : hd.b) * r;
    }
}

// Line t of the rows of T: modes with two right-hand sides have them next to
// each other, for the second to find the pivots in the XCD's L2.
__device__ __forceinline__ void rline_place(const RLines &L, int t, int &s, int &q, int &l)
{
    const int k = t / L.j1;
    l = t - k * L.j1;
    if (L.half) {
        q = (k + 1) >> 1;
        s = (k > 0 && !(k & 1)) ? L.half + q : q;
    } else {
        s = q = k;
    }
}

constexpr int RLT = 16;   // lines of a workgroup, neighbouring in l: 128 bytes of a row

// RLT lines a workgroup, U rows of one a thread, in registers from load to
// store (U = 16: 128 of them, and 3 dwords in scratch): the rows of T are read once and written once, and the pivots read
// once, which bounds it.  A lane a line, as before, formed its pivots with
// three divisions a row and went to memory for every group of rows: 75.8 us a
// solve at 129x129x257 and 17.6 at 33x33x161, now 30.5 and 5.5; at 512x256x256
// 308, now 212, side by side with the other stream's kernels.  (A tile of
// lines in LDS solved from both ends by one wavefront: 48.7, 6.5 and 691 us,
// LDS holding too few lines to cover the chain.)
template <int U>
__global__ void __launch_bounds__(1024) k_rlines(RLines L, double *__restrict__ T, int nlines, int nch)
{
    extern __shared__ double2 sh[];   // each chunk's map: forward, then back
    const int n = L.i1, j1 = L.j1, c = threadIdx.x & (RLT - 1), ch = threadIdx.x / RLT, i0 = ch * U;
    // an XCD's workgroups take neighbouring lines, which share 128-byte lines
    const int tile = xcd_padded((nlines + RLT - 1) / RLT);
    if (tile < 0) return;
    const int t = tile * RLT + c;
    const bool act = t < nlines && i0 < n;
    int s, q, l;
    rline_place(L, min(t, nlines - 1), s, q, l);
    double *x0 = T + (size_t)s * n * j1 + l;
    double x[U], g[U], b[U], f = 1.0, y = 0.0;
    if (act) {
        const double *p = L.piv + (size_t)q * n * j1 + l;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const size_t o = (size_t)min(i0 + u, n - 1) * j1;
            x[u] = x0[o];
            b[u] = p[o];
        }
        double xb = 0.0;   // row n-2 for the last row's fold
        const bool end = i0 + U >= n;
        if (end) xb = x0[(size_t)(n - 2) * j1];
        const double mu = L.lq[q], lam = L.lz[l];
        if (i0 == 0) {
            const REnd h = rline_first(L, mu, lam);
            x[0] -= h.f * x[1];
            g[0] = 0.0;
            x[0] *= b[0];
            b[0] = -h.b * b[0];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = i0 + u;
            if (i >= n) { x[u] = g[u] = b[u] = 0.0; continue; }
            if (u == 0 && i0 == 0) continue;
            const double r = b[u];
            if (i < n - 1) {
                g[u] = -(L.rt[i] * r);
                b[u] = -(L.rt[2 * n + i] * r);
            } else {
                const REnd h = rline_last(L, mu, lam);
                x[u] -= h.f * xb;
                g[u] = -(h.b * r);
                b[u] = 0.0;
            }
            x[u] *= r;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            y = __builtin_fma(g[u], y, x[u]);
            f *= g[u];
        }
        sh[ch * RLT + c] = make_double2(y, f);
    }
    __syncthreads();
    double2 *bk = sh + nch * RLT;
    if (act) {
        y = 0.0;
        for (int k = 0; k < ch; ++k) {
            const double2 v = sh[k * RLT + c];
            y = __builtin_fma(v.y, y, v.x);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) x[u] = y = __builtin_fma(g[u], y, x[u]);
        y = 0.0;
        f = 1.0;
#pragma unroll
        for (int u = U - 1; u >= 0; --u) {
            y = __builtin_fma(b[u], y, x[u]);
            f *= b[u];
        }
        bk[ch * RLT + c] = make_double2(y, f);
    }
    __syncthreads();
    if (!act) return;
    y = 0.0;
    for (int k = nch - 1; k > ch; --k) {
        const double2 v = bk[k * RLT + c];
        y = __builtin_fma(v.y, y, v.x);
    }
#pragma unroll
    for (int u = U - 1; u >= 0; --u) {
        y = __builtin_fma(b[u], y, x[u]);
        if (i0 + u < n) x0[(size_t)(i0 + u) * j1] = y;
    }
}

// Longer lines than a workgroup's threads hold, one a lane, bound by its trips
// to memory: U rows with their pivots and coefficients each (the coefficients
// row by row, as they may share memory with T for all that the compiler knows,
// took 485 us a solve at 1100x20x20; 8 rows 230, 16 rows 213).
static __global__ void __launch_bounds__(64) k_rlines_long(RLines L, double *__restrict__ T, int nlines)
{
    constexpr int U = 16;
    const int n = L.i1, j1 = L.j1, t = blockIdx.x * 64 + threadIdx.x;
    if (t >= nlines) return;
    int s, q, l;
    rline_place(L, t, s, q, l);
    double *x = T + (size_t)s * n * j1 + l;
    const double *p = L.piv + (size_t)q * n * j1 + l, *sub = L.rt, *sup = L.rt + 2 * n;
    const double mu = L.lq[q], lam = L.lz[l];
    const REnd hd = rline_first(L, mu, lam), tl = rline_last(L, mu, lam);
    const double xe = x[(size_t)(n - 1) * j1] - tl.f * x[(size_t)(n - 2) * j1];
    double y = (x[0] - hd.f * x[j1]) * p[0];
    x[0] = y;
    for (int i0 = 1; i0 < n - 1; i0 += U) {
        double xv[U], r[U], a[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = min(i0 + u, n - 2);
            const size_t o = (size_t)i * j1;
            xv[u] = x[o];
            r[u] = p[o];
            a[u] = sub[i];
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (i0 + u < n - 1) {
                y = __builtin_fma(-(a[u] * r[u]), y, xv[u] * r[u]);
                x[(size_t)(i0 + u) * j1] = y;
            }
    }
    y = (xe - tl.b * y) * p[(size_t)(n - 1) * j1];
    x[(size_t)(n - 1) * j1] = y;
    for (int i0 = n - 2; i0 >= 1; i0 -= U) {
        double xv[U], r[U], a[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = max(i0 - u, 1);
            const size_t o = (size_t)i * j1;
            xv[u] = x[o];
            r[u] = p[o];
            a[u] = sup[i];
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (i0 - u >= 1) {
                y = __builtin_fma(-(a[u] * r[u]), y, xv[u]);
                x[(size_t)(i0 - u) * j1] = y;
            }
    }
    x[0] = __builtin_fma(-(hd.b * p[0]), y, x[0]);
}

// The three operators of a run and what memory has room for, in this order:
// a pivot table each; two tables, the second operator's (whose solve runs
// beside the others') and one that the first and the third fill again before
// every solve; one table that every solve fills, with no second set of work
// arrays, so that no two solves run side by side.  Two tables and both sets
// take what two factor arrays and both sets took before pivots were tabulated.
// VV_RTABLES=1, 2 or 3 in the environment at create sets how many.
struct RSolve {
    RLines op[3];
    bool fill[3] = {false, false, false};   // the table is shared: filled before every solve
};

inline void rlines_pivots(const RLines &L, hipStream_t s)
{
    hipLaunchKernelGGL(k_rline_pivots, dim3((unsigned)((L.nq * L.j1 + 63) / 64)), dim3(64), 0, s, L);
}

// The tables, and the second set of work arrays (`words` each) or null.
inline hipError_t rsolve_setup(RSolve &R, double **S2, double **T2, size_t words)
{
    const char *env = std::getenv("VV_RTABLES");
    const int want = env ? std::atoi(env) : 3;
    size_t w[3], most = 0;
    for (int o = 0; o < 3; ++o) {
        w[o] = (size_t)R.op[o].i1 * R.op[o].j1 * R.op[o].nq;
        most = std::max(most, w[o]);
    }
    auto get = [](double **p, size_t n) { return hipMalloc(p, n * sizeof(double)) == hipSuccess; };
    hipError_t e = hipMalloc(&R.op[0].piv, most * sizeof(double));
    if (e != hipSuccess) return e;
    if (want < 2 || !get(S2, words) || !get(T2, words) || !get(&R.op[1].piv, w[1])) {
        for (double **p : {S2, T2, &R.op[1].piv})
            if (*p) { (void)hipFree(*p); *p = nullptr; }
        R.op[1].piv = R.op[2].piv = R.op[0].piv;
        R.fill[0] = R.fill[1] = R.fill[2] = true;
    } else if (want < 3 || !get(&R.op[2].piv, w[2])) {
        R.op[2].piv = R.op[0].piv;
        R.fill[0] = R.fill[2] = true;
    }
    (void)hipGetLastError();   // of the allocations
    for (int o = 0; o < 3; ++o)
        if (!R.fill[o]) rlines_pivots(R.op[o], nullptr);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    return hipStreamSynchronize(nullptr);
}

inline void rsolve_free(RSolve &R)
{
    for (int o = 0; o < 3; ++o)
        if (R.op[o].piv && (o == 0 || R.op[o].piv != R.op[0].piv)) (void)hipFree(R.op[o].piv);
    for (auto &L : R.op) L.piv = nullptr;
}

// T [q][i][l] <- the solutions of operator o (0, 1, 2)
inline void rsolve_launch(const RSolve &R, int o, double *T, hipStream_t s)
{
    const RLines &L = R.op[o];
    if (R.fill[o]) rlines_pivots(L, s);
    // rows of T: the modes, and the second parts of modes 1 .. half - 1
    const int nlines = (L.half ? 2 * L.half : L.nq) * L.j1;
    auto go = [&](auto k, int U) {
        const int nch = (L.i1 + U - 1) / U, tiles = (nlines + RLT - 1) / RLT;
        hipLaunchKernelGGL(k, dim3((unsigned)((tiles + 7) / 8 * 8)), dim3((unsigned)((nch * RLT + 63) / 64 * 64)),
                           2 * sizeof(double2) * nch * RLT, s, L, T, nlines, nch);
    };
    // 8 rows a thread up to 128 rows (100x42x50: 266 us a step; 16: 270), 16
    // above, where they halve the chunks to go through (512x256x256: 8289; 8:
    // 8319) and up to what a workgroup's 1024 threads hold
    if (L.i1 <= 128) go(k_rlines<8>, 8);
    else if (L.i1 <= 1024) go(k_rlines<16>, 16);
    else hipLaunchKernelGGL(k_rlines_long, dim3((unsigned)((nlines + 63) / 64)), dim3(64), 0, s, L, T, nlines);
}

}  // namespace vv
