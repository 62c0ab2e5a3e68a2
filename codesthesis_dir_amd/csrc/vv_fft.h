// vv_fft.h -- FFT stages in LDS over periodic lines, shared by the 2D and 3D
// solvers (device code; included by the .hip files only).
//
// A workgroup holds LP pairs of real lines; each pair is one complex line of
// n points (n a power of two, loaded in bit-reversed order; other even n
// through the mixed-radix stages below).  Stage s (radix 2) pairs
// positions p and p + h (h = 2^s) with the twiddle e^{-i 2 pi (p mod h)/(2h)},
// taken from tw[t] = (cos, -sin)(2 pi t/n), t < n/2 (conjugated for the
// inverse).  Z_m and Z_{n-m} separate the pair's two real spectra.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <vector>

namespace vv {

__device__ __forceinline__ unsigned bitrev(unsigned x, int bits) { return __builtin_bitreverse32(x) >> (32 - bits); }

template <bool INV>
__device__ __forceinline__ void fft_bfly(double2 &u, double2 &v, double2 w)
{
    if (INV) w.y = -w.y;
    const double2 vw = make_double2(v.x * w.x - v.y * w.y, v.x * w.y + v.y * w.x);
    const double2 a = u;
    u = make_double2(a.x + vw.x, a.y + vw.y);
    v = make_double2(a.x - vw.x, a.y - vw.y);
}

// The radix-2 stages, three per pass through LDS: the 8 points a + m h
// (m < 8, h = 2^s, a = (group) 8h + pos, pos < h) pair only among themselves
// in stages s, s+1 and s+2, so one thread loads them, applies the three
// stages' butterflies in registers -- each the radix-2 butterfly of that
// stage with its twiddle, so the same operations and the same bits -- and
// stores them; one or two stages left over take a pass of their own.
template <bool INV>
__device__ void fft_stages(double2 *z, const double2 *tw, int np, int bits, int LP)
{
    int s = 0;
    for (; s + 3 <= bits; s += 3) {
        const int h = 1 << s;
        const int nb = LP * (np >> 3);
        for (int b = threadIdx.x; b < nb; b += blockDim.x) {
            const int pr = b >> (bits - 3), t = b & ((np >> 3) - 1);
            const int pos = t & (h - 1), grp = t >> s;
            double2 *za = z + pr * np + grp * 8 * h + pos;
            double2 x[8];
#pragma unroll
            for (int m = 0; m < 8; ++m) x[m] = za[m * h];
            const double2 w0 = tw[pos << (bits - 1 - s)];   // stage s: pairs (m, m+1), m even
            fft_bfly<INV>(x[0], x[1], w0);
            fft_bfly<INV>(x[2], x[3], w0);
            fft_bfly<INV>(x[4], x[5], w0);
            fft_bfly<INV>(x[6], x[7], w0);
            // stage s+1: pairs (m, m+2), m = 0, 1, 4, 5, at positions pos + (m mod 4) h
            const double2 w1a = tw[pos << (bits - 2 - s)], w1b = tw[(pos + h) << (bits - 2 - s)];
            fft_bfly<INV>(x[0], x[2], w1a);
            fft_bfly<INV>(x[1], x[3], w1b);
            fft_bfly<INV>(x[4], x[6], w1a);
            fft_bfly<INV>(x[5], x[7], w1b);
            // stage s+2: pairs (m, m+4), m < 4, at positions pos + m h
#pragma unroll
            for (int m = 0; m < 4; ++m) fft_bfly<INV>(x[m], x[m + 4], tw[(pos + m * h) << (bits - 3 - s)]);
#pragma unroll
            for (int m = 0; m < 8; ++m) za[m * h] = x[m];
        }
        __syncthreads();
    }
    if (bits - s == 2) {   // stages s, s+1 (the last two)
        const int h = 1 << s;
        const int nb = LP * (np >> 2);
        for (int b = threadIdx.x; b < nb; b += blockDim.x) {
            const int pr = b >> (bits - 2), t = b & ((np >> 2) - 1);
            const int pos = t & (h - 1), grp = t >> s;
            double2 *za = z + pr * np + grp * 4 * h + pos;
            double2 x0 = za[0], x1 = za[h], x2 = za[2 * h], x3 = za[3 * h];
            const double2 w0 = tw[pos << (bits - 1 - s)];
            fft_bfly<INV>(x0, x1, w0);
            fft_bfly<INV>(x2, x3, w0);
            fft_bfly<INV>(x0, x2, tw[pos << (bits - 2 - s)]);
            fft_bfly<INV>(x1, x3, tw[(pos + h) << (bits - 2 - s)]);
            za[0] = x0; za[h] = x1; za[2 * h] = x2; za[3 * h] = x3;
        }
        __syncthreads();
    } else if (bits - s == 1) {   // the last stage
        const int h = 1 << s;
        const int nb = LP * (np >> 1);
        for (int b = threadIdx.x; b < nb; b += blockDim.x) {
            const int pr = b >> (bits - 1), t = b & ((np >> 1) - 1);
            const int pos = t & (h - 1), grp = t >> s;
            double2 *za = z + pr * np + grp * 2 * h + pos;
            double2 x0 = za[0], x1 = za[h];
            fft_bfly<INV>(x0, x1, tw[pos << (bits - 1 - s)]);
            za[0] = x0; za[h] = x1;
        }
        __syncthreads();
    }
}

// Mixed radix, n = 2^bits p_1 ... p_m points, the p odd primes: the radix-2
// stages transform the n / 2^bits sub-lines of n1 = 2^bits points, then each
// odd prime joins p neighbouring sub-lines A_j of L points into one of pL,
//   X_k = sum_{j<p} W_{pL}^{jk} A_j[k mod L],  W_n^t = twc[t] = (cos, -sin)(2 pi t/n)
// (conjugated twiddles give the inverse).  The p outputs k0 + L q, q < p,
// depend on the p inputs A_j[k0] only and take their places, so for p <= 13
// one thread does them in registers in place (mr_stage): O(n p) per stage and
// one pass through LDS, where one combination over the whole odd factor b
// was O(n b) (at n = 150 = 2 3 5 5: 13 products a point against 75).  Larger
// primes form their outputs R per thread, with a barrier before the stores
// (mr_stage_any).  Point k of a line is loaded at pos[k], the mixed-radix
// digit reversal.
constexpr int MR_MAXST = 9;   // odd prime factors of an even n <= 65535: 2 3^9 at most
struct MrPlan {
    int n, bits, nst;
    int p[MR_MAXST];
    const double2 *tw, *twc;       // radix-2 twiddles of n1 points (n1/2), of n points (n)
    const unsigned short *pos;
};

template <int P> struct OddRoots;  // cos, sin of 2 pi m/P
template <> struct OddRoots<3> {
    static constexpr double c[3] = {1.0, -0.5, -0.5};
    static constexpr double s[3] = {0.0, 0.8660254037844386, -0.8660254037844386};
};
template <> struct OddRoots<5> {
    static constexpr double c[5] = {1.0, 0.30901699437494745, -0.8090169943749475, -0.8090169943749475, 0.30901699437494745};
    static constexpr double s[5] = {0.0, 0.9510565162951535, 0.5877852522924731, -0.5877852522924731, -0.9510565162951535};
};
template <> struct OddRoots<7> {
    static constexpr double c[7] = {1.0, 0.6234898018587335, -0.2225209339563144, -0.9009688679024191, -0.9009688679024191, -0.2225209339563144, 0.6234898018587335};
    static constexpr double s[7] = {0.0, 0.7818314824680298, 0.9749279121818236, 0.4338837391175581, -0.4338837391175581, -0.9749279121818236, -0.7818314824680298};
};
template <> struct OddRoots<11> {
    static constexpr double c[11] = {1.0, 0.8412535328311812, 0.41541501300188644, -0.14231483827328514, -0.6548607339452851, -0.9594929736144974, -0.9594929736144974, -0.6548607339452851, -0.14231483827328514, 0.41541501300188644, 0.8412535328311812};
    static constexpr double s[11] = {0.0, 0.5406408174555976, 0.9096319953545183, 0.9898214418809327, 0.7557495743542583, 0.28173255684142967, -0.28173255684142967, -0.7557495743542583, -0.9898214418809327, -0.9096319953545183, -0.5406408174555976};
};
template <> struct OddRoots<13> {
    static constexpr double c[13] = {1.0, 0.8854560256532099, 0.5680647467311558, 0.12053668025532305, -0.3546048870425356, -0.7485107481711011, -0.970941817426052, -0.970941817426052, -0.7485107481711011, -0.3546048870425356, 0.12053668025532305, 0.5680647467311558, 0.8854560256532099};
    static constexpr double s[13] = {0.0, 0.46472317204376856, 0.8229838658936564, 0.992708874098054, 0.9350162426854148, 0.6631226582407952, 0.23931566428755777, -0.23931566428755777, -0.6631226582407952, -0.9350162426854148, -0.992708874098054, -0.8229838658936564, -0.46472317204376856};
};

template <bool INV, int P>
__device__ __forceinline__ void mr_stage(double2 *z, const double2 *twc, int n, int L, int LP)
{
    constexpr int H = (P - 1) / 2;
    using T = OddRoots<P>;
    const int M = P * L, nb = LP * (n / P), str = n / M;
    for (int b = threadIdx.x; b < nb; b += blockDim.x) {
        const int g = b / L, k0 = b - g * L;
        double2 *za = z + g * M + k0;
        double2 x[P];
        x[0] = za[0];
#pragma unroll
        for (int j = 1; j < P; ++j) {
            double2 w = twc[str * j * k0];
            if (INV) w.y = -w.y;
            const double2 v = za[j * L];
            x[j] = make_double2(v.x * w.x - v.y * w.y, v.x * w.y + v.y * w.x);
        }
        double2 s[H + 1], d[H + 1], t = x[0];
#pragma unroll
        for (int j = 1; j <= H; ++j) {
            s[j] = make_double2(x[j].x + x[P - j].x, x[j].y + x[P - j].y);
            d[j] = make_double2(x[j].x - x[P - j].x, x[j].y - x[P - j].y);
            t.x += s[j].x;
            t.y += s[j].y;
        }
        za[0] = t;
#pragma unroll
        for (int q = 1; q <= H; ++q) {   // X_q = E - i O, X_{P-q} = E + i O (the inverse: exchanged)
            double2 e = x[0], o = make_double2(0.0, 0.0);
#pragma unroll
            for (int j = 1; j <= H; ++j) {
                const double c = T::c[j * q % P], sn = T::s[j * q % P];
                e.x = __builtin_fma(c, s[j].x, e.x);
                e.y = __builtin_fma(c, s[j].y, e.y);
                o.x = __builtin_fma(sn, d[j].x, o.x);
                o.y = __builtin_fma(sn, d[j].y, o.y);
            }
            const double2 a = make_double2(e.x + o.y, e.y - o.x), c2 = make_double2(e.x - o.y, e.y + o.x);
            za[q * L] = INV ? c2 : a;
            za[(P - q) * L] = INV ? a : c2;
        }
    }
    __syncthreads();
}

// any odd p, R outputs per thread: LP n <= R blockDim.x (checked by the host)
template <bool INV, int R>
__device__ void mr_stage_any(double2 *z, const double2 *twc, int n, int L, int p, int LP)
{
    double2 acc[R];
    const int total = LP * n, M = p * L, str = n / M;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int e = (int)threadIdx.x + r * (int)blockDim.x;
        double re = 0.0, im = 0.0;
        if (e < total) {
            const int g = e / M, k = e - g * M;
            const double2 *zl = z + g * M + k % L;
            int t = 0;
            for (int j = 0; j < p; ++j) {
                double2 w = twc[t * str];
                if (INV) w.y = -w.y;
                const double2 v = zl[j * L];
                re += v.x * w.x - v.y * w.y;
                im += v.x * w.y + v.y * w.x;
                t += k;
                if (t >= M) t -= M;
            }
        }
        acc[r] = make_double2(re, im);
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int e = (int)threadIdx.x + r * (int)blockDim.x;
        if (e < total) z[e] = acc[r];
    }
    __syncthreads();
}

// position of point k: bit reversal (R = 0: a power of two) or the plan's
template <int R>
__device__ __forceinline__ int mr_pos(const MrPlan &F, int k)
{
    return R ? (int)F.pos[k] : (int)bitrev((unsigned)k, F.bits);
}

// The transform of LP lines in LDS.  R = 0: a power of two; 1: odd primes up
// to 13; more: any, R outputs per thread for the larger ones.  tw, twc: the
// plan's twiddles or their copies in LDS.
template <bool INV, int R>
__device__ __forceinline__ void mr_transform(double2 *z, const MrPlan &F, const double2 *tw, const double2 *twc, int LP)
{
    int L = 1 << F.bits;
    fft_stages<INV>(z, tw, L, F.bits, LP * (R ? F.n >> F.bits : 1));
    if constexpr (R > 0) {
        for (int t = 0; t < F.nst; ++t) {
            const int p = F.p[t];
            switch (p) {
            case 3: mr_stage<INV, 3>(z, twc, F.n, L, LP); break;
            case 5: mr_stage<INV, 5>(z, twc, F.n, L, LP); break;
            case 7: mr_stage<INV, 7>(z, twc, F.n, L, LP); break;
            case 11: mr_stage<INV, 11>(z, twc, F.n, L, LP); break;
            case 13: mr_stage<INV, 13>(z, twc, F.n, L, LP); break;
            default:
                if constexpr (R > 1) mr_stage_any<INV, R>(z, twc, F.n, L, p, LP);
            }
            L *= p;
        }
    }
}

// Host side: the plan of even n <= 65535 without its device pointers, the
// twiddles (n1/2, then n when n is no power of two) and the positions.
struct MrTables {
    MrPlan plan{};
    bool small = true;             // no prime above 13
    std::vector<double2> tw;
    std::vector<unsigned short> pos;
    size_t bytes() const { return tw.size() * sizeof(double2) + pos.size() * sizeof(unsigned short); }
    // the plan with its pointers into a device copy of tw and, behind it, pos
    MrPlan at(void *dev) const
    {
        MrPlan F = plan;
        F.tw = static_cast<const double2 *>(dev);
        F.twc = F.tw + ((size_t)1 << plan.bits) / 2;
        F.pos = reinterpret_cast<const unsigned short *>(F.tw + tw.size());
        return F;
    }
};
inline MrTables mr_tables(int n)
{
    MrTables T;
    MrPlan &F = T.plan;
    F.n = n;
    F.bits = __builtin_ctz((unsigned)n);
    const int n1 = 1 << F.bits;
    for (int b = n >> F.bits, p = 3; b > 1; p += 2)
        for (; b % p == 0; b /= p) {
            F.p[F.nst++] = p;
            if (p > 13) T.small = false;
        }
    const double pi = std::acos(-1.0);
    auto root = [&](int t, int m) { return make_double2(std::cos(2.0 * pi * t / m), -std::sin(2.0 * pi * t / m)); };
    for (int t = 0; t < n1 / 2; ++t) T.tw.push_back(root(t, n1));
    if (n1 == n) return T;
    for (int t = 0; t < n; ++t) T.tw.push_back(root(t, n));
    T.pos.resize(n);
    for (int k = 0; k < n; ++k) {
        int r = k, len = n, at = 0;
        for (int t = F.nst - 1; t >= 0; --t) {
            len /= F.p[t];
            at += r % F.p[t] * len;
            r /= F.p[t];
        }
        int rev = 0;
        for (int q = 0; q < F.bits; ++q) rev |= ((r >> q) & 1) << (F.bits - 1 - q);
        T.pos[k] = (unsigned short)(at + rev);
    }
    return T;
}
inline hipError_t mr_upload(const MrTables &T, void *dev)
{
    hipError_t e = hipMemcpy(dev, T.tw.data(), T.tw.size() * sizeof(double2), hipMemcpyHostToDevice);
    if (e == hipSuccess && !T.pos.empty())
        e = hipMemcpy(static_cast<char *>(dev) + T.tw.size() * sizeof(double2), T.pos.data(),
                      T.pos.size() * sizeof(unsigned short), hipMemcpyHostToDevice);
    return e;
}
// template argument R for LP lines of the plan and 256 threads
inline int mr_r(const MrTables &T, int LP)
{
    return T.plan.nst == 0 ? 0 : T.small ? 1 : (LP * T.plan.n <= 8 * 256) ? 8 : 32;
}
inline int pow2_floor(int v)
{
    int q = 1;
    while (2 * q <= v) q *= 2;
    return q;
}

// pairs of lines per workgroup: LP np complex values within 32 KB (64 KB for
// the longest lines)
inline int fft_pairs(int np) { return np >= 4096 ? 1 : std::max(1, 2048 / np); }

}  // namespace vv
