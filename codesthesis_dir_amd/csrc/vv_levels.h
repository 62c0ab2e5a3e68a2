// The time levels of the 3D solvers with side walls or a barrier in y or phi
// (fields of (nr+2) x (nz+2) x (np+2) points): Ap <- A <- An by exchanging
// the three buffers of A, B, C and th.  The old Ap buffer becomes the new An,
// whose values the reference's copies leave equal to A.
#pragma once
#include <hip/hip_runtime.h>

#include <utility>

namespace vv {

struct Levels {
    const double *src[4];
    double *dst[4];
};

static __global__ void __launch_bounds__(256) k_levels_all(Levels C, size_t n)
{
    const size_t t = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (t < n) C.dst[blockIdx.y][t] = C.src[blockIdx.y][t];
}

// The points outside i = 1..nr-1, j = 1..nz-1, k = 1..np-1: three whole
// planes, then the rim of the others.
__host__ __device__ inline unsigned levels_rim(int nr, int nz) { return 3u * (nz + 2) + 3u * (nr - 1); }

static __global__ void __launch_bounds__(256) k_levels_shell(Levels C, int nr, int nz, int np)
{
    const unsigned ldi = nr + 2, pl = ldi * (nz + 2), rim = levels_rim(nr, nz);
    unsigned t = blockIdx.x * 256 + threadIdx.x, o;
    if (t < 3 * pl) {
        o = t < pl ? t : (unsigned)(np - 1) * pl + t;   // planes 0, np, np + 1
    } else {
        t -= 3 * pl;
        const unsigned k = t / rim, e = t - k * rim;
        if (k >= (unsigned)(np - 1)) return;
        unsigned i, j;
        if (e < 3u * (nz + 2)) {
            j = e / 3;
            i = e - 3 * j;
            if (i) i += nr - 1;
        } else {
            const unsigned f = e - 3u * (nz + 2);
            j = f / (nr - 1);
            i = 1 + f - j * (nr - 1);
            if (j) j += nz - 1;
        }
        o = (k + 1) * pl + j * ldi + i;
    }
    C.dst[blockIdx.y][o] = C.src[blockIdx.y][o];
}

// f: the fields by index, lev: (p, current, n) of each quantity.  again: the
// next explicit step follows before anything else reads the n level.  It
// writes that level on i = 1..nr-1, j = 1..nz-1, k = 1..np-1 (each routine's
// range holds this box), so only the points around the box are copied: at
// 512x256x256 the whole copy took 380 us of an 8.18 ms step.
inline void levels_rotate(double **f, const int (&lev)[4][3], bool again, int nr, int nz, int np, hipStream_t s)
{
    Levels C;
    for (int q = 0; q < 4; ++q) {
        double *&p = f[lev[q][0]], *&c = f[lev[q][1]], *&n = f[lev[q][2]];
        std::swap(p, c);
        std::swap(c, n);
        C.src[q] = c;
        C.dst[q] = n;
    }
    const size_t pl = (size_t)(nr + 2) * (nz + 2), nf = pl * (np + 2);
    const size_t cnt = again ? 3 * pl + (size_t)(np - 1) * levels_rim(nr, nz) : nf;
    const dim3 grid((unsigned)((cnt + 255) / 256), 4);
    if (again) hipLaunchKernelGGL(k_levels_shell, grid, dim3(256), 0, s, C, nr, nz, np);
    else hipLaunchKernelGGL(k_levels_all, grid, dim3(256), 0, s, C, nf);
}

}  // namespace vv
