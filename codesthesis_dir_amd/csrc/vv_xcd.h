#pragma once
#include <hip/hip_runtime.h>

namespace vv {

// Workgroups are dispatched to the 8 XCDs (each with its own L2) in turn:
// xcd_block maps the dispatch index b of nb workgroups to a logical index so
// that each XCD works through one contiguous range, and neighbouring rows
// and planes of a field are read through the same L2.
__device__ __forceinline__ unsigned xcd_block(unsigned b, unsigned nb)
{
    const unsigned x = b & 7u, q = b >> 3, per = nb >> 3, rem = nb & 7u;
    return x * per + (x < rem ? x : rem) + q;
}

// the same over a grid of rows of workgroups: this one's column and row
__device__ __forceinline__ void xcd_tile(int &bx, int &by)
{
    const unsigned w = xcd_block(blockIdx.y * gridDim.x + blockIdx.x, gridDim.x * gridDim.y);
    by = (int)(w / gridDim.x);
    bx = (int)(w - (unsigned)by * gridDim.x);
}

// the same for n workgroups of a grid whose rows are padded to a multiple of
// 8, in each row by itself; -1 for the padding
__device__ __forceinline__ int xcd_padded(int n)
{
    const int per = (n + 7) >> 3, q = (int)(blockIdx.x >> 3), w = (int)(blockIdx.x & 7) * per + q;
    return q < per && w < n ? w : -1;
}

// Planes a workgroup of a march takes, of `planes` behind each of `nb` column
// blocks, `slots` workgroups being resident at once.  Eight rounds and more
// keep 16, which bounds how far the neighbouring columns of a plane drift
// apart in the L2 (the 512x256x256 tank's step: 7.87 ms, 8 planes 7.89, 32
// 7.93, 57 7.95).  A march of fewer rounds lasts its rounds times the planes
// of one and a plane's worth of its start: no nearly empty last round
// (129x129x257: 33 planes 701 us a step, 8 planes 727, 16 planes 760) and, on
// small grids, no idle CUs (the tank at 100x42x50: 2 planes 200 us, 16 planes
// 257).
inline int march_planes(long long nb, int planes, long long slots)
{
    if (nb * ((planes + 15) / 16) >= 8 * slots) return 16;
    int best = 1;
    long long least = -1;
    for (int kc = 1; kc <= planes && kc <= 64; ++kc) {
        const long long wgs = nb * ((planes + kc - 1) / kc), cost = ((wgs + slots - 1) / slots) * (kc + 1);
        if (least < 0 || cost <= least) {
            least = cost;
            best = kc;
        }
    }
    return best;
}

// workgroups of `threads` of kernel k resident on the device at once
template <typename K>
inline long long march_slots(K k, int threads, int device)
{
    int per = 0, cus = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, k, threads, 0) != hipSuccess || per < 1) per = 1;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess || cus < 1) cus = 1;
    (void)hipGetLastError();
    return (long long)per * cus;
}

}  // namespace vv
