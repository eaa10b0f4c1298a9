// Reference-format left-right cross check for gfx950.
//
// Restates CrossCheckDisparityMaps::Kernel::Transform (CrossCheckDisparityMaps.cu:62-109)
// per pixel on 4 x uint16 disparity-id maps: codes outside [First, Last] pass through,
// the right position is MapPixelPos(x, id - First, LtoR), positions outside the image
// and |id_R - id_L| > thresh become Inconsistent.  The reference accumulates the range of
// kept ids with two global atomics per pixel into a 128 x 2 buffer that the host then
// reduces (:86-94, :181-190).  Here a workgroup folds the ids it keeps into one minimum
// and one maximum before it touches the shared range, and the last workgroup to finish
// hands the range over and resets it for the next frame, in the same launch.
#include "common.hpp"
#include "kernels.hpp"

namespace stereo {
namespace {

constexpr uint32_t ID_FIRST = 1, ID_LAST = 0xFFF0 - 1, ID_INCONSISTENT = 0xFFFF - 5;

__device__ __forceinline__ uint32_t wave_min(uint32_t v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const uint32_t t = (uint32_t)__shfl_xor((int)v, o, 64);
        v = t < v ? t : v;
    }
    return v;
}

__device__ __forceinline__ uint32_t wave_max(uint32_t v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const uint32_t t = (uint32_t)__shfl_xor((int)v, o, 64);
        v = t > v ? t : v;
    }
    return v;
}

// What bounds it: 24 bytes per pixel of HBM traffic, two dependent loads deep (the right id
// is gathered at the left id's position), and the shared range: every workgroup of the launch
// meets on its words, at about 2.8 ns each.  With one atomic pair per wave the range took the
// whole kernel (1280x720: 323.8 us of 115 k atomics, and 4.6 us for a launch that reset it);
// a grid of at most XC_GRID workgroups of 16 waves, each taking segments of 256 pixels of a
// row with a thread's XC_U pixels loaded together, leaves three atomics per workgroup
// (the NCC / NCC / check / de-noise / colour sequence at 1280x720: 1204 -> 884 us a pass).
constexpr int XC_THREADS = 1024, XC_WAVES = XC_THREADS / 64, XC_U = 4, XC_SEG = 64 * XC_U;
constexpr int XC_GRID = 256;

// state: [0] minimum, [1] maximum of the kept ids, at their empty values between launches,
// [2] workgroups that have finished, back at 0 between launches.  result: the caller's copy
// of the range, host memory the device writes.
__global__ __launch_bounds__(XC_THREADS) void crosscheck_ref_kernel(View out, View lr, View rl, int thresh, int ltor,
                                                                    int offset, uint32_t* state, uint32_t* result)
{
    __shared__ uint32_t smin[XC_WAVES], smax[XC_WAVES];
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nsx = (lr.w + XC_SEG - 1) / XC_SEG, nseg = nsx * lr.h;
    uint32_t kmin = ID_LAST, kmax = ID_FIRST;
    for (int sg = blockIdx.x * XC_WAVES + wv; sg < nseg; sg += gridDim.x * XC_WAVES) {
        const int y = sg / nsx, x0 = (sg - y * nsx) * XC_SEG + lane;
        const ushort4* const lrow = row_ptr<const ushort4>(lr, y);
        const ushort4* const rrow = row_ptr<const ushort4>(rl, y);
        ushort4 pl[XC_U];
        int idr[XC_U];
#pragma unroll
        for (int u = 0; u < XC_U; ++u) pl[u] = lrow[min(x0 + 64 * u, lr.w - 1)];
#pragma unroll
        for (int u = 0; u < XC_U; ++u) {
            const int d = (int)pl[u].x - (int)ID_FIRST, x = x0 + 64 * u;
            const int xr = ltor ? x - d - offset : x + d + offset;
            // -1: the position lies outside the image
            idr[u] = (xr >= 0 && xr < rl.w) ? (int)rrow[xr].x : -1;
        }
#pragma unroll
        for (int u = 0; u < XC_U; ++u) {
            const int x = x0 + 64 * u;
            if (x >= lr.w) continue;
            const uint32_t id = pl[u].x;
            if (id >= ID_FIRST && id <= ID_LAST) {
                if (idr[u] >= 0 && abs(idr[u] - (int)id) <= thresh) {
                    kmin = min(kmin, id);
                    kmax = max(kmax, id);
                } else {
                    pl[u].x = (uint16_t)ID_INCONSISTENT;
                }
            }
            row_ptr<ushort4>(out, y)[x] = pl[u];
        }
    }
    kmin = wave_min(kmin);
    kmax = wave_max(kmax);
    if (lane == 0) {
        smin[wv] = kmin;
        smax[wv] = kmax;
    }
    __syncthreads();
    if (threadIdx.x != 0) return;
    for (int k = 1; k < XC_WAVES; ++k) {
        kmin = min(kmin, smin[k]);
        kmax = max(kmax, smax[k]);
    }
    if (kmin != ID_LAST) atomicMin(&state[0], kmin);
    if (kmax != ID_FIRST) atomicMax(&state[1], kmax);
    __threadfence();  // the range before the count
    // atomicInc wraps at the grid's size: the count is back at 0 when the last one has added
    if (atomicInc(&state[2], gridDim.x - 1) != gridDim.x - 1) return;
    __threadfence();
    result[0] = atomicExch(&state[0], ID_LAST);
    result[1] = atomicExch(&state[1], ID_FIRST);
}

}  // namespace

hipError_t crosscheck_state_init(uint32_t* state)
{
    const uint32_t empty[3] = {ID_LAST, ID_FIRST, 0};
    return hipMemcpy(state, empty, sizeof(empty), hipMemcpyHostToDevice);
}

hipError_t launch_crosscheck_ref(const View& out, const View& lr, const View& rl, int thresh, int ltor, int offset,
                                 uint32_t* state, uint32_t* result, hipStream_t s)
{
    const long nseg = (long)((lr.w + XC_SEG - 1) / XC_SEG) * lr.h;
    const long need = (nseg + XC_WAVES - 1) / XC_WAVES;
    if (nseg > 0x7fffffffL - (long)XC_GRID * XC_WAVES) return hipErrorInvalidValue;
    hipLaunchKernelGGL(crosscheck_ref_kernel, dim3((unsigned)(need < XC_GRID ? need : XC_GRID)), dim3(XC_THREADS), 0, s, out,
                       lr, rl, thresh, ltor, offset, state, result);
    return hipGetLastError();
}

}  // namespace stereo
