// onchip.hpp -- helpers of the solves whose vectors stay in a workgroup's registers and LDS.
#pragma once
#include "ycn_device.hpp"
#include "ycn_internal.hpp"

namespace ycn {

// The sum of v over the block in every thread.  red holds two rows of 16 slots, used in
// turn: between two uses of a row every thread passes the barrier of the other.
__device__ __forceinline__ double onchip_sum(double v, double (*red)[16], int &turn) {
    v = wave_sum(v);
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave, nw = blockDim.x / kWave;
    if (lane == 0) red[turn][wave] = v;
    __syncthreads();
    const int k = lane & 15;
    v = row_sum(k < nw ? red[turn][k] : 0.0);
    turn ^= 1;
    return lane_f64(v, 0);   // a scalar: the solve's sums and bounds take no vector registers
}

// the largest v (>= 0) over the block in every thread
__device__ __forceinline__ double onchip_max(double v, double (*red)[16], int &turn) {
    v = wave_max(v);
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave, nw = blockDim.x / kWave;
    if (lane == 0) red[turn][wave] = v;
    __syncthreads();
    const int k = lane & 15;
    v = wave_max(k < nw ? red[turn][k] : 0.0);
    turn ^= 1;
    return lane_f64(v, 0);
}

// u as a value the compiler knows nothing about: addresses unpacked from it are formed where
// they are used (a few instructions) instead of ahead of the iteration loop, where a site's
// dozen addresses would be spilled to memory and read back in every iteration
__device__ __forceinline__ unsigned fresh(unsigned u) {
    asm volatile("" : "+v"(u));
    return u;
}

}  // namespace ycn
