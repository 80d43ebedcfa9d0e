// scan.hpp - offsets of tiles in an ordered stream compaction.
#pragma once

#include <hip/hip_runtime.h>

namespace lumx {

// Up to this many tiles the kernel that scatters adds up the counts before its
// own tile (one load a thread and a reduction, beside its other loads); above
// it, where those sums grow with the square of the tiles, a launch of one
// workgroup turns the counts into offsets first.  At 18 tiles the sums save
// that launch, 4 us; at 2048 they read 8 MB in all, under 3 us.
constexpr int kSumTiles = 2048;

// Sum of counts[0 .. n), for a workgroup of full waves (at most 1024 threads).
__device__ __forceinline__ int sum_before(const int* counts, int n) {
    __shared__ int s_part[16];
    int v = 0;
    for (int i = threadIdx.x; i < n; i += blockDim.x) v += counts[i];
    for (int d = 32; d > 0; d >>= 1) v += __shfl_xor(v, d);
    if ((threadIdx.x & 63) == 0) s_part[threadIdx.x >> 6] = v;
    __syncthreads();
    int sum = 0;
    for (int i = 0; i < (int)(blockDim.x >> 6); ++i) sum += s_part[i];
    return sum;
}

// Bits set before each of n <= 64 words, by one wave.
__device__ __forceinline__ void word_prefix(const unsigned long long* words, int n, int* prefix) {
    const int lane = threadIdx.x & 63;
    const int v = lane < n ? __popcll(words[lane]) : 0;
    int x = v;
    for (int d = 1; d < 64; d <<= 1) {
        const int y = __shfl_up(x, d);
        if (lane >= d) x += y;
    }
    if (lane < n) prefix[lane] = x - v;
}

}  // namespace lumx
