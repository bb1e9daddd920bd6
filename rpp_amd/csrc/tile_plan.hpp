// tile_plan.hpp -- a ragged batch's tiles planned inside the workgroup that runs them: the exclusive
// prefix of the clips' tile counts in LDS, and the clip that owns a tile.
#pragma once

#include "common.hpp"

namespace rppa {

constexpr int kPlanClips = 2048;   // clips a plan holds (8 KB of LDS)

// start[0 .. B] = exclusive prefix of count(b) over the clips and the total.  Called by the whole
// workgroup (THREADS threads); `red` holds THREADS / 64 ints of LDS.
template <int THREADS, typename Count>
__device__ __forceinline__ void plan_clips(int *start, int B, int *red, const Count &count)
{
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    for (int b = tid; b < B; b += THREADS) start[b] = count(b);   // the length loads are all in flight together
    __syncthreads();
    const int per = (B + THREADS - 1) / THREADS, b0 = min(tid * per, B), b1 = min(b0 + per, B);
    int sum = 0;
    for (int b = b0; b < b1; b++) sum += start[b];
    int s = sum;
    for (int o = 1; o < kWave; o <<= 1) {
        const int u = __shfl_up(s, o);
        if (lane >= o) s += u;
    }
    if (lane == kWave - 1) red[wave] = s;
    __syncthreads();
    int at = s - sum;
    for (int w = 0; w < wave; w++) at += red[w];
    for (int b = b0; b < b1; b++) {
        const int n = start[b];
        start[b] = at;
        at += n;
    }
    if (tid == THREADS - 1) start[B] = at;
    __syncthreads();
}

// The clip whose tiles hold `tile` (start[b] <= tile < start[b + 1]); the whole wave asks for one tile.
// Two rounds of 64 probes, B <= 4096.
__device__ __forceinline__ int plan_owner(const int *start, int B, int tile)
{
    const int lane = threadIdx.x & 63, step = (B + 63) >> 6;
    const int p = lane * step;
    const int lo = (__popcll(__ballot(p < B && start[min(p, B)] <= tile)) - 1) * step;
    const int q = lo + lane;
    return lo + __popcll(__ballot(lane < step && q < B && start[min(q, B)] <= tile)) - 1;
}

// Tile of workgroup `block` of `grid` (a multiple of 8) in round i: the tiles of a round go to the eight
// XCDs (block mod 8) in contiguous runs, so tiles that run at the same time on one XCD are neighbours
// and share their halo and their output lines in its L2.
__host__ __device__ inline unsigned plan_tile(unsigned i, unsigned block, unsigned grid)
{
    return i * grid + (block & 7) * (grid >> 3) + (block >> 3);
}

// The grid of such a launch: at most `resident` workgroups, no more than there are tiles, and a multiple of 8
// whatever the CU count (with any other grid some tiles have no workgroup).
inline unsigned plan_grid(size_t resident, size_t tiles)
{
    const size_t most = resident / 8 * 8, need = (tiles + 7) / 8 * 8;
    const size_t grid = most < need ? most : need;
    return static_cast<unsigned>(grid > 8 ? grid : 8);
}

}  // namespace rppa
