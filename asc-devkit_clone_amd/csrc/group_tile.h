// group_tile.h -- which tile of a quantized group matmul a workgroup computes (gemm_i8.hip, gemm_pipe_group.hip).
#pragma once

#include "common.h"
#include "launch.h"

namespace ascq {

// a value every lane of the wave holds alike, moved to scalar registers
__device__ __forceinline__ int64_t uniform64(int64_t v)
{
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)((uint64_t)v >> 32));
    return (int64_t)(((uint64_t)hi << 32) | lo);
}

// QuantGroupMatmul: the m axis is split into G ragged groups (group_list), group g multiplies its rows by
// W[g].  The real tiles are ordered group-major, then n-tile, then m-tile within the group, and the order is cut
// into 8 contiguous ranges, one per XCD (workgroup ids go round-robin over the XCDs): an XCD then works on one
// or two experts' column ranges, so its L2 holds the weight columns it streams instead of every XCD fetching
// every expert's weights.  m-tiles never straddle a group.  The grid is sized for ceil(M / BM) + G m-tiles per
// n-tile; ids past the real tile count exit at once.
constexpr int GROUP_MAX = 1024;  // groups the tiled kernels take (the host refuses more)

// exclusive prefix sum over the workgroup of one value per thread (NT threads); *total gets the full sum
template <int NT>
__device__ __forceinline__ int64_t block_exclusive_scan(int64_t v, int64_t* wtot, int64_t* total)
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    int64_t x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int64_t y = __shfl_up(x, o, 64);
        if (lane >= o) x += y;
    }
    if (lane == 63) wtot[w] = x;
    __syncthreads();
    int64_t base = 0, tot = 0;
#pragma unroll
    for (int i = 0; i < NT / 64; ++i) {
        if (i < w) base += wtot[i];
        tot += wtot[i];
    }
    __syncthreads();  // wtot may be reused
    *total = tot;
    return base + x - v;
}

// the tile of this workgroup: its group, first row and column, and the end of the group's rows; false past the last tile
struct GroupTile {
    int g;
    int64_t m0, n0, m_end;
};
template <int NTT, int BM, int BN>
__device__ __forceinline__ bool find_group_tile(const GroupGemmArgs& p, GroupTile& out)
{
    __shared__ int64_t wtot[NTT / 64];
    __shared__ int64_t tile_info[4];  // group, first row, end row, first m-tile of this workgroup's tile
    const int G = (int)p.G;
    const int64_t M = p.M;
    // Group g's rows are [start_g, end_g) clamped to [0, M) (rows outside [0, M) exist in no group) and its
    // m-tiles follow those of groups 0 .. g-1.  Thread t owns groups [t * per, (t + 1) * per): two block-wide
    // prefix sums (rows, then m-tiles) give every thread its groups' starts, and the thread owning this
    // workgroup's tile publishes it -- no G-sized table, so the LDS stays with the stage ring.
    const int per = (G + NTT - 1) / NTT, ga = (int)threadIdx.x * per;
    auto count = [&](int g) {
        const int64_t c = p.list_type == 0 ? p.group_list[g + 1] - p.group_list[g] : p.group_list[g];
        return c < 0 ? (int64_t)0 : c;
    };
    auto clampM = [&](int64_t v) { return v < 0 ? (int64_t)0 : (v > M ? M : v); };
    const int64_t base = p.list_type == 0 ? p.group_list[0] : 0;
    int64_t rows_total, tiles_total, mine = 0;
    for (int k = 0; k < per; ++k)
        if (ga + k < G) mine += count(ga + k);
    const int64_t s0 = base + block_exclusive_scan<NTT>(mine, wtot, &rows_total);
    mine = 0;
    {
        int64_t st = s0;
        for (int k = 0; k < per; ++k)
            if (ga + k < G) {
                const int64_t c = count(ga + k);
                mine += (clampM(st + c) - clampM(st) + BM - 1) / BM;
                st += c;
            }
    }
    const int64_t tiles_n = (p.N + BN - 1) / BN;
    const int64_t t0 = block_exclusive_scan<NTT>(mine, wtot, &tiles_total);
    const int64_t total = tiles_total * tiles_n;  // real (m-tile, n-tile) pairs
    const int64_t per_xcd = (total + 7) / 8;
    const int64_t lin = (int64_t)(blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
    if ((int64_t)(blockIdx.x / 8) >= per_xcd || lin >= total) return false;
    int64_t st = s0, tf = t0;
    for (int k = 0; k < per; ++k)
        if (ga + k < G) {
            const int64_t c = count(ga + k), a0 = clampM(st), a1 = clampM(st + c);
            const int64_t nt = (a1 - a0 + BM - 1) / BM;
            if (nt > 0 && tf * tiles_n <= lin && lin < (tf + nt) * tiles_n) {
                tile_info[0] = ga + k;
                tile_info[1] = a0;
                tile_info[2] = a1;
                tile_info[3] = tf;
            }
            st += c;
            tf += nt;
        }
    __syncthreads();
    // every lane reads the same values; readfirstlane keeps them (and the buffer resources built from them)
    // in scalar registers -- a resource in VGPRs costs a waterfall loop around every access
    const int g = __builtin_amdgcn_readfirstlane((int)tile_info[0]);
    const int64_t g_first = uniform64(tile_info[1]), m_end = uniform64(tile_info[2]);
    const int64_t g_tile0 = uniform64(tile_info[3]);
    const int64_t mt_g = (m_end - g_first + BM - 1) / BM;  // m-tiles of group g (>= 1 here)
    const int64_t rem = lin - g_tile0 * tiles_n;
    const int tn = __builtin_amdgcn_readfirstlane((int)(rem / mt_g));
    const int64_t m0 = uniform64(g_first + (rem % mt_g) * BM);
    out.g = g;
    out.m0 = m0;
    out.n0 = (int64_t)tn * BN;
    out.m_end = m_end;
    return true;
}

}  // namespace ascq
