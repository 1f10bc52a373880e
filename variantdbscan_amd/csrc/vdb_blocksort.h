// Stable ranking of a block's items by one digit of their keys (wave64).
#pragma once

#include "vdb_common.h"

namespace vdb {

constexpr int kSortItems = 8; // items a thread holds in a tile of the device-wide sort

// Items sit striped inside a wave: item i < per of a lane is element
// wave * 64 * per + i * 64 + lane of the block (per <= ITEMS rounds a wave).
__device__ __forceinline__ uint32_t block_rank_item(int i, int per)
{
    return (threadIdx.x / kWave) * (uint32_t)(kWave * per) + (uint32_t)(i * kWave) +
           (uint32_t)lane_id();
}

template <int BITS, int WAVES> struct BlockRank {
    uint32_t cnt[WAVES][1 << BITS]; // a wave's items per digit, then those of waves before it
    uint32_t start[1 << BITS];      // first place of a digit in the block
    uint32_t wsum[WAVES];
};

// pos[i] = place of item i < per in the block's stable order by digit (key >>
// shift) & (2^BITS - 1), in the low half of its word (the high half is kept).
// Ends with a barrier; sm.start stays valid after it. A wave
// counts its own rounds of 64 items in LDS without barriers: the lanes of one
// digit (BITS ballots) take consecutive ranks, the first of them adds them.
template <int ITEMS, int BITS, int WAVES>
__device__ __forceinline__ void block_rank(const uint32_t (&key)[ITEMS], int per, int shift,
                                           uint32_t (&pos)[ITEMS], BlockRank<BITS, WAVES> &sm)
{
    constexpr int D = 1 << BITS, T = WAVES * kWave;
    const int w = threadIdx.x / kWave;
    for (int d = lane_id(); d < D; d += kWave) sm.cnt[w][d] = 0;
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int i = 0; i < ITEMS; i++) {
        if (i >= per) continue;
        const uint32_t d = (key[i] >> shift) & (D - 1);
        uint64_t peers = ~0ull;
#pragma unroll
        for (int b = 0; b < BITS; b++) {
            bool bit = (d >> b) & 1u;
            uint64_t bal = ballot(bit);
            peers &= bit ? bal : ~bal;
        }
        const uint32_t r = (uint32_t)mask_rank(peers), before = sm.cnt[w][d];
        __builtin_amdgcn_wave_barrier(); // all lanes have read before the first adds
        if (r == 0) sm.cnt[w][d] = before + (uint32_t)popc64(peers);
        __builtin_amdgcn_wave_barrier();
        pos[i] = (pos[i] & 0xffff0000u) | (before + r);
    }
    __syncthreads();
    // waves before each wave, digit by digit, and the digits' starts
    uint32_t carry = 0;
    for (int d0 = 0; d0 < D; d0 += T) {
        const int d = d0 + (int)threadIdx.x;
        uint32_t tot = 0;
        if (d < D) {
#pragma unroll
            for (int q = 0; q < WAVES; q++) {
                uint32_t t = sm.cnt[q][d];
                sm.cnt[q][d] = tot;
                tot += t;
            }
        }
        uint32_t incl = tot;
        for (int o = 1; o < kWave; o <<= 1) {
            uint32_t t = __shfl_up(incl, o);
            if (lane_id() >= o) incl += t;
        }
        if (lane_id() == kWave - 1) sm.wsum[w] = incl;
        __syncthreads();
        uint32_t below = carry;
        for (int q = 0; q < w; q++) below += sm.wsum[q];
        if (d < D) sm.start[d] = below + incl - tot;
        if (d0 + T < D) {
            for (int q = 0; q < WAVES; q++) carry += sm.wsum[q];
            __syncthreads();
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < ITEMS; i++) {
        if (i >= per) continue;
        const uint32_t d = (key[i] >> shift) & (D - 1);
        pos[i] += sm.start[d] + sm.cnt[w][d];
    }
    __syncthreads();
}

} // namespace vdb
