// radix.hpp -- the tile of a stable radix sort pass, shared by the sort of
// whole key arrays and the sort of rows by column.
#pragma once

#include "clb_internal.hpp"
#include "device_utils.hpp"

namespace clb {

constexpr int RX_WG = 256;
constexpr int RX_ITEMS = 16;
constexpr u32 RX_TILE = RX_WG * RX_ITEMS;
constexpr int RX_RADIX = 256;
constexpr u32 RX_COPIES = 4;

// Counts digit d of a valid lane in h[RX_RADIX * RX_COPIES].  RX_COPIES
// counters per digit, taken by lane, because equal digits of a wave's lanes
// (sorted or skewed input) would queue on one word, and a wave whose lanes all
// hold one digit adds them at once.
__device__ __forceinline__ void radix_count(u32 d, bool valid, u32 *h, u32 copy) {
    const unsigned long long all = __ballot(valid);
    const u32 f = __builtin_amdgcn_readfirstlane(d);
    u32 *c = &h[d * RX_COPIES + copy];
    if (__ballot(valid && d == f) == all) {
        if (valid && dev::lanes_below(all) == 0) atomicAdd(c, (u32)__popcll(all));
    } else if (valid) {
        atomicAdd(c, 1u);
    }
}

// A tile of cnt keys: wave w holds keys [w * WKEYS, (w + 1) * WKEYS), 64 per
// item.  Orders them by digit in skey (per wave, by ballots over the digit's
// bits and a counter per digit in LDS) and leaves in gbase[d] digit d's first
// place in the output (`place` of thread d) minus its first place in the tile.
template <typename K, typename D>
__device__ __forceinline__ void radix_tile(const K (&key)[RX_ITEMS], u32 cnt, int digit_bits, u32 place, K *skey,
                                           u32 (*wcnt)[RX_RADIX], u32 *gbase, u32 *red, D &&digit) {
    static_assert(RX_WG == RX_RADIX, "a thread per digit");
    constexpr int NW = RX_WG / dev::WAVE;
    constexpr u32 WKEYS = RX_TILE / NW;
    const int l = dev::lane(), w = dev::wave_id();
    const u32 o0 = (u32)w * WKEYS + (u32)l;
    const u32 d = threadIdx.x;
    // wcnt: keys of each digit so far per wave, then the waves' offsets
    for (int v = 0; v < NW; ++v) wcnt[v][d] = 0;
    __syncthreads();
    const unsigned long long lt = (1ull << l) - 1ull;
    u32 rank[RX_ITEMS];
#pragma unroll
    for (int q = 0; q < RX_ITEMS; ++q) {
        const bool valid = o0 + q * dev::WAVE < cnt;
        const u32 d = digit(key[q]);
        unsigned long long peers = __ballot(valid);
        for (int b = 0; b < digit_bits; ++b) {
            const bool bit = (d >> b) & 1u;
            const unsigned long long m = __ballot(bit);
            peers &= bit ? m : ~m;
        }
        const u32 below = (u32)__popcll(peers & lt);
        const u32 before = wcnt[w][d];
        rank[q] = before + below;
        __builtin_amdgcn_wave_barrier();
        if (valid && below == 0) wcnt[w][d] = before + (u32)__popcll(peers);
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
    // digit d's count in the tile and the waves' offsets, from the tile's start
    u32 mine = 0, total;
#pragma unroll
    for (int v = 0; v < NW; ++v) {
        const u32 c = wcnt[v][d];
        wcnt[v][d] = mine;
        mine += c;
    }
    const u32 ls = dev::block_excl_scan<u32, RX_WG>(mine, red, total);
#pragma unroll
    for (int v = 0; v < NW; ++v) wcnt[v][d] += ls;
    gbase[d] = place - ls;
    __syncthreads();
#pragma unroll
    for (int q = 0; q < RX_ITEMS; ++q)
        if (o0 + q * dev::WAVE < cnt) skey[wcnt[w][digit(key[q])] + rank[q]] = key[q];
    __syncthreads();
}

}  // namespace clb
