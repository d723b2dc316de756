// expand.hpp -- a pass over the nonzeros of a CSR or DCSR matrix that knows
// each one's row.
//
// f(e, r, id) is called for every nonzero e of [e_lo, e_hi) with the stored row
// r that holds it and that row's id (rows[r], or r without rows).  The work is
// cut into tiles of EX_TILE nonzeros: k_tile_rows, one thread per row, notes
// the row in which each tile begins, and a workgroup per tile copies its rows'
// pointers and ids into LDS, where every thread looks its nonzeros' rows up.
// Consecutive threads take consecutive nonzeros, so f's reads and writes are
// coalesced whatever the row lengths.
//
// What bounds it: HBM, at the bytes f moves.  One wave per row, which few rows or
// long ones still get (k_expand_by_rows), is bound by the chain row pointer ->
// columns and leaves most lanes idle on short rows (keys of 15.3 million nonzeros
// in 532 thousand rows: 258 us, 68 us now; row ids of 16.1 million nonzeros: 94
// us, 39 us now); finding each tile's first row inside its workgroup (a 256-way
// search, three dependent rounds) took 71 and 57 us.
#pragma once

#include "clb_internal.hpp"
#include "device_utils.hpp"

namespace clb {

constexpr u32 EX_WG = 256, EX_ITEMS = 8, EX_TILE = EX_WG * EX_ITEMS;

// first[t] = the row of nonzero e_lo + t * TILE, for every tile of [e_lo, e_hi)
// (e_hi == 0: of the rows' own nonzeros, which only the device knows).  Row
// pointers that cover less than [e_lo, e_hi), as of a CSR matrix with unused
// columns at its end, leave the rest to the first and the last row.
template <u32 TILE>
__device__ __forceinline__ void tile_rows(const u32 *__restrict__ rpt, u32 r_lo, u32 r_hi, u32 e_lo, u32 e_hi,
                                          u32 *__restrict__ first, u32 block) {
    const u64 r = (u64)r_lo + (u64)block * EX_WG + threadIdx.x;
    if (e_hi == 0) {
        e_lo = rpt[r_lo];
        e_hi = rpt[r_hi];
    }
    u32 t0 = 0, n = 0;  // tiles that begin in row r
    if (r < r_hi) {
        const u32 b = r != r_lo && rpt[r] > e_lo ? rpt[r] - e_lo : 0u;
        const u32 end = r + 1 != r_hi && rpt[r + 1] < e_hi ? rpt[r + 1] : e_hi;
        const u32 e = end > e_lo ? end - e_lo : 0u;
        t0 = (u32)(((u64)b + TILE - 1) / TILE);
        const u32 t1 = (u32)(((u64)e + TILE - 1) / TILE);
        n = e > b && t1 > t0 ? t1 - t0 : 0u;
        if (n <= 4) {
            for (u32 k = 0; k < n; ++k) first[t0 + k] = (u32)r;
            n = 0;
        }
    }
    // a row over many tiles: by the whole wave
    unsigned long long m = __ballot(n != 0);
    while (m) {
        const int s = __ffsll(m) - 1;
        m &= m - 1;
        const u32 st = __shfl(t0, s, dev::WAVE), sn = __shfl(n, s, dev::WAVE), sr = __shfl((u32)r, s, dev::WAVE);
        for (u32 k = (u32)dev::lane(); k < sn; k += dev::WAVE) first[st + k] = sr;
    }
}

template <u32 TILE>
__global__ __launch_bounds__(EX_WG) void k_tile_rows(const u32 *__restrict__ rpt, u32 r_lo, u32 r_hi, u32 e_lo,
                                                     u32 e_hi, u32 *__restrict__ first) {
    tile_rows<TILE>(rpt, r_lo, r_hi, e_lo, e_hi, first, blockIdx.x);
}

// Nonzeros [e_lo, e_hi) of rows [r_lo, r_hi).  rpt[r_lo .. r_hi] ascends (equal
// entries: empty rows), rpt[r_lo] <= e_lo and e_hi <= rpt[r_hi].
template <typename F>
struct Expand {
    const u32 *rpt, *rows;
    u32 r_lo, r_hi, e_lo, e_hi;
    F f;
    u32 tiles() const { return e_lo < e_hi && r_lo < r_hi ? div_up((u64)e_hi - e_lo, EX_TILE) : 0; }
};

// Tile `tile` of `tiles`.
template <typename F>
__device__ __forceinline__ void expand_tile(const Expand<F> &x, const u32 *__restrict__ first, u32 tile, u32 tiles) {
    __shared__ u32 srpt[EX_TILE], srow[EX_TILE];
    const u32 *__restrict__ rpt = x.rpt, *__restrict__ rows = x.rows;
    const F &f = x.f;
    const u64 e0 = (u64)x.e_lo + (u64)tile * EX_TILE;
    const u64 e1 = e0 + EX_TILE < x.e_hi ? e0 + EX_TILE : x.e_hi;
    const u32 r0 = first[tile];
    const u32 nr = (tile + 1 < tiles ? first[tile + 1] : x.r_hi - 1) - r0 + 1;
    const bool staged = nr <= EX_TILE;  // else: more (empty) rows in the tile than the copy holds
    if (staged) {
        for (u32 j = threadIdx.x; j < nr; j += EX_WG) {
            srpt[j] = rpt[r0 + j];
            srow[j] = rows ? rows[r0 + j] : r0 + j;
        }
    }
    __syncthreads();
#pragma unroll
    for (u32 q = 0; q < EX_ITEMS; ++q) {
        const u64 e = e0 + q * EX_WG + threadIdx.x;
        if (e >= e1) break;
        u32 a = 0, b = nr;  // the last row that starts at or before e
        if (staged) {
            while (b - a > 1) {
                const u32 m = (a + b) >> 1;
                if (srpt[m] <= e) a = m;
                else b = m;
            }
            f((u32)e, r0 + a, srow[a]);
        } else {
            while (b - a > 1) {
                const u32 m = a + ((b - a) >> 1);
                if (rpt[r0 + m] <= e) a = m;
                else b = m;
            }
            f((u32)e, r0 + a, rows ? rows[r0 + a] : r0 + a);
        }
    }
}

template <typename F>
__global__ __launch_bounds__(EX_WG) void k_expand(Expand<F> x, const u32 *__restrict__ first) {
    expand_tile(x, first, blockIdx.x, gridDim.x);
}

// A wave per row instead, for its first ER_LONG nonzeros, and one per ER_LONG
// nonzeros for what their first one's row has past that.  Rows that begin among
// them are written that far by their own waves, so nothing else is left to it.
constexpr u32 ER_LONG = 4096;
template <typename F>
__global__ __launch_bounds__(EX_WG) void k_expand_by_rows(Expand<F> x) {
    const u32 n = x.r_hi - x.r_lo, l = (u32)dev::lane();
    const u64 w = (u64)blockIdx.x * (EX_WG / dev::WAVE) + __builtin_amdgcn_readfirstlane(threadIdx.x / dev::WAVE);
    const u32 *__restrict__ rpt = x.rpt;
    // row r's nonzeros from its `skip`-th on, up to position stop
    auto fill = [&](u32 r, u32 skip, u64 pos, u64 stop) {
        u32 b = rpt[r], end = rpt[r + 1];
        const u32 id = x.rows ? x.rows[r] : r;
        if (r == x.r_lo || b < x.e_lo) b = x.e_lo;
        if (r + 1 == x.r_hi || end > x.e_hi) end = x.e_hi;
        if (b >= end || end - b <= skip) return;
        b += skip;
        if (b < pos) b = (u32)pos;
        if (end > stop) end = (u32)stop;
        if (b >= end) return;
        const u32 cnt = skip || end - b <= ER_LONG ? end - b : ER_LONG;
#pragma unroll 4
        for (u32 o = l; o < cnt; o += dev::WAVE) x.f(b + o, r, id);
    };
    if (w < n) {
        fill(x.r_lo + (u32)w, 0, 0, x.e_hi);
        return;
    }
    const u64 pos = x.e_lo + (w - n) * ER_LONG;
    if (pos >= x.e_hi) return;
    u32 r = x.r_lo, hi = x.r_hi;
    while (hi - r > 1) {  // the last row that starts at or before pos
        const u32 step = (hi - r + dev::WAVE - 1) / dev::WAVE;
        const u64 c = (u64)r + (u64)l * step;
        const u32 cnt = (u32)__popcll(__ballot(l == 0 || (c < hi && rpt[c] <= pos)));
        r += (cnt - 1) * step;
        hi = hi - r < step ? hi : r + step;
    }
    fill(r, ER_LONG, pos, pos + ER_LONG);
}

template <typename F>
void expand_rows(clb_controls_s *ctl, const Expand<F> &x) {
    const u32 tiles = x.tiles();
    if (!tiles) return;
    // One launch instead of two, but a wave for every row, however short: where
    // that takes no longer than the other launch and the search of a tile's rows.
    // Row ids in a call, by rows / by tiles (us): 1000 rows of 20 14.3 / 22.1, 30
    // thousand of 500 25.2 / 35.7, 100 thousand of 64 24.8 / 29.8, 200 thousand of
    // 30 36 / 31, a million of 17 129 / 53.
    const u32 n = x.r_hi - x.r_lo;
    if (n <= (1u << 16) + (x.e_hi - x.e_lo) / 64) {
        const u64 waves = (u64)n + div_up((u64)x.e_hi - x.e_lo, ER_LONG);
        k_expand_by_rows<F><<<div_up(waves, EX_WG / dev::WAVE), EX_WG, 0, ctl->stream>>>(x);
        CLB_LAUNCHED("expand_rows");
        return;
    }
    DevArray<u32> first(ctl, tiles);
    k_tile_rows<EX_TILE>
        <<<div_up(x.r_hi - x.r_lo, EX_WG), EX_WG, 0, ctl->stream>>>(x.rpt, x.r_lo, x.r_hi, x.e_lo, x.e_hi, first.ptr);
    CLB_LAUNCHED("tile_rows");
    k_expand<F><<<tiles, EX_WG, 0, ctl->stream>>>(x, first.ptr);
    CLB_LAUNCHED("expand_rows");
}

// Two matrices in the same launches (a small union is bound by its launches:
// 8000 rows, 64 and 32 thousand nonzeros, 88 us with four, 74 with two): the
// first `n` workgroups are a's.
template <typename F>
__global__ __launch_bounds__(EX_WG) void k_tile_rows_two(Expand<F> a, Expand<F> b, u32 n, u32 *__restrict__ first_a,
                                                         u32 *__restrict__ first_b) {
    const bool in_a = blockIdx.x < n;
    tile_rows<EX_TILE>(in_a ? a.rpt : b.rpt, in_a ? a.r_lo : b.r_lo, in_a ? a.r_hi : b.r_hi, in_a ? a.e_lo : b.e_lo,
                       in_a ? a.e_hi : b.e_hi, in_a ? first_a : first_b, in_a ? blockIdx.x : blockIdx.x - n);
}
template <typename F>
__global__ __launch_bounds__(EX_WG) void k_expand_two(Expand<F> a, Expand<F> b, u32 n, const u32 *__restrict__ first_a,
                                                      const u32 *__restrict__ first_b) {
    const bool in_a = blockIdx.x < n;
    const Expand<F> x = in_a ? a : b;
    expand_tile(x, in_a ? first_a : first_b, in_a ? blockIdx.x : blockIdx.x - n, in_a ? n : gridDim.x - n);
}
template <typename F>
void expand_rows_two(clb_controls_s *ctl, const Expand<F> &a, const Expand<F> &b) {
    const u32 ta = a.tiles(), tb = b.tiles();
    if (!ta || !tb) {
        expand_rows(ctl, a);
        expand_rows(ctl, b);
        return;
    }
    DevArray<u32> first(ctl, (u64)ta + tb);
    const u32 ra = div_up(a.r_hi - a.r_lo, EX_WG), rb = div_up(b.r_hi - b.r_lo, EX_WG);
    k_tile_rows_two<F><<<ra + rb, EX_WG, 0, ctl->stream>>>(a, b, ra, first.ptr, first.ptr + ta);
    CLB_LAUNCHED("tile_rows");
    k_expand_two<F><<<ta + tb, EX_WG, 0, ctl->stream>>>(a, b, ta, first.ptr, first.ptr + ta);
    CLB_LAUNCHED("expand_rows");
}

// keys[e - base] = (row id + shift) << 32 | cols[e]
struct KeyOfNonzero {
    const u32 *cols;
    u32 shift, base;
    u64 *keys;
    __device__ __forceinline__ void operator()(u32 e, u32, u32 id) const {
        keys[e - base] = ((u64)(id + shift) << 32) | cols[e];
    }
};

}  // namespace clb
