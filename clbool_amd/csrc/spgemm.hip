// spgemm.hip -- host driver of the boolean SpGEMM C = A * B (DCSR).
//
// Plain mode follows the two-pass structure of clBool's
// dcsr::matrix_multiplication_hash (src/dcsr/dcsr_matrix_multiplication_hash.cpp:51-119):
// count products per row (count_workload, dcsr_matrix_multiplication.cpp:388-404),
// bin rows (build_groups_and_allocate_hash, hash.cpp:301-345 -- here on the
// device, no per-row host loop), symbolic pass (count_nnz, :122-201), scan
// (fill_nnz's prefix_sum, :218), numeric pass (:235-280), drop empty rows
// (prepare_positions + set_positions, :282-296).  Learned mode lives in
// learned.hip and shares the kernels.
#include "expand.hpp"
#include "spgemm.hpp"

#include <chrono>
#include <sstream>
#include <type_traits>

namespace clb {
namespace spg {

// Mats::splits of B: for each stored row, the start of each column slice of
// `span` columns (lower bounds in the sorted row) and its end.  A thread per
// entry: one per row walked its slices' searches one after the other (150 us
// for 168 thousand rows of 16 slices, 22 us now).  b_rows == nullptr: the
// table is by stored row.
__global__ void k_slice_splits(const u32 *__restrict__ b_rpt, const u32 *__restrict__ b_rows,
                               const u32 *__restrict__ b_cols, u32 b_nzr, u32 mapn, u32 nsl, u64 span,
                               u32 *__restrict__ splits) {
    const u64 t = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (u64)b_nzr * (nsl + 1)) return;  // below 2^32: the table is
    const u32 i = (u32)t / (nsl + 1), s = (u32)t - i * (nsl + 1);
    const u32 k = b_rows ? b_rows[i] : i;
    if (k >= mapn) return;
    u32 lo = b_rpt[i];
    const u32 end = b_rpt[i + 1];
    const u64 bound = (u64)s * span;
    u32 hi = s ? end : lo;
    if (s == nsl) lo = end;
    while (lo < hi) {  // first column >= bound
        const u32 mid = lo + (hi - lo) / 2;
        if ((u64)b_cols[mid] < bound) lo = mid + 1;
        else hi = mid;
    }
    splits[(u64)k * (nsl + 1) + s] = lo;
}

// Packed B (Mats::b_packs): a pack begins at every column that starts a row or
// a new group of 16.  The count pass gives each tile of EX_TILE columns its
// packs; once these are scanned, the thread of a pack's first column collects
// the columns of its group from the lanes after it (past its wave, and past
// the tile, from memory) and writes the pack and where its first column is.
// Rows' first packs come from the number of packs before the row's position,
// so that stored rows without entries have an empty range.  A search of every
// column's row and a walk along its group took 0.95 and 2.9 ms for 191 million
// columns (0.27 and 1.1 ms now).
constexpr u32 PK_WORDS = EX_TILE / 32;
struct PackTile {
    u64 e0, e1;
    u32 r0, nr;  // rows from the one that holds e0 to the one that holds e1
    bool last;
    // (columns past the last row's end are no entries)
    __device__ __forceinline__ PackTile(const u32 *__restrict__ first, const u32 *__restrict__ b_rpt, u32 b_nzr,
                                        u32 b_nnz) {
        const u32 end = b_rpt[b_nzr];
        const u64 n = end < b_nnz ? end : b_nnz;
        e0 = (u64)blockIdx.x * EX_TILE;
        e1 = e0 + EX_TILE < n ? e0 + EX_TILE : n;
        last = e1 == n;
        r0 = first[blockIdx.x];
        nr = (last ? b_nzr - 1 : first[blockIdx.x + 1]) - r0 + 1;
    }
    __device__ __forceinline__ bool empty() const { return e0 >= e1; }
    // c[q] = column e0 + q * EX_WG + threadIdx.x, sb = a bit per column that
    // begins a pack (complete after a barrier).
    __device__ __forceinline__ void starts(const u32 *__restrict__ b_rpt, const u32 *__restrict__ b_cols,
                                           u32 (&c)[EX_ITEMS], u32 *sb) const {
        __shared__ u32 mk[PK_WORDS];  // row starts
        if (threadIdx.x < PK_WORDS) mk[threadIdx.x] = 0;
        u32 before[EX_ITEMS];  // lane 0: the column before its own
#pragma unroll
        for (u32 q = 0; q < EX_ITEMS; ++q) {
            const u64 e = e0 + q * EX_WG + threadIdx.x;
            c[q] = e < e1 ? b_cols[e] : 0u;
            before[q] = dev::lane() == 0 && e && e < e1 ? b_cols[e - 1] : 0u;
        }
        __syncthreads();
        for (u32 j = threadIdx.x; j < nr; j += EX_WG) {
            const u32 pos = b_rpt[r0 + j];
            if (pos >= e0 && pos < e1) atomicOr(&mk[(pos - e0) >> 5], 1u << ((pos - e0) & 31u));
        }
        __syncthreads();
#pragma unroll
        for (u32 q = 0; q < EX_ITEMS; ++q) {
            const u32 o = q * EX_WG + threadIdx.x;
            u32 p = __shfl_up(c[q], 1, dev::WAVE);
            if (dev::lane() == 0) p = before[q];
            const bool st = e0 + o < e1 && (((mk[o >> 5] >> (o & 31u)) & 1u) || (p >> 4) != (c[q] >> 4));
            const unsigned long long m = __ballot(st);
            if ((dev::lane() & 31) == 0) sb[o >> 5] = (u32)(dev::lane() ? m >> 32 : m);
        }
    }
};

__global__ __launch_bounds__(EX_WG) void k_pack_count(const u32 *__restrict__ b_rpt, const u32 *__restrict__ b_cols,
                                                      u32 b_nzr, u32 b_nnz, const u32 *__restrict__ first,
                                                      u32 *__restrict__ counts) {
    __shared__ u32 sb[PK_WORDS];
    const PackTile t(first, b_rpt, b_nzr, b_nnz);
    if (t.empty()) {  // uniform
        if (threadIdx.x == 0) counts[blockIdx.x] = 0;
        return;
    }
    u32 c[EX_ITEMS];
    t.starts(b_rpt, b_cols, c, sb);
    __syncthreads();
    if (threadIdx.x >= dev::WAVE) return;
    static_assert(PK_WORDS == dev::WAVE, "one wave counts a tile");
    const u32 sum = dev::wave_sum((u32)__popc(sb[threadIdx.x]));
    if (threadIdx.x == 0) counts[blockIdx.x] = sum;
}

__global__ __launch_bounds__(EX_WG) void k_pack_place(const u32 *__restrict__ b_rpt, const u32 *__restrict__ b_cols,
                                                      u32 b_nzr, u32 b_nnz, const u32 *__restrict__ first,
                                                      const u32 *__restrict__ offs, u32 *__restrict__ prpt,
                                                      u32 *__restrict__ packs, u32 *__restrict__ pfirst) {
    __shared__ u32 sb[PK_WORDS], spre[PK_WORDS + 1];
    const PackTile t(first, b_rpt, b_nzr, b_nnz);
    if (t.empty()) return;  // uniform
    u32 c[EX_ITEMS];
    t.starts(b_rpt, b_cols, c, sb);
    __syncthreads();
    if (threadIdx.x < dev::WAVE) {
        const u32 n = (u32)__popc(sb[threadIdx.x]), inc = dev::wave_incl_scan(n);
        spre[threadIdx.x] = offs[blockIdx.x] + inc - n;
        if (threadIdx.x == dev::WAVE - 1) spre[PK_WORDS] = offs[blockIdx.x] + inc;
    }
    __syncthreads();
    // packs before position e0 + o
    auto rank = [&](u32 o) {
        return o == EX_TILE ? spre[PK_WORDS] : spre[o >> 5] + (u32)__popc(sb[o >> 5] & ((1u << (o & 31u)) - 1u));
    };
    // where the row that holds the tile's last column ends
    const u32 rn = t.r0 + t.nr - 1;
    const u64 limit = !t.last && b_rpt[rn] < t.e1 ? b_rpt[rn + 1] : t.e1;
    const int l = dev::lane();
#pragma unroll
    for (u32 q = 0; q < EX_ITEMS; ++q) {
        const u32 o = q * EX_WG + threadIdx.x;
        const u32 ow = o & ~63u;  // the wave's first
        const unsigned long long m = ((unsigned long long)sb[(ow >> 5) + 1] << 32) | sb[ow >> 5];
        const unsigned long long later = l == 63 ? 0ull : m >> (l + 1);
        const u32 left = t.e1 - t.e0 > ow ? (u32)(t.e1 - t.e0 - ow) : 0u;  // the wave's columns
        const u32 valid = left < 64u ? left : 64u;
        const u32 end = later ? (u32)l + (u32)__ffsll(later) : valid;  // of this lane's group in the wave
        const u32 w = c[q] >> 4;
        u32 mask = (u32)l < valid ? 1u << (c[q] & 15u) : 0u;
#pragma unroll
        for (u32 d = 1; d < 16; d <<= 1) {
            const u32 x = __shfl_down(mask, d, dev::WAVE);
            if ((u32)l + d < end) mask |= x;
        }
        if (!((m >> l) & 1u)) continue;
        if (!later) {  // the group may go on after the wave
            u64 k = t.e0 + ow + 64;
            for (; k < t.e1 && !((sb[(u32)(k - t.e0) >> 5] >> ((u32)(k - t.e0) & 31u)) & 1u); ++k)
                mask |= 1u << (b_cols[k] & 15u);
            if (k >= t.e1)
                for (k = t.e1; k < limit && (b_cols[k] >> 4) == w; ++k) mask |= 1u << (b_cols[k] & 15u);
        }
        const u32 p = rank(o);
        packs[p] = (w << 16) | mask;
        if (pfirst) pfirst[p] = (u32)(t.e0 + o);
    }
    for (u32 j = threadIdx.x; j < t.nr; j += EX_WG) {
        const u32 pos = b_rpt[t.r0 + j];
        if (pos >= t.e0 && pos <= t.e1) prpt[t.r0 + j] = rank((u32)(pos - t.e0));
    }
    if (blockIdx.x == 0)
        for (u32 r = threadIdx.x; r < t.r0; r += EX_WG) prpt[r] = 0;  // without entries
    if (t.last && threadIdx.x == 0) prpt[b_nzr] = spre[PK_WORDS];
}

// Mats::psplits from Mats::splits: slices begin at multiples of 16 columns, so
// the pack that a slice begins with has the slice's first column first.
__global__ void k_pack_splits(const u32 *__restrict__ prpt, const u32 *__restrict__ b_rows,
                              const u32 *__restrict__ pfirst, const u32 *__restrict__ splits, u32 b_nzr, u32 mapn,
                              u32 nsl, u32 *__restrict__ psplits) {
    const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= b_nzr) return;
    const u32 k = b_rows ? b_rows[i] : i;
    if (k >= mapn) return;
    const u32 end = prpt[i + 1];
    const u64 at = (u64)k * (nsl + 1);
    u32 lo = prpt[i];
    psplits[at] = lo;
    for (u32 s = 1; s < nsl; ++s) {
        const u32 e = splits[at + s];
        u32 hi = end;
        while (lo < hi) {
            const u32 mid = lo + (hi - lo) / 2;
            if (pfirst[mid] < e) lo = mid + 1;
            else hi = mid;
        }
        psplits[at + s] = lo;
    }
    psplits[at + nsl] = end;
}

// brange by row id (b_rows == nullptr: by stored row); for a filtered A also
// the stored row of each id (bidx) and the ranges by stored row (crange).
__global__ void k_brange_set(const u32 *__restrict__ b_rpt, const u32 *__restrict__ b_rows, u32 b_nzr, u32 mapn,
                             uint2 *__restrict__ brange, u32 *__restrict__ bpres, u32 *__restrict__ bidx,
                             uint2 *__restrict__ crange) {
    const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= b_nzr) return;
    const uint2 range = make_uint2(b_rpt[i], b_rpt[i + 1]);
    if (crange) crange[i] = range;
    const u32 r = b_rows ? b_rows[i] : i;
    if (r >= mapn) return;
    brange[r] = range;
    if (bidx) bidx[r] = i;
    if (bpres) atomicOr(&bpres[r >> 5], 1u << (r & 31));
}

// Per-row statistics of rows [row0, row0 + nrows) of A over its B rows, cut by
// nonzeros: a tile of RSTAT_WG * ITEMS of them per workgroup, whose rows come
// from k_tile_rows.  A thread takes ITEMS consecutive nonzeros, sums them up
// while the row stays the same, and adds to the row's place in LDS; a row
// inside the tile is stored, one that crosses its border is merged with global
// atomics (a row spread over several tiles from each).  Random reads of B's
// row map bound it.  No total is kept here: the row sums are binned anyway,
// and one counter for all workgroups took 11 ns for each of them (64 thousand
// workgroups of 256 nonzeros: 728 us for 16.5 million nonzeros, 124 us now).
//   prod[r] = products (border rows must start at 0);
//   FEAT: also mn/mx (min/max B-row length, border rows start at ~0 / 0) and
//   fc/lc (first column of any of its B rows / last column, ~0 / 0).
// With fmask also a bit per nonzero, set if its B row has entries, and each
// tile's number of them (for k_filter).
constexpr u32 RSTAT_WG = 256;
template <bool FEAT>
constexpr u32 rstat_tile() { return RSTAT_WG * (FEAT ? 4 : 8); }
template <bool FEAT>
__global__ __launch_bounds__(RSTAT_WG) void k_row_stats(Mats g, u32 nrows, const u32 *__restrict__ first,
                                                        u32 *__restrict__ prod, RowFeat o,
                                                        u32 *__restrict__ fmask, u32 *__restrict__ fcount) {
    constexpr u32 TILE = rstat_tile<FEAT>(), ITEMS = TILE / RSTAT_WG;
    __shared__ u32 red[RSTAT_WG / dev::WAVE + 1];
    __shared__ u32 rs[TILE + 1], sp[TILE];
    __shared__ u32 smn[FEAT ? TILE : 1], smx[FEAT ? TILE : 1], sfc[FEAT ? TILE : 1], slc[FEAT ? TILE : 1];
    const u32 rend = g.row0 + nrows;
    const u32 jbase = g.a_all[g.row0], jend = g.a_all[rend];
    const u64 j0 = (u64)jbase + (u64)blockIdx.x * TILE;
    if (j0 >= jend) {  // uniform: the grid covers all of A's nonzeros
        if (fmask && threadIdx.x == 0) fcount[blockIdx.x] = 0;
        return;
    }
    const u64 j1 = j0 + TILE < jend ? j0 + TILE : jend;
    const u32 r0 = first[blockIdx.x];
    const u32 nr = (j1 < jend ? first[blockIdx.x + 1] : rend - 1) - r0 + 1;
    const bool staged = nr <= TILE;  // else: some stored rows are empty
    if (staged) {
        for (u32 t = threadIdx.x; t <= nr; t += RSTAT_WG) rs[t] = g.a_all[r0 + t];
        for (u32 t = threadIdx.x; t < nr; t += RSTAT_WG) {
            sp[t] = 0;
            if (FEAT) {
                smn[t] = sfc[t] = 0xFFFFFFFFu;
                smx[t] = slc[t] = 0;
            }
        }
    }
    __syncthreads();
    const u64 js = j0 + (u64)threadIdx.x * ITEMS;
    u32 bits = 0;  // this thread's nonzeros with a B row
    if (js < j1) {
        uint2 b[ITEMS];
        u32 c0[ITEMS], c1[ITEMS];
#pragma unroll
        for (u32 k = 0; k < ITEMS; ++k) b[k] = js + k < j1 ? b_range(g, g.a_cols[js + k]) : make_uint2(0u, 0u);
#pragma unroll
        for (u32 k = 0; k < ITEMS; ++k) bits |= (b[k].y > b[k].x ? 1u : 0u) << k;
        if (FEAT) {
#pragma unroll
            for (u32 k = 0; k < ITEMS; ++k) {
                c0[k] = b[k].y > b[k].x ? g.b_cols[b[k].x] : 0xFFFFFFFFu;
                c1[k] = b[k].y > b[k].x ? g.b_cols[b[k].y - 1] : 0u;
            }
        }
        u32 lo = 0, hi = nr;  // the last row that starts at or before js
        while (hi - lo > 1) {
            const u32 mid = lo + (hi - lo) / 2;
            if ((staged ? rs[mid] : g.a_all[r0 + mid]) <= js) lo = mid;
            else hi = mid;
        }
        u32 sum = 0, n0 = 0xFFFFFFFFu, n1 = 0, f0 = 0xFFFFFFFFu, f1 = 0;
        auto flush = [&]() {
            if (!sum) return;
            u32 *pp = staged ? &sp[lo] : &prod[r0 + lo - g.row0];
            atomicAdd(pp, sum);
            if (FEAT) {
                const u32 q = r0 + lo - g.row0;
                atomicMin(staged ? &smn[lo] : &o.mn[q], n0);
                atomicMax(staged ? &smx[lo] : &o.mx[q], n1);
                atomicMin(staged ? &sfc[lo] : &o.fc[q], f0);
                atomicMax(staged ? &slc[lo] : &o.lc[q], f1);
            }
            sum = 0;
            n0 = f0 = 0xFFFFFFFFu;
            n1 = f1 = 0;
        };
#pragma unroll
        for (u32 k = 0; k < ITEMS; ++k) {
            if (js + k >= j1) break;
            while ((staged ? rs[lo + 1] : g.a_all[r0 + lo + 1]) <= js + k) {
                flush();
                ++lo;
            }
            const u32 len = b[k].y - b[k].x;
            sum += len;
            if (FEAT && len) {
                n0 = len < n0 ? len : n0;
                n1 = len > n1 ? len : n1;
                f0 = c0[k] < f0 ? c0[k] : f0;
                f1 = c1[k] > f1 ? c1[k] : f1;
            }
        }
        flush();
    }
    if (fmask) {  // uniform
        constexpr u32 PER = 32 / ITEMS;  // threads of a word
        u32 w = bits << (threadIdx.x % PER * ITEMS);
#pragma unroll
        for (u32 d = 1; d < PER; d <<= 1) w |= __shfl_xor(w, d, dev::WAVE);
        if (threadIdx.x % PER == 0) fmask[(u64)blockIdx.x * (TILE / 32) + threadIdx.x / PER] = w;
        const u32 sum = dev::block_sum<u32, RSTAT_WG>((u32)__popc(bits), red);
        if (threadIdx.x == 0) fcount[blockIdx.x] = sum;
    }
    __syncthreads();
    if (!staged) return;
    for (u32 t = threadIdx.x; t < nr; t += RSTAT_WG) {
        const u32 row = r0 + t - g.row0;
        if (rs[t] >= j0 && rs[t + 1] <= j1) {  // the whole row
            prod[row] = sp[t];
            if (FEAT) {
                o.mn[row] = smn[t];
                o.mx[row] = smx[t];
                o.fc[row] = sfc[t];
                o.lc[row] = slc[t];
            }
        } else if (sp[t]) {
            atomicAdd(&prod[row], sp[t]);
            if (FEAT) {
                atomicMin(&o.mn[row], smn[t]);
                atomicMax(&o.mx[row], smx[t]);
                atomicMin(&o.fc[row], sfc[t]);
                atomicMax(&o.lc[row], slc[t]);
            }
        }
    }
}

// A without the nonzeros whose B row is absent or empty, its columns renumbered
// to B's stored rows: the first `tiles` workgroups place the columns of a tile
// of k_row_stats each, the others the row pointers.
template <u32 TILE>
__global__ __launch_bounds__(256) void k_filter(Mats g, u32 nrows, u32 tiles, const u32 *__restrict__ fmask,
                                                const u32 *__restrict__ offs, const u32 *__restrict__ bidx,
                                                u32 *__restrict__ f_rpt, u32 *__restrict__ f_cols) {
    constexpr u32 W = TILE / 32;
    static_assert(W <= dev::WAVE, "one wave scans a tile's words");
    const u32 jbase = g.a_all[g.row0];
    if (blockIdx.x >= tiles) {
        const u64 r = (u64)(blockIdx.x - tiles) * 256 + threadIdx.x;
        if (r > nrows) return;
        const u32 e = g.a_all[g.row0 + r] - jbase, t = e / TILE;
        u32 n = offs[t];  // offs[tiles]: all of them
        const u32 *m = fmask + (u64)t * W;
        for (u32 q = 0; q < e % TILE / 32; ++q) n += (u32)__popc(m[q]);
        if (e % 32) n += (u32)__popc(m[e % TILE / 32] & ((1u << e % 32) - 1u));
        f_rpt[r] = n;
        return;
    }
    const u64 n = (u64)g.a_all[g.row0 + nrows] - jbase, e0 = (u64)blockIdx.x * TILE;
    if (e0 >= n) return;
    __shared__ u32 sw[W], sp[W];
    if (threadIdx.x < dev::WAVE) {
        const u32 w = threadIdx.x < W ? fmask[(u64)blockIdx.x * W + threadIdx.x] : 0u;
        const u32 c = (u32)__popc(w), inc = dev::wave_incl_scan(c);
        if (threadIdx.x < W) {
            sw[threadIdx.x] = w;
            sp[threadIdx.x] = offs[blockIdx.x] + inc - c;
        }
    }
    __syncthreads();
#pragma unroll
    for (u32 q = 0; q < TILE / 256; ++q) {
        const u32 e = q * 256 + threadIdx.x, w = sw[e / 32], bit = 1u << e % 32;
        if (w & bit) f_cols[sp[e / 32] + (u32)__popc(w & (bit - 1u))] = bidx[g.a_cols[(u64)jbase + e0 + e]];
    }
}

// The start values of a product's buffers in one launch: the B row map (or its
// presence bits), the scalars, the row statistics.
__global__ void k_init(u64 *__restrict__ map, u64 nmap, u32 *__restrict__ bits, u64 nbits, u64 *__restrict__ scal,
                       u32 nscal, u32 *__restrict__ prod, u32 nrows, RowFeat o) {
    const u64 stride = (u64)gridDim.x * blockDim.x;
    const u64 i0 = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    for (u64 i = i0; i < nmap; i += stride) map[i] = 0;
    for (u64 i = i0; i < nbits; i += stride) bits[i] = 0;
    if (i0 < nscal) scal[i0] = 0;
    if (!prod) return;
    for (u64 i = i0; i < nrows; i += stride) {
        prod[i] = 0;
        if (o.mn) {
            o.mn[i] = o.fc[i] = 0xFFFFFFFFu;
            o.mx[i] = o.lc[i] = 0;
        }
    }
}

// Binning in two launches over the same split of the rows into gridDim.x
// stretches: k_bin_count leaves each stretch's counts and sums per bin,
// k_bin_place adds up the stretches before its own, places its rows and (the
// first workgroup) leaves the totals with the product's scalars in host
// memory.  Few workgroups and no shared counters: 2276 of them adding to 128
// words took 35 us, and 28 us to place them, for 582 thousand rows; 16 and 13 now.
//
// key == nullptr: key = min(P, ncols) (symbolic sizing).  Rows in BIN_EMPTY
// get nnz_row = 0 when nnz_row is given.  A row with a slot (slot_of, may be
// null) is a BIN_STORED row.  The order inside a bin is not significant:
// output positions come from the scan of row sizes.
constexpr u32 BIN_WG = 256, BIN_GRID = 128;
struct BinPart {
    u32 rows[NBINS];
    u64 sums[3][NBINS];  // products, A nonzeros, key (output nnz)
};
__device__ __forceinline__ u32 bin_of(u32 i, const u32 *P, const u32 *key, const BinCfg &c, const u32 *slot_of,
                                      u32 &p, u32 &k) {
    p = P[i];
    k = key ? key[i] : (p < c.ncols ? p : c.ncols);
    return slot_of && slot_of[i] ? BIN_STORED : classify(p, k, c);
}

__global__ __launch_bounds__(BIN_WG) void k_bin_count(Mats g, const u32 *__restrict__ P, const u32 *__restrict__ key,
                                                      u32 n, u32 per, BinCfg c, BinPart *__restrict__ parts,
                                                      u32 *__restrict__ nnz_row, const u32 *__restrict__ slot_of) {
    __shared__ u32 h[NBINS];
    __shared__ unsigned long long hs[3][NBINS];
    if (threadIdx.x < NBINS) {
        h[threadIdx.x] = 0;
        hs[0][threadIdx.x] = hs[1][threadIdx.x] = hs[2][threadIdx.x] = 0;
    }
    __syncthreads();
    const u64 i0 = (u64)blockIdx.x * per, i1 = i0 + per < n ? i0 + per : n;
    for (u64 i = i0 + threadIdx.x; i < i1; i += BIN_WG) {
        u32 p, k;
        const u32 b = bin_of((u32)i, P, key, c, slot_of, p, k);
        atomicAdd(&h[b], 1u);
        if (p) atomicAdd(&hs[0][b], (unsigned long long)p);
        atomicAdd(&hs[1][b], (unsigned long long)(g.a_all[g.row0 + i + 1] - g.a_all[g.row0 + i]));
        if (key && k) atomicAdd(&hs[2][b], (unsigned long long)k);
        if (b == BIN_EMPTY && nnz_row) nnz_row[i] = 0;
    }
    __syncthreads();
    if (threadIdx.x < NBINS) {
        parts[blockIdx.x].rows[threadIdx.x] = h[threadIdx.x];
        for (int q = 0; q < 3; ++q) parts[blockIdx.x].sums[q][threadIdx.x] = hs[q][threadIdx.x];
    }
}

__global__ __launch_bounds__(BIN_WG) void k_bin_place(const u32 *__restrict__ P, const u32 *__restrict__ key, u32 n,
                                                      u32 per, BinCfg c, const BinPart *__restrict__ parts,
                                                      u32 *__restrict__ perm, const u32 *__restrict__ slot_of,
                                                      const u64 *__restrict__ scal, BinTotals *__restrict__ host) {
    __shared__ u32 cursor[NBINS], total[NBINS];
    __shared__ unsigned long long hs[3 * NBINS];
    if (threadIdx.x < NBINS) cursor[threadIdx.x] = total[threadIdx.x] = 0;
    __syncthreads();
    const u32 b = threadIdx.x % NBINS;
    u32 before = 0, all = 0;
#pragma unroll 4
    for (u32 w = threadIdx.x / NBINS; w < gridDim.x; w += BIN_WG / NBINS) {
        const u32 v = parts[w].rows[b];
        before += w < blockIdx.x ? v : 0u;
        all += v;
    }
    atomicAdd(&cursor[b], before);
    atomicAdd(&total[b], all);
    __syncthreads();
    if (threadIdx.x < dev::WAVE) {  // one wave: the bins' starts
        const u32 v = threadIdx.x < NBINS ? total[threadIdx.x] : 0u;
        const u32 start = dev::wave_incl_scan(v) - v;
        if (threadIdx.x < NBINS) cursor[threadIdx.x] += start;
    }
    __syncthreads();
    const u64 i0 = (u64)blockIdx.x * per, i1 = i0 + per < n ? i0 + per : n;
    for (u64 i = i0 + threadIdx.x; i < i1; i += BIN_WG) {
        u32 p, k;
        const u32 q = bin_of((u32)i, P, key, c, slot_of, p, k);
        if (q != BIN_EMPTY) perm[atomicAdd(&cursor[q], 1u)] = (u32)i;
    }
    if (blockIdx.x == 0) {
        if (threadIdx.x < 3 * NBINS) hs[threadIdx.x] = 0;
        __syncthreads();
        for (u32 q = 0; q < 3; ++q) {
            u64 v = 0;
#pragma unroll 4
            for (u32 w = threadIdx.x / NBINS; w < gridDim.x; w += BIN_WG / NBINS) v += parts[w].sums[q][b];
            if (v) atomicAdd(&hs[q * NBINS + b], (unsigned long long)v);
        }
        __syncthreads();
        if (threadIdx.x < NBINS) host->rows[threadIdx.x] = total[threadIdx.x];
        if (threadIdx.x < 3 * NBINS) host->sums[threadIdx.x] = hs[threadIdx.x];
        if (threadIdx.x < SCALARS) host->scal[threadIdx.x] = scal[threadIdx.x];
    }
}

// Offsets (off[i], u64; off[n] the total) and stored-row positions (pos[i]: the
// nonempty rows before i) of the exact row sizes, in tiles of SZ_TILE rows: sums
// per tile, their scan by one workgroup, and the tiles again.  scal[1] and
// scal[2] receive the totals.
constexpr u32 SZ_WG = 256, SZ_ITEMS = 8, SZ_TILE = SZ_WG * SZ_ITEMS;
struct SizeSum {
    u64 nnz;
    u64 rows;
};
__device__ __forceinline__ void load_sizes(const u32 *__restrict__ nnz_row, u32 n, u64 i, u32 (&v)[SZ_ITEMS]) {
    if (i + SZ_ITEMS <= n && (reinterpret_cast<uintptr_t>(nnz_row) & 15u) == 0) {  // i is a multiple of 8
        const uint4 a = *reinterpret_cast<const uint4 *>(nnz_row + i);
        const uint4 b = *reinterpret_cast<const uint4 *>(nnz_row + i + 4);
        v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
        v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
    } else {
#pragma unroll
        for (u32 k = 0; k < SZ_ITEMS; ++k) v[k] = i + k < n ? nnz_row[i + k] : 0u;
    }
}

__global__ __launch_bounds__(SZ_WG) void k_sizes_sum(const u32 *__restrict__ nnz_row, u32 n,
                                                     SizeSum *__restrict__ sums) {
    __shared__ u64 red[SZ_WG / dev::WAVE + 1];
    u32 v[SZ_ITEMS];
    load_sizes(nnz_row, n, (u64)blockIdx.x * SZ_TILE + (u64)threadIdx.x * SZ_ITEMS, v);
    u64 s = 0, r = 0;
#pragma unroll
    for (u32 k = 0; k < SZ_ITEMS; ++k) {
        s += v[k];
        r += v[k] != 0u;
    }
    const u64 ts = dev::block_sum<u64, SZ_WG>(s, red), tr = dev::block_sum<u64, SZ_WG>(r, red);
    if (threadIdx.x == 0) sums[blockIdx.x] = SizeSum{ts, tr};
}

__global__ __launch_bounds__(SZ_WG) void k_sizes_scan(SizeSum *__restrict__ sums, u32 tiles, u64 *__restrict__ last,
                                                      u64 *__restrict__ scal) {
    __shared__ u64 red[SZ_WG / dev::WAVE + 1];
    u64 cs = 0, cr = 0;
    for (u32 t0 = 0; t0 < tiles; t0 += SZ_WG) {
        const u32 t = t0 + threadIdx.x;
        const SizeSum v = t < tiles ? sums[t] : SizeSum{0, 0};
        u64 as, ar;
        const u64 s = dev::block_excl_scan<u64, SZ_WG>(v.nnz, red, as);
        const u64 r = dev::block_excl_scan<u64, SZ_WG>(v.rows, red, ar);
        if (t < tiles) sums[t] = SizeSum{cs + s, cr + r};
        cs += as;
        cr += ar;
    }
    if (threadIdx.x == 0) {
        *last = scal[1] = cs;
        scal[2] = cr;
    }
}

// sums == nullptr: the only tile, which also leaves the totals.
__global__ __launch_bounds__(SZ_WG) void k_sizes_place(const u32 *__restrict__ nnz_row, u32 n,
                                                       const SizeSum *__restrict__ sums, u64 *__restrict__ off,
                                                       u32 *__restrict__ pos, u64 *__restrict__ scal) {
    __shared__ u64 red[SZ_WG / dev::WAVE + 1];
    const u64 i = (u64)blockIdx.x * SZ_TILE + (u64)threadIdx.x * SZ_ITEMS;
    u32 v[SZ_ITEMS];
    load_sizes(nnz_row, n, i, v);
    u64 s = 0, r = 0;
#pragma unroll
    for (u32 k = 0; k < SZ_ITEMS; ++k) {
        s += v[k];
        r += v[k] != 0u;
    }
    u64 as, ar;
    u64 o = dev::block_excl_scan<u64, SZ_WG>(s, red, as);
    u64 q = dev::block_excl_scan<u64, SZ_WG>(r, red, ar);
    if (sums) {
        o += sums[blockIdx.x].nnz;
        q += sums[blockIdx.x].rows;
    } else if (threadIdx.x == 0) {
        off[n] = scal[1] = as;
        scal[2] = ar;
    }
#pragma unroll
    for (u32 k = 0; k < SZ_ITEMS; ++k) {
        if (i + k < n) {
            off[i + k] = o;
            pos[i + k] = (u32)q;
        }
        o += v[k];
        q += v[k] != 0u;
    }
}

// prepare_for_shift_empty_rows + set_positions_pointers_and_rows
// (prepare_positions.cl:69-84, set_positions.cl:46-66).
__global__ void k_set_positions(const u32 *__restrict__ nnz_row, const u64 *__restrict__ off,
                                const u32 *__restrict__ pos, u32 n, const u32 *__restrict__ a_rows, u32 row0,
                                u32 *__restrict__ c_rpt, u32 *__restrict__ c_rows, u32 nnz, u32 nzr) {
    const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i == 0) c_rpt[nzr] = nnz;
    if (i >= n || nnz_row[i] == 0) return;
    const u32 q = pos[i];
    c_rpt[q] = static_cast<u32>(off[i]);
    c_rows[q] = a_rows[row0 + i];
}

// Writes one dumped row (`parts` workgroups per row) into its columns at their
// final positions.  Each of the 2 waves owns a contiguous half of its part of the
// row's words; its start position is the prefix of the chunk counts before its
// first chunk, so the waves need no exchange.  A bitmap slice is loaded 1024
// words at a time (four rounds of 256, 16 bytes per lane per round),
// double-buffered (the next 1024 words' loads are in flight while the
// current ones are expanded); a slice dumped as (word index, word) pairs is
// read 256 pairs per round.  Either way the words are expanded by rank
// (dev::emit_round4_ranked), a lane per column, so every store instruction is
// one contiguous run.  Two-wave workgroups let more rows share a CU, so one
// row's load latency overlaps another's expansion.  gpre = exclusive prefix of chunk_cnt over all slots.
// A wave's expansion is a chain of LDS reads, so few rows with a workgroup each
// would leave the chip idle: the one pass of 10 rows of 0.9 million products over
// 2^22 columns takes 2.24 ms so, 0.99 with 32 workgroups a row; of 300 rows of 150
// thousand products 1.01, 0.70 with 8 (0.73 with 4); of 2000 rows 1.52 either way.
constexpr int EMIT_WG = 128;
constexpr u32 EMIT_PART = 2048, EMIT_MIN_GRID = 2048;
__global__ __launch_bounds__(EMIT_WG) void k_bitmap_emit(const uint4 *__restrict__ store, u32 nch,
                                                         const u64 *__restrict__ gpre, const u32 *__restrict__ list,
                                                         const u32 *__restrict__ perm, const u64 *__restrict__ off,
                                                         u32 words_per_row, u32 slice_words, u32 parts,
                                                         const u32 *__restrict__ fmt, u32 *__restrict__ cols) {
    constexpr u32 NW = EMIT_WG / 64, ROUNDS = 4, SPAN = ROUNDS * 256;
    __shared__ dev::RankLds stage[NW];
    __shared__ __align__(8) uint8_t tab[2048];
    dev::rank_table(tab);
    __syncthreads();
    const u32 slot = blockIdx.x / parts;  // slots are claimed densely from 0
    const u32 r = perm[list[slot]];
    u32 *out = cols + off[r];
    const u64 lim = off[r + 1] - off[r];
    const u32 wv = dev::wave_id(), l = (u32)dev::lane();
    // slice_words is a multiple of 2^14, and so are words_per_row and its parts
    // or the parts divide a slice (emit_launch), so wpw and every slice boundary
    // inside it are multiples of 2 * SPAN and of EMIT_CHUNK
    const u32 wpw = words_per_row / (NW * parts);
    const u32 first = (blockIdx.x % parts * NW + wv) * wpw, last = first + wpw;
    const u32 nsl = words_per_row / slice_words;
    const u32 *row = reinterpret_cast<const u32 *>(store) + (u64)slot * words_per_row;
    u64 p = gpre[(u64)slot * nch + first / EMIT_CHUNK] - gpre[(u64)slot * nch];
    // a bitmap batch is ROUNDS rounds of 256 words, lane l holding words
    // 4l .. 4l + 3 of each (16-byte loads); s0 counts words from the row's start
    auto load = [&](u32(&w)[ROUNDS][4], u32 s0) {
#pragma unroll
        for (u32 k = 0; k < ROUNDS; ++k) {
            const uint4 v = *reinterpret_cast<const uint4 *>(row + s0 + k * 256 + 4 * l);
            w[k][0] = v.x;
            w[k][1] = v.y;
            w[k][2] = v.z;
            w[k][3] = v.w;
        }
    };
    auto expand = [&](const u32(&w)[ROUNDS][4], u32 s0) {
#pragma unroll
        for (u32 k = 0; k < ROUNDS; ++k) {
            const u32 i0 = 4 * l;
            const u32 wi[4] = {i0, i0 + 1, i0 + 2, i0 + 3};
            p += dev::emit_round4_ranked(w[k], wi, (s0 + k * 256) * 32u, p, out, lim, &stage[wv], tab);
        }
    };
    // the wave's words one slice at a time
    for (u32 seg = first; seg < last;) {
        const u32 sidx = seg / slice_words, s0w = sidx * slice_words;
        const u32 send = s0w + slice_words < last ? s0w + slice_words : last;
        const u32 f = fmt[(u64)slot * nsl + sidx];
        if (f) {
            // the pairs whose (slice-relative) word index is in [seg, send)
            const uint2 *pairs = reinterpret_cast<const uint2 *>(row + (u64)s0w);
            const u32 npairs = f - 1u;
            auto lower = [&](u32 key) {
                u32 lo = 0, hi = npairs;
                while (lo < hi) {
                    const u32 mid = (lo + hi) / 2;
                    if (pairs[mid].x < key) lo = mid + 1;
                    else hi = mid;
                }
                return lo;
            };
            const u32 pa = seg == s0w ? 0u : lower(seg - s0w);
            const u32 pb = send == s0w + slice_words ? npairs : lower(send - s0w);
            for (u32 k0 = pa; k0 < pb; k0 += 256) {
                u32 x[4], wi[4];
#pragma unroll
                for (u32 e = 0; e < 4; ++e) {
                    const u32 k = k0 + 4 * l + e;
                    const uint2 pr = k < pb ? pairs[k] : make_uint2(0u, 0u);
                    x[e] = pr.y;
                    wi[e] = pr.x;  // slice-relative, below 2^15
                }
                p += dev::emit_round4_ranked(x, wi, s0w * 32u, p, out, lim, &stage[wv], tab);
            }
        } else {
            u32 wa[ROUNDS][4], wb[ROUNDS][4];
            load(wa, seg);
            for (u32 s0 = seg; s0 < send; s0 += 2 * SPAN) {
                load(wb, s0 + SPAN);
                expand(wa, s0);
                if (s0 + 2 * SPAN < send) load(wa, s0 + 2 * SPAN);
                expand(wb, s0 + SPAN);
            }
        }
        seg = send;
    }
}

// Writes kept rows (Store) at their final positions: one wave per row and
// chunk of words, whose place is the row's offset plus the sums of the chunks
// before it.  What bounds it: HBM, the columns written; every store
// instruction is one contiguous run (dev::emit_round4_ranked).
constexpr int ES_WG = 256;
__global__ __launch_bounds__(ES_WG) void k_emit_stored(const u32 *__restrict__ perm, u32 n, Store k,
                                                       const u64 *__restrict__ off, u32 *__restrict__ cols) {
    __shared__ dev::RankLds stage[ES_WG / 64];
    __shared__ __align__(8) uint8_t tab[2048];
    dev::rank_table(tab);
    __syncthreads();
    const u32 l = (u32)dev::lane(), wv = dev::wave_id();
    const u64 item = (u64)blockIdx.x * (ES_WG / 64) + wv;
    const u32 row = (u32)(item / k.nch), c = (u32)(item % k.nch);
    if (row >= n) return;
    const u32 r = perm[row];
    const u32 slot = k.slot_of[r] - 1u;
    const u32 cw = store_chunk(k.win_words), per_slice = k.win_words / cw;  // chunk words, chunks of a slice
    const u32 s = c / per_slice, c0 = s * per_slice;                       // the slice and its first chunk
    const u32 *sums = k.chunks + (u64)slot * k.nch;
    const u32 own = sums[c];
    if (!own) return;  // uniform
    u64 before = 0;
    u32 nz = 0;
    for (u32 q = l; q < c; q += 64) {
        const u32 v = sums[q];
        before += v >> 12;
        nz += q >= c0 ? v & 0xFFFu : 0u;
    }
    u64 p = dev::wave_sum(before);
    u32 *out = cols + off[r];
    const u64 lim = off[r + 1] - off[r];
    const u32 *slice = reinterpret_cast<const u32 *>(k.words) + (u64)slot * k.row_words + (u64)s * k.win_words;
    const u32 col0 = s * k.win_words * 32u;
    if (k.fmt[(u64)slot * (k.row_words / k.win_words) + s]) {
        const uint2 *pairs = reinterpret_cast<const uint2 *>(slice) + dev::wave_sum(nz);
        const u32 np = own & 0xFFFu;
        for (u32 k0 = 0; k0 < np; k0 += 256) {
            u32 x[4], wi[4];
#pragma unroll
            for (u32 e = 0; e < 4; ++e) {
                const u32 q = k0 + 4 * l + e;
                const uint2 pr = q < np ? pairs[q] : make_uint2(0u, 0u);
                x[e] = pr.y;
                wi[e] = pr.x;
            }
            p += dev::emit_round4_ranked(x, wi, col0, p, out, lim, &stage[wv], tab);
        }
        return;
    }
    const u32 w0 = (c - c0) * cw;
    uint4 v[4];
#pragma unroll
    for (u32 q = 0; q < 4; ++q) {
        const u32 i = q * 256 + 4 * l;
        v[q] = i < cw ? *reinterpret_cast<const uint4 *>(slice + w0 + i) : make_uint4(0, 0, 0, 0);
    }
#pragma unroll
    for (u32 q = 0; q < 4; ++q) {
        const u32 x[4] = {v[q].x, v[q].y, v[q].z, v[q].w};
        const u32 i0 = w0 + q * 256 + 4 * l;
        const u32 wi[4] = {i0, i0 + 1, i0 + 2, i0 + 3};
        p += dev::emit_round4_ranked(x, wi, col0, p, out, lim, &stage[wv], tab);
    }
}

void emit_stored(hipStream_t st, const u32 *perm, u32 n, const Store &keep, const u64 *off, u32 *cols) {
    if (!n) return;
    k_emit_stored<<<div_up((u64)n * keep.nch, ES_WG / 64), ES_WG, 0, st>>>(perm, n, keep, off, cols);
    CLB_LAUNCHED("emit_stored");
}

// Room for `want` bytes of scratch that may be smaller: a share of the memory at
// hand, so that most of it stays for the operands and the output (what the pool
// caches counts as free: it hands that back when an allocation fails).  Not new
// memory where the largest free block nearly does, since HIP takes back and
// gives out again at some 30 ms a GB:
//  * the memory at hand is never twice quite the same, so a block limited by it
//    would be a little larger at every call.  R-MAT 22 planned and run in a loop
//    took another 77 GB of kept bitmaps three times, then handed 249 GB back:
//    2.9 s of one call, 1.5 s of each on average, 0.65 now.
//  * where HIP has not got that much left, a new block costs the pool all it
//    caches: half is enough then.  The first learned R-MAT 22 product, whose 18
//    blocks dump more and more rows, took 5.0 s, 0.45 now.
static u64 scratch_bytes(clb_controls_s *ctl, u64 want, u64 share) {
    size_t free_b = 0, total_b = 0;
    if (hipMemGetInfo(&free_b, &total_b) != hipSuccess) {
        (void)hipGetLastError();
        return 0;
    }
    Pool &pool = pool_for(ctl->device);
    const u64 budget = (free_b + pool.cached_bytes()) / share, have = pool.largest_free();
    const u64 bytes = want < budget ? want : budget;
    if (have >= bytes) return bytes;
    if (bytes > free_b) return have >= bytes / 2 ? have : bytes;
    return bytes < want && have >= bytes - bytes / 8 ? have : bytes;
}

void setup_store(clb_controls_s *ctl, const Setup &s, const BinHost &h, u32 bits, StoreBufs &b) {
    b.keep = Store{};
    if (s.lean) return;
    // with dump_bits_per_chunk set, the numeric pass gathers its rows and dumps
    // the dense ones, as asked
    const u32 knob = ctl->tuning.dump_bits_per_chunk;
    if (knob && knob < 65536u) return;
    u64 products = 0;
    for (u32 q = BIN_BITMAP0; q < NBINS; ++q) products += h.products[q];
    if (products < KEEP_MIN_PRODUCTS) return;
    const u32 win = 1u << bits;
    const u64 nsl = ((u64)s.g.ncols + 32ull * win - 1) / (32ull * win);
    const u64 words = nsl * win;
    // worth it for rows with at least half as many products as words: writing
    // and reading a word costs about what gathering a product does
    u32 lp = 0;
    while ((2ull << lp) < words) ++lp;
    const u32 end = lp <= 13 ? h.off[NBINS] : (lp > 31 ? h.off[BIN_BITMAP0] : h.off[bitmap_bin_below(lp)]);
    u64 slots = end - h.off[BIN_BITMAP0];
    if (!slots) return;
    if (slots * words * 4 > (1ull << 30)) slots = scratch_bytes(ctl, slots * words * 4, 4) / (words * 4);
    if (!slots) return;
    const u64 nch = words / store_chunk(win);
    try {
        b.words.reset(ctl, slots * words / 4);
        b.chunks.reset(ctl, slots * nch);
        b.fmt.reset(ctl, slots * nsl);
        b.slot_of.reset(ctl, s.nrows);
    } catch (const Error &e) {
        if (!no_room(e)) throw;
        b.drop();
        return;  // the numeric pass gathers as usual
    }
    fill_u32(ctl, b.slot_of.ptr, s.nrows, 0u);
    b.keep = Store{b.words.ptr, b.chunks.ptr, b.fmt.ptr, b.slot_of.ptr, (u32)slots, (u32)nch, (u32)words, win};
}

// ---------------------------------------------------------------------------
// Rows of the bitmap range of perm whose size key (capacity or exact size)
// reaches thr: the rows likely to be dumped.
__global__ void k_dump_candidates(const u32 *__restrict__ perm, u32 n, const u32 *__restrict__ key, u32 thr,
                                  u32 *__restrict__ count) {
    const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
    const bool hit = i < n && key[perm[i]] >= thr;
    const unsigned long long m = __ballot(hit);
    if (dev::lane() == 0 && m) atomicAdd(count, (u32)__popcll(m));
}

void setup_dump(clb_controls_s *ctl, const Setup &s, const BinHost &h, DumpBufs &d, Out &o, bool one_pass,
                const u32 *perm, const u32 *key) {
    o.dump = Dump{};
    d.on = false;
    // default: on in the one pass (its in-kernel emission writes a temporary
    // slot that the compaction copies again), off in the numeric pass (which
    // writes the final positions directly)
    const u32 knob = ctl->tuning.dump_bits_per_chunk ? ctl->tuning.dump_bits_per_chunk : (one_pass ? (s.lean ? 1024u : 64u) : 65536u);
    if (s.cfg.bm_bits < 14 || knob >= 65536u) return;
    const u64 nslices = ((u64)s.g.ncols + (32ull << s.cfg.bm_bits) - 1) / (32ull << s.cfg.bm_bits);
    d.nbm = h.off[NBINS] - h.off[BIN_BITMAP0];
    // a dumped row keeps every slice: nslices windows of 2^bm_bits words
    if (d.nbm == 0 || (nslices << s.cfg.bm_bits) > (1ull << 26)) return;
    d.words = (u32)(nslices << s.cfg.bm_bits);
    d.slice_words = 1u << s.cfg.bm_bits;
    d.nch = d.words / EMIT_CHUNK;
    const u32 dense_min = ((1u << s.cfg.bm_bits) / 1024u) * knob;
    // slots for the rows likely to be dumped: those whose size key reaches a
    // quarter of the dense threshold over all slices, plus a margin for rows
    // the one pass dumps because they outgrow their capacity
    u32 slots = d.nbm;
    if (key && perm) {
        DevArray<u32> cnt(ctl, 1);
        fill_u32(ctl, cnt.ptr, 1, 0u);
        const u64 thr = (u64)dense_min * nslices / 4;
        k_dump_candidates<<<div_up(d.nbm, 256), 256, 0, ctl->stream>>>(
            perm + h.off[BIN_BITMAP0], d.nbm, key, (u32)(thr < 0xFFFFFFFFull ? thr : 0xFFFFFFFFull), cnt.ptr);
        CLB_LAUNCHED("dump_candidates");
        u32 cand = 0;
        readback(ctl, &cand, cnt.ptr, 4);
        const u64 want = (u64)cand + cand / 8 + 256;
        slots = want < d.nbm ? (u32)want : d.nbm;
    }
    const u64 per_slot = (u64)d.words * 4;
    slots = (u32)(scratch_bytes(ctl, slots * per_slot, 3) / per_slot);
    if (slots == 0) return;
    d.slots = slots;
    d.store.reset(ctl, (u64)slots * d.words / 4);
    d.cnt.reset(ctl, (u64)slots * d.nch);
    d.list.reset(ctl, slots);
    d.count.reset(ctl, 1);
    d.isdense.reset(ctl, s.nrows);
    d.fmt.reset(ctl, (u64)slots * nslices);  // written for every slice of a claimed slot
    fill_u32(ctl, d.cnt.ptr, d.cnt.n, 0);
    fill_u32(ctl, d.count.ptr, 1, 0);
    fill_u32(ctl, d.isdense.ptr, s.nrows, 0);
    // the decision is taken on slice 0's count
    o.dump = Dump{d.store.ptr, d.cnt.ptr, d.list.ptr, d.count.ptr, d.isdense.ptr, dense_min, slots, d.fmt.ptr};
    d.on = true;
}

u32 emit_prepare(clb_controls_s *ctl, DumpBufs &d, DevArray<u64> &gpre, clb_spgemm_stats *st) {
    if (!d.on) return 0;
    u32 count = 0;
    readback(ctl, &count, d.count.ptr, 4);
    if (count > d.slots) count = d.slots;  // claims beyond the last slot were refused
    if (!count) return 0;
    if (d.words % (1u << 14)) raise(RUN_KERNEL_FAILURE, "dumped rows must hold whole 2^14-word windows");
    gpre.reset(ctl, d.cnt.n + 1);
    exclusive_scan_u32_to_u64(ctl, d.cnt.ptr, gpre.ptr, d.cnt.n, gpre.ptr + d.cnt.n);
    if (st) {
        u64 total = 0;
        readback(ctl, &total, gpre.ptr + d.cnt.n, 8);
        st->dense_rows += count;
        st->dense_nnz += total;
    }
    return count;
}

void emit_launch(hipStream_t es, u32 count, const u32 *perm, const BinHost &h, const DumpBufs &d, const u64 *gpre,
                 const u64 *off, u32 *cols, LaunchTimer *lt, int pass) {
    if (!count) return;
    if (lt) lt->begin(es);
    // few rows: several workgroups to each, until EMIT_MIN_GRID or parts of two
    // rounds for each wave
    u32 parts = 1;
    while (count * parts < EMIT_MIN_GRID && d.words % (2 * parts * EMIT_WG / 64 * EMIT_PART) == 0) parts *= 2;
    k_bitmap_emit<<<count * parts, EMIT_WG, 0, es>>>(d.store.ptr, d.nch, gpre, d.list.ptr, perm + h.off[BIN_BITMAP0],
                                                     off, d.words, d.slice_words, parts, d.fmt.ptr, cols);
    CLB_LAUNCHED("bitmap_emit");
    if (lt) lt->end((int)CLB_KF(pass, CLB_KK_EMIT), es);
}

void emit_dense(clb_controls_s *ctl, const u32 *perm, const BinHost &h, DumpBufs &d, const u64 *off, u32 *cols,
                LaunchTimer *lt, int pass, clb_spgemm_stats *st) {
    DevArray<u64> gpre;  // released after the launch: later work on this stream is ordered after it
    const u32 count = emit_prepare(ctl, d, gpre, st);
    emit_launch(ctl->stream, count, perm, h, d, gpre.ptr, off, cols, lt, pass);
}

BinCfg make_bincfg(const clb_controls_s *ctl, u32 ncols) {
    BinCfg c{};
    c.ncols = ncols;
    c.tiny_max = ctl->tuning.tiny_max_products;
    u32 hb = 0;
    while ((1u << (hb + 1)) <= ctl->tuning.hash_max_slots) ++hb;
    c.hash_max_bits = hb < HASH_MIN_BITS ? HASH_MIN_BITS : (hb > HASH_MAX_BITS ? HASH_MAX_BITS : hb);
    c.bitmap_min = ctl->tuning.bitmap_min_products;
    c.bitmap_ratio = ctl->tuning.bitmap_slot_ratio;
    // Window of a bitmap kernel: the matrix width rounded up to a power of
    // two words, at most 2^15 words (128 KB of LDS, one 1024-thread workgroup
    // per CU); wider matrices are processed in column slices.  The kernels
    // that also write columns use 2^14 words (64 KB, two 512-thread
    // workgroups per CU, so one row's emission overlaps the other's gather)
    // when that costs at most one extra slice, i.e. up to 2^20 columns.  On
    // wider matrices each extra slice re-reads the A row and its B-row
    // pieces; whether the overlap still pays depends on the rows (with
    // dense-row dumps and the ESC bin it does at R-MAT scale 22), so the
    // bitmap_window_bits knob can force the window.
    const u64 words = ((u64)ncols + 31) / 32;
    u32 wb = 6;
    while (wb < 15 && (1ull << wb) < words) ++wb;
    c.sym_bits = wb;
    c.bm_bits = (wb == 15 && words <= (1ull << 15)) ? 14 : wb;
    const u32 forced = ctl->tuning.reserved[CLB_TUNE_BITMAP_WINDOW_BITS];
    if (forced >= 13 && forced <= 15) c.bm_bits = forced < wb ? forced : wb;
    c.multi_slice = (u64)ncols > (32ull << c.bm_bits) ? 1u : 0u;
    c.tables_over_slices = (ctl->tuning.reserved[CLB_TUNE_HASH_WIDE] >> CLB_TUNE_TABLES_OVER_SLICES_BIT) & 1u;
    const u32 em = ctl->tuning.reserved[CLB_TUNE_ESC_MAX_PRODUCTS];
    c.esc_max = em < (1u << ESC_MAX_BITS) ? em : (1u << ESC_MAX_BITS);
    c.esc_only = 0;
    return c;
}

// Slices of a bitmap row and entries of the split table over B's row ids.
static u64 split_slices(const Setup &s) {
    const u64 span = 32ull << s.cfg.bm_bits;
    return ((u64)s.b.ncols + span - 1) / span;
}
static u64 split_entries(const Setup &s) {
    const u64 nsl = split_slices(s);
    return nsl > 1 ? (u64)s.mapn * (nsl + 1) : 0;
}

// From here on the row kernels run over the filtered A (prepare left what of A
// has a B row).
static void filter_a(clb_controls_s *ctl, Setup &s) {
    const u32 tiles = (u32)(s.foffs.n - 1), grid = tiles + div_up((u64)s.nrows + 1, 256);
    exclusive_scan_u32(ctl, s.foffs.ptr, s.foffs.ptr, tiles, s.foffs.ptr + tiles);
    s.f_rpt.reset(ctl, (u64)s.nrows + 1);
    s.f_cols.reset(ctl, s.a_nnz);  // how many stay only the device knows
    auto run = [&](auto tile) {
        k_filter<decltype(tile)::value><<<grid, 256, 0, ctl->stream>>>(s.g, s.nrows, tiles, s.fmask.ptr, s.foffs.ptr,
                                                                       s.bidx.ptr, s.f_rpt.ptr, s.f_cols.ptr);
    };
    if (s.ftile == rstat_tile<true>()) run(std::integral_constant<u32, rstat_tile<true>()>{});
    else run(std::integral_constant<u32, rstat_tile<false>()>{});
    CLB_LAUNCHED("filter");
    s.filtered = true;
    s.g.a_rpt = s.f_rpt.ptr - s.row0;  // by A's stored rows, as a_all
    s.g.a_cols = s.f_cols.ptr;
    s.g.brange = s.crange.ptr;
    s.g.bpres = nullptr;
    s.g.mapn = s.mapn = s.b.nzr;
}

// The per-slice split table of B (Mats::splits) for bitmap rows over
// several column windows: built on the first pass that has bitmap rows.
void ensure_splits(clb_controls_s *ctl, Setup &s, const BinHost &h) {
    if (s.g.splits || h.off[NBINS] == h.off[BIN_BITMAP0]) return;
    const clb_dcsr &b = s.b;
    const u64 span = 32ull << s.cfg.bm_bits, nsl = split_slices(s);
    if (nsl > 1 && s.fmask.ptr && !s.filtered) filter_a(ctl, s);
    if (nsl <= 1 || !b.nzr || (u64)s.mapn * (nsl + 1) >= (1ull << 32)) return;
    // zero for the rows B does not store (an empty part in every slice), so
    // the gather reads it without looking the row up in brange
    s.splits.reset(ctl, (u64)s.mapn * (nsl + 1));
    if (!s.filtered) fill_u32(ctl, s.splits.ptr, s.splits.n, 0u);
    k_slice_splits<<<div_up((u64)b.nzr * (nsl + 1), 256), 256, 0, ctl->stream>>>(
        u32p(b.rpt), s.filtered ? nullptr : u32p(b.rows), u32p(b.cols), b.nzr, s.mapn, (u32)nsl, span, s.splits.ptr);
    CLB_LAUNCHED("slice_splits");
    s.g.splits = s.splits.ptr;
    s.g.nsl = (u32)nsl;
}

// Packs B for the bitmap kernels when their rows will read it often enough.
void ensure_packed(clb_controls_s *ctl, Setup &s, const BinHost &h) {
    if (s.lean || s.g.b_packs || s.pack_tried || s.g.combine || ctl->tuning.bitmap_persistent) return;
    u64 products = 0;
    for (u32 b = BIN_BITMAP0; b < NBINS; ++b) products += h.products[b];
    const clb_dcsr &b = s.b;
    if (!b.nzr || !b.nnz || !pack_pays(products, b.nnz)) return;
    s.pack_tried = true;
    // a pack's group is known modulo 2^20 columns: wider matrices need slices
    if (b.ncols > (1u << 20) && !s.g.splits) return;
    const u32 tiles = div_up(b.nnz, EX_TILE);
    DevArray<u32> first(ctl, tiles), offs(ctl, (u64)tiles + 1);
    k_tile_rows<EX_TILE><<<div_up(b.nzr, EX_WG), EX_WG, 0, ctl->stream>>>(u32p(b.rpt), 0, b.nzr, 0, b.nnz, first.ptr);
    CLB_LAUNCHED("tile_rows");
    k_pack_count<<<tiles, EX_WG, 0, ctl->stream>>>(u32p(b.rpt), u32p(b.cols), b.nzr, b.nnz, first.ptr, offs.ptr);
    CLB_LAUNCHED("pack_count");
    exclusive_scan_u32(ctl, offs.ptr, offs.ptr, tiles, offs.ptr + tiles);
    u32 npacks = 0;
    readback(ctl, &npacks, offs.ptr + tiles, 4);
    if ((u64)npacks * 100 > (u64)b.nnz * PACK_MAX_PCT) return;
    s.packs.reset(ctl, npacks);
    DevArray<u32> pfirst(ctl, s.g.splits ? npacks : 0);
    s.prange.reset(ctl, s.mapn);
    DevArray<u32> prpt(ctl, (u64)b.nzr + 1);
    k_pack_place<<<tiles, EX_WG, 0, ctl->stream>>>(u32p(b.rpt), u32p(b.cols), b.nzr, b.nnz, first.ptr, offs.ptr,
                                                   prpt.ptr, s.packs.ptr, pfirst.ptr);
    CLB_LAUNCHED("pack_place");
    if (!s.g.bpres && !s.filtered) fill_u64(ctl, reinterpret_cast<u64 *>(s.prange.ptr), s.mapn, 0ull);
    const u32 *rows = s.filtered ? nullptr : u32p(b.rows);
    k_brange_set<<<div_up(b.nzr, 256), 256, 0, ctl->stream>>>(prpt.ptr, rows, b.nzr, s.mapn, s.prange.ptr, nullptr,
                                                              nullptr, nullptr);
    CLB_LAUNCHED("brange_set");
    if (s.g.splits) {
        // (the split table may be a plan's: s.splits is then empty)
        s.psplits.reset(ctl, (u64)s.mapn * (s.g.nsl + 1));
        if (!s.filtered) fill_u32(ctl, s.psplits.ptr, s.psplits.n, 0u);
        k_pack_splits<<<div_up(b.nzr, 256), 256, 0, ctl->stream>>>(prpt.ptr, rows, pfirst.ptr, s.g.splits, b.nzr,
                                                                    s.mapn, s.g.nsl, s.psplits.ptr);
        CLB_LAUNCHED("pack_splits");
    }
    s.g.b_packs = s.packs.ptr;
    s.g.prange = s.prange.ptr;
    s.g.psplits = s.g.splits ? s.psplits.ptr : nullptr;
}

void drop_packed(Setup &s) {
    s.packs.free_();
    s.prange.free_();
    s.psplits.free_();
    s.g.b_packs = nullptr;
    s.g.prange = nullptr;
    s.g.psplits = nullptr;
    s.pack_tried = true;
}

void prepare(clb_controls_s *ctl, const clb_dcsr &a, const clb_dcsr &b, u32 row_begin, u32 nrows, Setup &s,
             bool stats, const Setup *shared, const RowFeat *feat) {
    s.nrows = nrows;
    s.row0 = row_begin;
    if (shared) {
        // a plan's block: B's row map and split table were built once
        s.mapn = shared->mapn;
        s.pack_tried = shared->pack_tried;
        s.filtered = shared->filtered;
        s.lean = shared->lean;
        s.g = shared->g;
        s.cfg = shared->cfg;
        s.b = shared->b;
    } else {
        s.mapn = b.nrows;
        s.brange.reset(ctl, s.mapn ? s.mapn : 1);
        // hypersparse B (under one stored row in 16): a presence bit per row id
        // instead of clearing the whole row map
        const bool sparse_map = (u64)b.nzr * 16 < s.mapn;
        if (sparse_map) s.bpres.reset(ctl, ((u64)s.mapn + 31) / 32);
        s.g.bpres = sparse_map ? s.bpres.ptr : nullptr;
        s.g.a_all = s.g.a_rpt = u32p(a.rpt);
        s.g.a_rows = u32p(a.rows);
        s.g.a_cols = u32p(a.cols);
        s.g.brange = s.brange.ptr;
        s.g.b_cols = u32p(b.cols);
        s.g.mapn = s.mapn;
        s.g.ncols = b.ncols;
        s.g.emit = ctl->tuning.emit_lane_bits_min;
        const u32 sb = ctl->tuning.reserved[CLB_TUNE_EMIT_SPARSE_BITS];
        s.g.sparse_bits = sb ? sb : 256u;
        s.g.combine = ctl->tuning.reserved[CLB_TUNE_GATHER_COMBINE];
        s.cfg = make_bincfg(ctl, b.ncols);
        s.g.splits = nullptr;
        s.g.b_packs = nullptr;
        s.g.prange = nullptr;
        s.g.psplits = nullptr;
        s.pack_tried = false;
        s.filtered = false;
        s.a_nnz = a.nnz;
        s.g.nsl = 0;
        s.g.split_bits = s.cfg.bm_bits;
        s.b = b;  // the split table is built by ensure_splits, once bitmap rows exist
    }
    s.g.row0 = row_begin;
    s.ctr.reset(ctl, 4);
    s.scal.reset(ctl, SCALARS);  // [1] nnz total, [2] nzr total, [3] overflow flag, ...
    if (stats) {
        s.prod.reset(ctl, nrows);
        s.P = s.prod.ptr;
    }
    const bool filter = !shared && !s.lean && stats && s.bpres.ptr && b.nzr && split_entries(s) >= FILTER_MIN_ENTRIES;
    const u64 nmap = shared || s.bpres.ptr ? 0 : s.mapn, nbits = shared ? 0 : s.bpres.n;
    u64 most = nmap > nbits ? nmap : nbits;
    if (stats && nrows > most) most = nrows;
    const u32 cap = ctl->cu_count * 16, grid = div_up(most ? most : 1, 256);
    k_init<<<grid < cap ? grid : cap, 256, 0, ctl->stream>>>(reinterpret_cast<u64 *>(s.brange.ptr), nmap, s.bpres.ptr,
                                                             nbits, s.scal.ptr, SCALARS, stats ? s.prod.ptr : nullptr,
                                                             nrows, feat ? *feat : RowFeat{});
    CLB_LAUNCHED("init");
    if (!shared && b.nzr) {
        if (filter) {
            s.bidx.reset(ctl, s.mapn);
            s.crange.reset(ctl, b.nzr);
        }
        k_brange_set<<<div_up(b.nzr, 256), 256, 0, ctl->stream>>>(u32p(b.rpt), u32p(b.rows), b.nzr, s.mapn,
                                                                   s.brange.ptr, s.bpres.ptr, s.bidx.ptr, s.crange.ptr);
        CLB_LAUNCHED("brange_set");
    }
    if (!stats) return;
    // count_workload (count_workload.cl:30-53): products of each A row
    auto run = [&](auto feat_c) {
        constexpr bool FEAT = decltype(feat_c)::value;
        const u32 tiles = div_up(a.nnz, rstat_tile<FEAT>());
        DevArray<u32> first(ctl, tiles);
        k_tile_rows<rstat_tile<FEAT>()><<<div_up(nrows, EX_WG), EX_WG, 0, ctl->stream>>>(
            s.g.a_rpt, row_begin, row_begin + nrows, 0, 0, first.ptr);
        CLB_LAUNCHED("tile_rows");
        if (filter) {
            s.ftile = rstat_tile<FEAT>();
            s.fmask.reset(ctl, (u64)tiles * (s.ftile / 32));
            s.foffs.reset(ctl, (u64)tiles + 1);
        }
        k_row_stats<FEAT><<<tiles, RSTAT_WG, 0, ctl->stream>>>(s.g, nrows, first.ptr, s.prod.ptr,
                                                               feat ? *feat : RowFeat{}, s.fmask.ptr, s.foffs.ptr);
        CLB_LAUNCHED("count_workload");
    };
    if (feat) run(std::true_type{});
    else run(std::false_type{});
}

void bin_rows(clb_controls_s *ctl, const Setup &s, const u32 *key, u32 *nnz_row_zero, DevArray<u32> &perm,
              const u32 *slot_of) {
    static_assert(sizeof(BinTotals) <= PINNED_BYTES, "pinned staging");
    perm.reset(ctl, s.nrows ? s.nrows : 1);
    // stretches of at least four rows per thread
    u32 grid = div_up(s.nrows ? s.nrows : 1, 4 * BIN_WG);
    if (grid > BIN_GRID) grid = BIN_GRID;
    const u32 per = div_up(s.nrows, grid);
    DevArray<BinPart> parts(ctl, grid);
    k_bin_count<<<grid, BIN_WG, 0, ctl->stream>>>(s.g, s.P, key, s.nrows, per, s.cfg, parts.ptr, nnz_row_zero,
                                                  slot_of);
    CLB_LAUNCHED("bin_count");
    k_bin_place<<<grid, BIN_WG, 0, ctl->stream>>>(s.P, key, s.nrows, per, s.cfg, parts.ptr, perm.ptr, slot_of,
                                                  s.scal.ptr, reinterpret_cast<BinTotals *>(ctl->pinned));
    CLB_LAUNCHED("bin_place");
}

void read_bins(clb_controls_s *ctl, Setup &s, BinHost &h) {
    sync(ctl);
    BinTotals t;
    std::memcpy(&t, ctl->pinned, sizeof(t));
    h.off[0] = 0;
    h.total = 0;
    s.bin_work = 0;
    for (u32 b = 0; b < NBINS; ++b) {
        h.off[b + 1] = h.off[b] + t.rows[b];
        h.products[b] = t.sums[b];
        h.a_nnz[b] = t.sums[NBINS + b];
        h.out_nnz[b] = t.sums[2 * NBINS + b];
        s.bin_products[b] = t.sums[b];
        h.total += t.sums[b];
        s.bin_work += t.sums[b] + 4 * t.sums[NBINS + b];
    }
    std::memcpy(h.scal, t.scal, sizeof(h.scal));
}

// Sums nnz_row over the rows of bins 1..NBINS-1 (perm[off[1] .. off[NBINS]));
// the EMPTY bin's range of perm is never written by the scatter.
__global__ __launch_bounds__(256) void k_sum_by_bin(const u32 *__restrict__ perm, const u32 *__restrict__ off,
                                                    u32 nrows, const u32 *__restrict__ nnz_row,
                                                    u64 *__restrict__ sums) {
    __shared__ unsigned long long hs[NBINS];
    __shared__ u32 so[NBINS + 1];
    if (threadIdx.x < NBINS) hs[threadIdx.x] = 0;
    if (threadIdx.x <= NBINS) so[threadIdx.x] = off[threadIdx.x];
    __syncthreads();
    const u32 i = so[1] + blockIdx.x * 256 + threadIdx.x;
    if (i < so[NBINS]) {
        u32 b = 1;
        while (b + 1 < NBINS && so[b + 1] <= i) ++b;
        const u32 row = perm[i];
        const u32 v = row < nrows ? nnz_row[row] : 0u;
        if (v != FAILED) atomicAdd(&hs[b], (unsigned long long)v);
    }
    __syncthreads();
    if (threadIdx.x < NBINS && hs[threadIdx.x])
        atomicAdd(reinterpret_cast<unsigned long long *>(&sums[threadIdx.x]), hs[threadIdx.x]);
}

void sum_by_bin(clb_controls_s *ctl, const u32 *perm, const BinHost &h, u32 nrows, const u32 *nnz_row,
                u64 out[NBINS]) {
    const u32 n = h.off[NBINS] - h.off[1];
    DevArray<u32> off(ctl, NBINS + 1);
    DevArray<u64> sums(ctl, NBINS);
    CLB_HIP(hipMemcpyAsync(off.ptr, h.off, 4 * (NBINS + 1), hipMemcpyHostToDevice, ctl->stream), WRITE_BUFFER_ERROR);
    fill_u64(ctl, sums.ptr, NBINS, 0ull);
    if (n) {
        k_sum_by_bin<<<div_up(n, 256), 256, 0, ctl->stream>>>(perm, off.ptr, nrows, nnz_row, sums.ptr);
        CLB_LAUNCHED("sum_by_bin");
    }
    readback(ctl, out, sums.ptr, NBINS * 8);
}

void LaunchTimer::begin(hipStream_t st) {
    if (!on) return;
    CLB_HIP(hipEventCreate(&pending), EVENT_WAITING_ERROR);
    CLB_HIP(hipEventRecord(pending, st), EVENT_WAITING_ERROR);
}

void LaunchTimer::end(int family, hipStream_t st) {
    if (!on) return;
    hipEvent_t e;
    CLB_HIP(hipEventCreate(&e), EVENT_WAITING_ERROR);
    CLB_HIP(hipEventRecord(e, st), EVENT_WAITING_ERROR);
    recs.push_back({family, pending, e});
    pending = nullptr;
}

void LaunchTimer::collect(clb_spgemm_stats &st) {
    for (auto &r : recs) {
        float m = 0;
        if (hipEventElapsedTime(&m, r.a, r.b) == hipSuccess) {
            st.ms_kernel[r.family] += m;
            st.launches[r.family] += 1;
        }
    }
}

LaunchTimer::~LaunchTimer() {
    for (auto &r : recs) {
        (void)hipEventDestroy(r.a);
        (void)hipEventDestroy(r.b);
    }
    if (pending) (void)hipEventDestroy(pending);
}

void join_deferred(clb_controls_s *ctl, const hipEvent_t *defer) {
    for (int k = 0; k < clb_controls_s::NSIDE; ++k)
        CLB_HIP(hipStreamWaitEvent(ctl->stream, defer[k], 0), EVENT_WAITING_ERROR);
}

// Launch the per-bin kernels of one pass.  off[b]..off[b+1] is bin b's range
// of perm.  mode SYM writes nnz_row, NUM the columns, ONE both.
void launch_bins(clb_controls_s *ctl, const Setup &s, const u32 *perm, const u32 off[NBINS + 1], int mode,
                 const Out &o, LaunchTimer *lt, int family, hipEvent_t *defer, bool one_stream, bool open) {
    constexpr int NS = clb_controls_s::NSIDE;
    // A fork and a join cost about 50 us of a small product (186 us with both
    // passes on three side streams, 102 on the controls' stream alone): a single
    // kernel, and kernels over little work, run on the controls' stream one
    // after the other, and only streams that get a kernel are waited for.
    // Otherwise the longest kernels have slots of their own, kept rows slot 0,
    // bitmap rows and heavy bitmap rows 0 and 1, and the table kernels alternate
    // over the rest.  Slot 0 is the controls' stream itself, unless the caller
    // has other work for it meanwhile: there the heavy rows start first, as
    // they end last (behind the other bitmap rows R-MAT 2^16 took 979 us, before
    // them 859); of two overlapping blocks they take slot 1, not behind the
    // previous block's bitmap rows.
    u32 kernels = 0;
    for (u32 b = BIN_TINY; b < BIN_BITMAP0; ++b)
        kernels += off[b + 1] != off[b] && (b != BIN_STORED || (mode == NUM && o.keep.words));
    kernels += off[NBINS] != off[BIN_BITMAP0] && !s.cfg.esc_only ? 2 : 0;
    if (!open && s.bin_work <= ONE_STREAM_WORK) one_stream = true;
    const bool main0 = !defer && !open;
    if (main0 && kernels <= 1) one_stream = true;
    if (!one_stream) CLB_HIP(hipEventRecord(ctl->ev_fork, ctl->stream), EVENT_WAITING_ERROR);
    bool forked[NS] = {}, taken[NS] = {};
    auto on = [&](int w) {
        if (one_stream || (main0 && w == 0)) return ctl->stream;
        if (!forked[w]) CLB_HIP(hipStreamWaitEvent(ctl->side[w], ctl->ev_fork, 0), EVENT_WAITING_ERROR);
        forked[w] = true;
        return ctl->side[w];
    };
    int k = NS - 1;
    auto next = [&]() {
        if (one_stream) return ctl->stream;
        do k = (k + 1) % NS;
        while (taken[k] && k != NS - 1);
        return on(k);
    };
    LaunchTimer dummy;
    LaunchTimer &t = lt ? *lt : dummy;
    // family = the pass (CLB_KP_*); < 0 picks symbolic / numeric from the mode
    const int pass = family >= 0 ? family : (mode == SYM ? (int)CLB_KP_SYMBOLIC : (int)CLB_KP_NUMERIC);
    auto fam = [&](int kind) { return (int)CLB_KF(pass, kind); };
#define DISPATCH3(KERNEL, GRID, WG, ST, ...)                                                       \
    do {                                                                                          \
        if (mode == SYM) KERNEL<__VA_ARGS__, SYM><<<GRID, WG, 0, ST>>>(s.g, pp, o);               \
        else if (mode == NUM) KERNEL<__VA_ARGS__, NUM><<<GRID, WG, 0, ST>>>(s.g, pp, o);          \
        else KERNEL<__VA_ARGS__, ONE><<<GRID, WG, 0, ST>>>(s.g, pp, o);                           \
    } while (0)
    // BITMAP (all classes in one launch, largest rows first; the ESC SpGEMM
    // sorts these rows in global memory instead).  The longest kernel of the
    // pass goes first and on a side stream of its own, so that it never
    // queues behind a table kernel; the table kernels fill the CUs around it.
    if (!s.cfg.esc_only) {
        const u32 ns = off[BIN_STORED + 1] - off[BIN_STORED];
        if (ns && mode == NUM && o.keep.words) {
            hipStream_t st = on(0);
            taken[0] = true;
            t.begin(st);
            emit_stored(st, perm + off[BIN_STORED], ns, o.keep, o.off, o.cols);
            t.end(fam(CLB_KK_BITMAP), st);
        }
        const u32 n = off[NBINS] - off[BIN_BITMAP0];
        if (n) {
            const u32 *pp = perm + off[BIN_BITMAP0];
            const u32 bits = mode == SYM ? s.cfg.sym_bits : s.cfg.bm_bits;
            // rows that a workgroup of the usual size would work on for longer
            // than half of what an even share of the pass takes run with the
            // widest workgroup, beside the others (R-MAT 2^16, symbolic: its
            // CUs were busy for 228 of 583 us, waiting for rows of up to 645
            // thousand products on 256 threads; 421 us with the 493 largest
            // rows on 1024); the widest have no word-combining gather, which is
            // asked for by a knob
            const u32 slots = ctl->cu_count * bitmap_resident(bits);
            u64 products = 0;
            for (u32 b = BIN_BITMAP0; b < NBINS; ++b) products += s.bin_products[b];
            u32 lp = 14;
            while (lp < 32 && (1ull << lp) * 2 * slots < products) ++lp;
            u32 heavy = 0;
            if (bitmap_wide(bits) > bitmap_wg(bits) && !ctl->tuning.bitmap_persistent && !s.g.combine && lp < 32)
                heavy = off[bitmap_bin_below(lp)] - off[BIN_BITMAP0];
            for (int wide = 1; wide >= 0; --wide) {
                const u32 r0 = wide ? 0 : heavy, nr = wide ? heavy : n - heavy;
                if (!nr) continue;
                const int slot = (ns && mode == NUM) || (wide != 0) != main0 ? 1 : 0;
                hipStream_t st = on(slot);
                taken[slot] = true;
                t.begin(st);
                if (mode == SYM) launch_bitmap_sym(ctl, st, s, pp, r0, nr, bits, wide != 0, o);
                else if (mode == NUM) launch_bitmap_num(ctl, st, s, pp, r0, nr, bits, wide != 0, o);
                else launch_bitmap_one(ctl, st, s, pp, r0, nr, bits, wide != 0, o);
                CLB_LAUNCHED("bitmap");
                t.end(fam(2), st);
            }
        }
    }
    // TINY
    {
        const u32 n = off[BIN_TINY + 1] - off[BIN_TINY];
        if (n) {
            hipStream_t st = next();
            const u32 *pp = perm + off[BIN_TINY];
            t.begin(st);
            if (mode == SYM) k_tiny<4, SYM><<<div_up(n, 4), 256, 0, st>>>(s.g, pp, n, o);
            else if (mode == NUM) k_tiny<4, NUM><<<div_up(n, 4), 256, 0, st>>>(s.g, pp, n, o);
            else k_tiny<4, ONE><<<div_up(n, 4), 256, 0, st>>>(s.g, pp, n, o);
            CLB_LAUNCHED("tiny");
            t.end(fam(0), st);
        }
    }
    // HASH
    for (u32 bits = HASH_MIN_BITS; bits <= HASH_MAX_BITS; ++bits) {
        const u32 b = BIN_HASH0 + (bits - HASH_MIN_BITS);
        const u32 n = off[b + 1] - off[b];
        if (!n) continue;
        const u32 *pp = perm + off[b];
        hipStream_t st = next();
        t.begin(st);
        // workgroup shape per table size: the default, or twice the threads
        // when the table size's bit of the hash_wide knob is set
        const bool wide = (ctl->tuning.reserved[CLB_TUNE_HASH_WIDE] >> (bits - HASH_MIN_BITS)) & 1u;
        switch (bits * 2 + (wide ? 1 : 0)) {
            case 14: DISPATCH3(k_hash, n, 64, st, 7, 64); break;
            case 15: DISPATCH3(k_hash, n, 128, st, 7, 128); break;
            case 16: DISPATCH3(k_hash, n, 64, st, 8, 64); break;
            case 17: DISPATCH3(k_hash, n, 128, st, 8, 128); break;
            case 18: DISPATCH3(k_hash, n, 64, st, 9, 64); break;
            case 19: DISPATCH3(k_hash, n, 128, st, 9, 128); break;
            case 20: DISPATCH3(k_hash, n, 128, st, 10, 128); break;
            case 21: DISPATCH3(k_hash, n, 256, st, 10, 256); break;
            case 22: DISPATCH3(k_hash, n, 128, st, 11, 128); break;
            case 23: DISPATCH3(k_hash, n, 256, st, 11, 256); break;
            case 24: DISPATCH3(k_hash, n, 256, st, 12, 256); break;
            case 25: DISPATCH3(k_hash, n, 512, st, 12, 512); break;
            case 26: DISPATCH3(k_hash, n, 512, st, 13, 512); break;
            case 27: DISPATCH3(k_hash, n, 1024, st, 13, 1024); break;
            case 28:
            case 29: DISPATCH3(k_hash, n, 1024, st, 14, 1024); break;
        }
        CLB_LAUNCHED("hash");
        t.end(fam(1), st);
    }
    // ESC (rows of at most 2^11 / 2^12 / 2^13 products)
    for (u32 bits = ESC_MIN_BITS; bits <= ESC_MAX_BITS; ++bits) {
        const u32 b = BIN_ESC0 + (bits - ESC_MIN_BITS);
        const u32 n = off[b + 1] - off[b];
        if (!n) continue;
        const u32 *pp = perm + off[b];
        hipStream_t st = next();
        t.begin(st);
        switch (bits) {
            case 11: DISPATCH3(k_esc, n, 256, st, 11, 256); break;
            case 12: DISPATCH3(k_esc, n, 512, st, 12, 512); break;
            case 13: DISPATCH3(k_esc, n, 1024, st, 13, 1024); break;
        }
        CLB_LAUNCHED("esc");
        t.end(fam(1), st);
    }
#undef DISPATCH3
    if (open) return;
    if (defer) {
        for (int j = 0; j < NS; ++j)
            CLB_HIP(hipEventRecord(defer[j], forked[j] ? ctl->side[j] : ctl->stream), EVENT_WAITING_ERROR);
        return;
    }
    for (int j = 0; j < NS; ++j) {
        if (!forked[j]) continue;
        CLB_HIP(hipEventRecord(ctl->ev_join[j], ctl->side[j]), EVENT_WAITING_ERROR);
        CLB_HIP(hipStreamWaitEvent(ctl->stream, ctl->ev_join[j], 0), EVENT_WAITING_ERROR);
    }
}

struct Timer {
    bool on;
    hipStream_t st;
    std::vector<hipEvent_t> ev;
    Timer(bool enable, hipStream_t s) : on(enable), st(s) {}
    void mark() {
        if (!on) return;
        hipEvent_t e;
        CLB_HIP(hipEventCreate(&e), EVENT_WAITING_ERROR);
        CLB_HIP(hipEventRecord(e, st), EVENT_WAITING_ERROR);
        ev.push_back(e);
    }
    double ms(size_t i, size_t j) const {
        if (!on || j >= ev.size()) return 0;
        float m = 0;
        (void)hipEventElapsedTime(&m, ev[i], ev[j]);
        return m;
    }
    ~Timer() {
        for (auto e : ev) (void)hipEventDestroy(e);
    }
};

void assemble(clb_controls_s *ctl, const Setup &s, const clb_dcsr &a, const u32 *nnz_row, const u64 *off,
              const u32 *pos, u64 nnz, u32 nzr, clb_buffer_s *cols, clb_dcsr &out) {
    out.cols = cols;
    out.rpt = buffer_new(ctl, 4ull * (nzr + 1));
    out.rows = buffer_new(ctl, 4ull * (nzr ? nzr : 1));
    k_set_positions<<<div_up(s.nrows ? s.nrows : 1, 256), 256, 0, ctl->stream>>>(
        nnz_row, off, pos, s.nrows, s.g.a_rows, s.row0, u32p(out.rpt), u32p(out.rows), (u32)nnz, nzr);
    CLB_LAUNCHED("set_positions");
    out.nnz = (u32)nnz;
    out.nzr = nzr;
}

// Offsets and empty-row compaction of the exact row sizes.  Results land in
// s.scal[1] (nnz) and s.scal[2] (nzr).
void scan_sizes(clb_controls_s *ctl, Setup &s, const u32 *nnz_row, DevArray<u64> &off, DevArray<u32> &pos) {
    off.reset(ctl, s.nrows + 1);
    pos.reset(ctl, s.nrows + 1);
    // off[nrows] holds the total too (row r's size is off[r + 1] - off[r])
    const u32 tiles = div_up(s.nrows, SZ_TILE);
    if (tiles <= 1) {
        k_sizes_place<<<1, SZ_WG, 0, ctl->stream>>>(nnz_row, s.nrows, nullptr, off.ptr, pos.ptr, s.scal.ptr);
        CLB_LAUNCHED("sizes");
        return;
    }
    DevArray<SizeSum> sums(ctl, tiles);
    k_sizes_sum<<<tiles, SZ_WG, 0, ctl->stream>>>(nnz_row, s.nrows, sums.ptr);
    CLB_LAUNCHED("sizes_sum");
    k_sizes_scan<<<1, SZ_WG, 0, ctl->stream>>>(sums.ptr, tiles, off.ptr + s.nrows, s.scal.ptr);
    CLB_LAUNCHED("sizes_scan");
    k_sizes_place<<<tiles, SZ_WG, 0, ctl->stream>>>(nnz_row, s.nrows, sums.ptr, off.ptr, pos.ptr, s.scal.ptr);
    CLB_LAUNCHED("sizes_place");
}

void spgemm_plain(clb_controls_s *ctl, const clb_dcsr &a, const clb_dcsr &b, u32 row_begin, u32 row_end,
                  bool timing, clb_dcsr &out, clb_spgemm_stats &st, const PlanRows *pr, bool lean) {
    Timer tm(timing, ctl->stream);
    tm.mark();  // 0
    const u32 nrows = row_end - row_begin;
    Setup s;
    s.lean = lean;
    prepare(ctl, a, b, row_begin, nrows, s, pr == nullptr, pr ? pr->shared : nullptr);
    LaunchTimer lt;
    lt.on = timing;
    st.rows = nrows;
    st.n_bins = NBINS;
    DevArray<u32> nnz_row_own;
    u32 *nnz_row = nullptr;
    StoreBufs store;
    Store keep{};  // bitmaps the symbolic pass kept
    if (pr) {
        keep = pr->keep;
        // planned block: products and exact row sizes come from the plan
        s.P = pr->prod;
        nnz_row = pr->size;
        st.products = pr->products;
        tm.mark();  // 1
        tm.mark();  // 2
    } else {
        DevArray<u32> perm;
        BinHost h1;
        nnz_row_own.reset(ctl, nrows);
        nnz_row = nnz_row_own.ptr;
        bin_rows(ctl, s, nullptr, nnz_row, perm);
        read_bins(ctl, s, h1);
        st.products = h1.total;
        tm.mark();  // 1
        if (h1.total == 0) {
            out.nrows = a.nrows;
            out.ncols = b.ncols;
            return;
        }
        setup_store(ctl, s, h1, s.cfg.sym_bits, store);
        keep = store.keep;
        Out o1{nnz_row, nullptr, nullptr, nullptr, reinterpret_cast<u32 *>(s.scal.ptr + 3), Dump{}, 0, keep};
        ensure_splits(ctl, s, h1);
        ensure_packed(ctl, s, h1);
        launch_bins(ctl, s, perm.ptr, h1.off, SYM, o1, &lt, -1);
        tm.mark();  // 2
    }
    if (st.products == 0) {
        out.nrows = a.nrows;
        out.ncols = b.ncols;
        return;
    }
    DevArray<u64> offs;
    DevArray<u32> pos;
    scan_sizes(ctl, s, nnz_row, offs, pos);
    DevArray<u32> perm2;
    BinHost h2;
    bin_rows(ctl, s, nnz_row, nullptr, perm2, keep.words ? keep.slot_of : nullptr);
    read_bins(ctl, s, h2);
    for (u32 k = 0; k < NBINS; ++k) {
        st.bin_rows[k] = h2.off[k + 1] - h2.off[k];
        st.bin_products[k] = h2.products[k];
        st.bin_a_nnz[k] = h2.a_nnz[k];
        st.bin_out_nnz[k] = h2.out_nnz[k];
    }
    const u64 *sc = h2.scal;  // taken with the bins
    tm.mark();  // 3
    if (sc[3]) raise(RUN_KERNEL_FAILURE, "hash table overflow in the symbolic pass");
    const u64 nnz = sc[1];
    const u32 nzr = static_cast<u32>(sc[2]);
    if (nnz > 0xFFFFFFFFull) {
        std::ostringstream os;
        os << "result has " << nnz << " nonzeros, more than uint32 indices allow; multiply by row blocks";
        raise(INVALID_VALUE, os.str());
    }
    out.nrows = a.nrows;
    out.ncols = b.ncols;
    if (nnz == 0) return;
    clb_buffer_s *cols = buffer_new(ctl, 4ull * nnz);
    try {
        Out o2{nnz_row, offs.ptr, u32p(cols), nullptr, reinterpret_cast<u32 *>(s.scal.ptr + 3), Dump{}, 0, keep};
        DumpBufs dump;
        setup_dump(ctl, s, h2, dump, o2, false, perm2.ptr, nnz_row);
        ensure_splits(ctl, s, h2);
        ensure_packed(ctl, s, h2);
        launch_bins(ctl, s, perm2.ptr, h2.off, NUM, o2, &lt, -1);
        emit_dense(ctl, perm2.ptr, h2, dump, offs.ptr, u32p(cols), &lt, CLB_KP_NUMERIC, timing ? &st : nullptr);
        tm.mark();  // 4
        assemble(ctl, s, a, nnz_row, offs.ptr, pos.ptr, nnz, nzr, cols, out);
        tm.mark();  // 5
        u64 flag = 0;
        readback(ctl, &flag, s.scal.ptr + 3, 8);
        if (flag) raise(RUN_KERNEL_FAILURE, "numeric pass disagreed with the symbolic row sizes");
    } catch (...) {
        settle(ctl);
        if (!out.cols) buffer_release(cols);  // else out's
        clb_dcsr_release(&out);
        throw;
    }
    st.nnz = nnz;
    st.nzr = nzr;
    lt.collect(st);
    if (timing) {
        st.ms_setup = tm.ms(0, 1);
        st.ms_symbolic = tm.ms(1, 2);
        st.ms_numeric = tm.ms(3, 4);
        st.ms_assemble = tm.ms(2, 3) + tm.ms(4, 5);
        st.ms_total = tm.ms(0, 5);
    }
}

void plan_sizes_plain(clb_controls_s *ctl, Setup &s, u32 *size, StoreBufs &store) {
    // the symbolic pass of spgemm_plain over every stored row of A
    DevArray<u32> perm;
    BinHost h;
    bin_rows(ctl, s, nullptr, size, perm);
    read_bins(ctl, s, h);
    setup_store(ctl, s, h, s.cfg.sym_bits, store);
    Out o{size, nullptr, nullptr, nullptr, reinterpret_cast<u32 *>(s.scal.ptr + 3), Dump{}, 0, store.keep};
    ensure_splits(ctl, s, h);
    ensure_packed(ctl, s, h);
    launch_bins(ctl, s, perm.ptr, h.off, SYM, o, nullptr, -1);
    u64 flag = 0;
    readback(ctl, &flag, s.scal.ptr + 3, 8);
    if (flag) raise(RUN_KERNEL_FAILURE, "hash table overflow in the symbolic pass");
}

void check_dims(const clb_dcsr &a, const clb_dcsr &b) {
    // hash.cpp:56-61
    if (a.ncols != b.nrows) {
        std::ostringstream s;
        s << "Invalid input matrix size! a : " << a.nrows << " x " << a.ncols << ", b: " << b.nrows << " x "
          << b.ncols;
        raise(INVALID_ARGUMENT, s.str());
    }
}

void spgemm_dispatch(clb_controls_s *ctl, const clb_dcsr &a, const clb_dcsr &b, const clb_spgemm_opts &o,
                     clb_dcsr &out, clb_spgemm_stats &st) {
    std::memset(&st, 0, sizeof(st));
    check_dims(a, b);
    clb_dcsr r{};
    r.nrows = a.nrows;
    r.ncols = b.ncols;
    u32 rb = o.row_begin, re = o.row_end ? o.row_end : a.nzr;
    if (re > a.nzr || rb > re) raise(INVALID_ARGUMENT, "row block outside the stored rows of A");
    // hash.cpp:64-67: an empty operand gives an empty result
    if (a.nnz == 0 || b.nnz == 0 || rb == re) {
        out = r;
        return;
    }
    auto t0 = std::chrono::steady_clock::now();
    const bool one_pass = o.mode == CLB_SPGEMM_LEARNED || o.mode == CLB_SPGEMM_BOUND;
    if (!one_pass && o.mode != CLB_SPGEMM_PLAIN) raise(INVALID_ARGUMENT, "unknown SpGEMM mode");
    with_room(ctl, [&](bool lean) {
        std::memset(&st, 0, sizeof(st));
        if (one_pass)
            spgemm_learned(ctl, a, b, rb, re, o.timing != 0, r, st, o.mode == CLB_SPGEMM_BOUND, nullptr, lean);
        else
            spgemm_plain(ctl, a, b, rb, re, o.timing != 0, r, st, nullptr, lean);
    });
    if (!o.timing)
        st.ms_total = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    ctl->last = st;
    out = r;
}

}  // namespace spg
}  // namespace clb

using namespace clb;

extern "C" {

clb_status clb_dcsr_spgemm_hash(clb_controls ctl, const clb_dcsr *a, const clb_dcsr *b, clb_dcsr *out) {
    return run_guarded(ctl, [&] {
        clb_spgemm_opts o{};
        o.mode = CLB_SPGEMM_PLAIN;
        clb_spgemm_stats st;
        clb_dcsr r{};
        spg::spgemm_dispatch(ctl, *a, *b, o, r, st);
        *out = r;
    });
}

clb_status clb_dcsr_spgemm(clb_controls ctl, const clb_dcsr *a, const clb_dcsr *b, const clb_spgemm_opts *opts,
                           clb_dcsr *out, clb_spgemm_stats *stats) {
    return run_guarded(ctl, [&] {
        clb_spgemm_opts o{};
        if (opts) o = *opts;
        clb_spgemm_stats st;
        clb_dcsr r{};
        spg::spgemm_dispatch(ctl, *a, *b, o, r, st);
        *out = r;
        if (stats) *stats = st;
    });
}

}  // extern "C"
