// esc.hip -- the expand-sort-compress SpGEMM, dcsr::matrix_multiplication
// (src/dcsr/dcsr_matrix_multiplication.cpp:26-168).
//
// A second GPU SpGEMM that shares no accumulator with the hash path, so the
// two cross-check each other.  The reference sizes every row by its product
// count (count_workload, :388-404; "pre" matrix at the products prefix,
// :279-334), then writes each row's sorted unique columns into its slot with
// a kernel per bin (copy_one_value for one product, heap_merge up to 32,
// bitonic_esc up to 512, merge_large_rows above, :192-275) and compacts
// (create_final_matrix, :97-158).  Here, with the same one-pass structure:
//  * rows of at most 64 products: one wave, register bitonic sort (k_tiny);
//  * up to 2^13 products: one workgroup expands the products into LDS,
//    radix-sorts them there and keeps the first of each run (k_esc);
//  * longer rows: all their products are expanded at once into HBM, a stretch
//    per row, each stretch is radix-sorted by column and deduplicated, instead
//    of the reference's pairwise merges of B rows per row; beside the kernels
//    of the other rows, on their own streams;
//  * exact sizes are scanned and every row is copied to its final place.
#include "radix.hpp"
#include "spgemm.hpp"

namespace clb {
namespace spg {

// Slots of the rows sorted in LDS or in registers: their product count; rows
// sorted in HBM get 0.
__global__ void k_esc_sizes(const u32 *__restrict__ prod, u32 n, u32 lds_max, u32 *__restrict__ tlen,
                            u32 *__restrict__ from_side) {
    const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const u32 P = prod[i];
    tlen[i] = P <= lds_max ? P : 0u;
    from_side[i] = 0;
}

// A tile of a long row: values [start, start + count), one of the `ntiles`
// tiles from `tile0` of its row.
struct EscTile {
    u32 start, count, tile0, ntiles;
};

// First value and first tile of each long row (one workgroup).
constexpr int SEG_WG = 1024;
__global__ __launch_bounds__(SEG_WG) void k_esc_segs(const u32 *__restrict__ perm, u32 n, const u32 *__restrict__ prod,
                                                     uint2 *__restrict__ segs) {
    __shared__ u64 red[SEG_WG / dev::WAVE + 1];
    u64 carry = 0;  // values << 32 | tiles: both below 2^32, no carry between them
    for (u32 i0 = 0; i0 < n; i0 += SEG_WG) {
        const u32 i = i0 + threadIdx.x;
        const u32 P = i < n ? prod[perm[i]] : 0u;
        u64 all;
        const u32 nt = P / RX_TILE + (P % RX_TILE ? 1u : 0u);
        const u64 x = carry + dev::block_excl_scan<u64, SEG_WG>(((u64)P << 32) | nt, red, all);
        if (i < n) segs[i] = make_uint2((u32)(x >> 32), (u32)x);
        carry += all;
    }
    if (threadIdx.x == 0) segs[n] = make_uint2((u32)(carry >> 32), (u32)carry);
}

// Expands the products of long row blockIdx.x into its stretch of vals, slots
// taken by wave-aggregated appends, and describes its tiles.  The longest row
// is its tail, beside the rows sorted in LDS: the whole product of R-MAT 10000
// x 10 takes 388 / 349 / 386 us with 256 / 512 / 1024 threads, of 20000 x 12
// 639 / 597 / 682.
constexpr int EXP_WG = 512;
__global__ __launch_bounds__(EXP_WG) void k_esc_expand(Mats g, const u32 *__restrict__ perm,
                                                       const uint2 *__restrict__ segs, u32 *__restrict__ vals,
                                                       EscTile *__restrict__ tiles) {
    __shared__ __align__(8) u32 big[BIG_WORDS(EXP_WG)];
    __shared__ u32 cnt;
    const u32 r = perm[blockIdx.x];
    const u32 i = g.row0 + r;
    const uint2 s0 = segs[blockIdx.x], s1 = segs[blockIdx.x + 1];
    const u32 nt = s1.y - s0.y;
    for (u32 t = threadIdx.x; t < nt; t += EXP_WG) {
        const u32 a = s0.x + t * RX_TILE;
        tiles[s0.y + t] = EscTile{a, t + 1 < nt ? RX_TILE : s1.x - a, s0.y, nt};
    }
    if (threadIdx.x == 0) cnt = 0;
    __syncthreads();
    u32 *dst = vals + s0.x;
    auto append = [&](u32 col) {
        const unsigned long long m = __ballot(1);
        const u32 leader = (u32)__ffsll(m) - 1u;
        u32 base = 0;
        if ((u32)dev::lane() == leader) base = atomicAdd(&cnt, (u32)__popcll(m));
        base = __shfl(base, (int)leader, dev::WAVE);
        dst[base + dev::lanes_below(m)] = col;
    };
    for_each_product<EXP_WG, 8, BIG_ROW>(g, g.a_rpt[i], g.a_rpt[i + 1], big, append);
}

// The sort of the long rows: columns only, 32 bits a value, since the rows'
// stretches are in place already.  R-MAT 20000 x 12 has 20.4 million such
// values of 15 bits: two passes of 96 us (64-bit keys with the row in front
// took four of 115), 70 of them in k_seg_pass at 2.3 TB/s, which the ranking
// of its tiles bounds.
//
// Digit counts of a tile, at hist[tile0 * R + d * ntiles + tile - tile0] with R
// digits: their prefix over the whole array is where the tile's keys of that
// digit go, since the rows' stretches follow each other.  Tiles past the last
// one (the host knows a bound only) have no keys.
__global__ __launch_bounds__(RX_WG) void k_seg_hist(const EscTile *__restrict__ tiles, const uint2 *__restrict__ last,
                                                    const u32 *__restrict__ vals, int shift, int digit_bits,
                                                    u32 *__restrict__ hist) {
    __shared__ u32 h[RX_RADIX * RX_COPIES];
    const u32 R = 1u << digit_bits;
    if (blockIdx.x >= last->y) {  // uniform
        if (threadIdx.x < R) hist[(u64)blockIdx.x * R + threadIdx.x] = 0;
        return;
    }
    uint4 *mine = reinterpret_cast<uint4 *>(&h[threadIdx.x * RX_COPIES]);
    *mine = make_uint4(0, 0, 0, 0);
    __syncthreads();
    const EscTile t = tiles[blockIdx.x];
    const u32 copy = (u32)dev::lane() % RX_COPIES;
    u32 k[RX_ITEMS];
#pragma unroll
    for (int q = 0; q < RX_ITEMS; ++q) {
        const u32 o = q * RX_WG + threadIdx.x;
        k[q] = o < t.count ? vals[t.start + o] : 0u;
    }
#pragma unroll
    for (int q = 0; q < RX_ITEMS; ++q)
        radix_count((k[q] >> shift) & (R - 1u), q * RX_WG + threadIdx.x < t.count, h, copy);
    __syncthreads();
    if (threadIdx.x < R)
        hist[(u64)t.tile0 * R + (u64)threadIdx.x * t.ntiles + (blockIdx.x - t.tile0)] =
            mine->x + mine->y + mine->z + mine->w;
}

__global__ __launch_bounds__(RX_WG, 5) void k_seg_pass(const EscTile *__restrict__ tiles, const uint2 *__restrict__ last,
                                                    const u32 *__restrict__ in, u32 *__restrict__ out, int shift,
                                                    int digit_bits, const u32 *__restrict__ place) {
    constexpr int NW = RX_WG / dev::WAVE;
    __shared__ u32 skey[RX_TILE];
    __shared__ u32 wcnt[NW][RX_RADIX];
    __shared__ u32 gbase[RX_RADIX];
    __shared__ u32 red[NW + 1];
    if (blockIdx.x >= last->y) return;
    const EscTile t = tiles[blockIdx.x];
    const u32 R = 1u << digit_bits;
    const u32 o0 = (u32)dev::wave_id() * (RX_TILE / NW) + (u32)dev::lane();
    u32 key[RX_ITEMS];
#pragma unroll
    for (int q = 0; q < RX_ITEMS; ++q) {
        const u32 o = o0 + q * dev::WAVE;
        key[q] = o < t.count ? in[t.start + o] : 0u;
    }
    const u32 p = threadIdx.x < R ? place[(u64)t.tile0 * R + (u64)threadIdx.x * t.ntiles + (blockIdx.x - t.tile0)] : 0u;
    auto digit = [&](u32 k) { return (k >> shift) & (R - 1u); };
    radix_tile(key, t.count, digit_bits, p, skey, wcnt, gbase, red, digit);
#pragma unroll
    for (int q = 0; q < RX_ITEMS; ++q) {
        const u32 o = q * RX_WG + threadIdx.x;
        if (o < t.count) out[gbase[digit(skey[o])] + o] = skey[o];
    }
}

// The sorted values of a tile that begin a run of equal ones in their row:
// counted, and with their first places known copied to cols.
template <bool COPY>
__global__ __launch_bounds__(RX_WG) void k_seg_unique(const EscTile *__restrict__ tiles,
                                                      const uint2 *__restrict__ last, const u32 *__restrict__ vals,
                                                      u32 *__restrict__ counts, u32 *__restrict__ cols) {
    constexpr int NW = RX_WG / dev::WAVE;
    __shared__ u32 sc[RX_ITEMS][NW];
    if (blockIdx.x >= last->y) {
        if (!COPY && threadIdx.x == 0) counts[blockIdx.x] = 0;
        return;
    }
    const EscTile t = tiles[blockIdx.x];
    const u32 *v = vals + t.start;
    const bool first = blockIdx.x == t.tile0;
    u32 k[RX_ITEMS];
    u32 fl = 0;
#pragma unroll
    for (int q = 0; q < RX_ITEMS; ++q) {
        const u32 o = q * RX_WG + threadIdx.x;
        k[q] = o < t.count ? v[o] : 0u;
        const bool keep = o < t.count && ((first && o == 0) || v[(long long)o - 1] != k[q]);
        fl |= (keep ? 1u : 0u) << q;
        const unsigned long long m = __ballot(keep);
        if (dev::lane() == 0) sc[q][dev::wave_id()] = (u32)__popcll(m);
    }
    __syncthreads();
    u32 at = COPY ? counts[blockIdx.x] : 0u;
#pragma unroll
    for (int q = 0; q < RX_ITEMS; ++q) {
        u32 before = 0, all = 0;
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            before += w < dev::wave_id() ? sc[q][w] : 0u;
            all += sc[q][w];
        }
        const bool keep = (fl >> q) & 1u;
        if (COPY) {
            const unsigned long long m = __ballot(keep);
            if (keep) cols[at + before + dev::lanes_below(m)] = k[q];
        }
        at += all;
    }
    if (!COPY && threadIdx.x == 0) counts[blockIdx.x] = at;
}

// Sizes and sources of the long rows: nnz_row, the flag that the row comes
// from the sorted stretches, its start there.
__global__ void k_esc_long_rows(const u32 *__restrict__ perm, const uint2 *__restrict__ segs, u32 n,
                                const u32 *__restrict__ places, u32 *__restrict__ nnz_row,
                                u32 *__restrict__ from_side, u64 *__restrict__ soff) {
    const u32 q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= n) return;
    const u32 r = perm[q], a = places[segs[q].y];
    nnz_row[r] = places[segs[q + 1].y] - a;
    from_side[r] = 1;
    soff[r] = a;
}

static int bits_of(u64 maxv) {
    int b = 0;
    while (b < 32 && (1ull << b) <= maxv) ++b;
    return b;
}

void spgemm_esc(clb_controls_s *ctl, const clb_dcsr &a, const clb_dcsr &b, clb_dcsr &out, clb_spgemm_stats &st) {
    std::memset(&st, 0, sizeof(st));
    check_dims(a, b);
    out = clb_dcsr{};
    out.nrows = a.nrows;
    out.ncols = b.ncols;
    // dcsr_matrix_multiplication.cpp:37-40: an empty operand gives an empty result
    if (a.nnz == 0 || b.nnz == 0 || a.nzr == 0) return;
    const u32 nrows = a.nzr;
    Setup s;
    s.lean = true;  // no bitmap rows
    prepare(ctl, a, b, 0, nrows, s, true);
    s.cfg.esc_only = 1;
    s.cfg.tiny_max = 64;
    const u32 lds_max = 1u << ESC_MAX_BITS;
    DevArray<u32> nnz_row(ctl, nrows), tlen(ctl, nrows), from_side(ctl, nrows);
    DevArray<u64> toff(ctl, (u64)nrows + 1), soff(ctl, nrows);
    k_esc_sizes<<<div_up(nrows, 256), 256, 0, ctl->stream>>>(s.P, nrows, lds_max, tlen.ptr, from_side.ptr);
    CLB_LAUNCHED("esc_sizes");
    exclusive_scan_u32_to_u64(ctl, tlen.ptr, toff.ptr, nrows, s.scal.ptr + 1);
    DevArray<u32> perm;
    BinHost h;
    bin_rows(ctl, s, nullptr, nnz_row.ptr, perm);
    read_bins(ctl, s, h);
    const u64 tot[2] = {h.total, h.scal[1]};
    st.products = tot[0];
    st.rows = nrows;
    st.n_bins = NBINS;
    if (tot[0] == 0) return;
    // rows sorted in registers or in LDS: one pass into slots of their
    // product count (never too small)
    DevArray<u32> temp(ctl, tot[1] ? tot[1] : 1);
    Out o{nnz_row.ptr, toff.ptr, temp.ptr, s.P, reinterpret_cast<u32 *>(s.scal.ptr + 5), Dump{}, 0};
    const u32 nlong = h.off[NBINS] - h.off[BIN_BITMAP0];
    const u64 nvals = tot[0] - tot[1];
    if (nvals >= 0xFFFFFFFFull) raise(INVALID_VALUE, "more keys than uint32 indices allow");
    // long rows: expanded, sorted and deduplicated in HBM
    DevArray<uint2> segs;
    DevArray<EscTile> tiles;
    DevArray<u32> vals, other, hist, places;
    u32 *side_cols = nullptr;
    try {
        launch_bins(ctl, s, perm.ptr, h.off, ONE, o, nullptr, CLB_KP_ONEPASS, nullptr, false, true);
        if (nlong) {
            const u32 *lp = perm.ptr + h.off[BIN_BITMAP0];
            const u32 nt = (u32)(nvals / RX_TILE) + nlong;  // at least as many as there are
            const int bits = bits_of(b.ncols ? b.ncols - 1 : 0);
            const int passes = (bits + 7) / 8, digit_bits = passes ? (bits + passes - 1) / passes : 0;
            segs.reset(ctl, (u64)nlong + 1);
            tiles.reset(ctl, nt);
            vals.reset(ctl, nvals);
            other.reset(ctl, passes ? nvals : 0);
            hist.reset(ctl, (u64)nt << digit_bits);
            places.reset(ctl, (u64)nt + 1);
            k_esc_segs<<<1, SEG_WG, 0, ctl->stream>>>(lp, nlong, s.P, segs.ptr);
            CLB_LAUNCHED("esc_segs");
            k_esc_expand<<<nlong, EXP_WG, 0, ctl->stream>>>(s.g, lp, segs.ptr, vals.ptr, tiles.ptr);
            CLB_LAUNCHED("esc_expand");
            const uint2 *last = segs.ptr + nlong;
            u32 *in = vals.ptr, *out_v = other.ptr;
            for (int p = 0; p < passes; ++p) {
                k_seg_hist<<<nt, RX_WG, 0, ctl->stream>>>(tiles.ptr, last, in, p * digit_bits, digit_bits, hist.ptr);
                CLB_LAUNCHED("seg_hist");
                exclusive_scan_u32(ctl, hist.ptr, hist.ptr, (u64)nt << digit_bits, nullptr);
                k_seg_pass<<<nt, RX_WG, 0, ctl->stream>>>(tiles.ptr, last, in, out_v, p * digit_bits, digit_bits,
                                                          hist.ptr);
                CLB_LAUNCHED("seg_pass");
                std::swap(in, out_v);
            }
            k_seg_unique<false><<<nt, RX_WG, 0, ctl->stream>>>(tiles.ptr, last, in, places.ptr, nullptr);
            CLB_LAUNCHED("seg_unique");
            exclusive_scan_u32(ctl, places.ptr, places.ptr, nt, places.ptr + nt);
            k_esc_long_rows<<<div_up(nlong, 256), 256, 0, ctl->stream>>>(lp, segs.ptr, nlong, places.ptr, nnz_row.ptr,
                                                                         from_side.ptr, soff.ptr);
            CLB_LAUNCHED("esc_long_rows");
            // the distinct values go to the other buffer
            if (!passes) other.reset(ctl, nvals);
            side_cols = passes ? out_v : other.ptr;
            k_seg_unique<true><<<nt, RX_WG, 0, ctl->stream>>>(tiles.ptr, last, in, places.ptr, side_cols);
            CLB_LAUNCHED("seg_unique");
        }
        join_side(ctl);
        u64 fails = 0;
        readback(ctl, &fails, s.scal.ptr + 5, 4);
        if ((u32)fails) raise(RUN_KERNEL_FAILURE, "ESC row overflowed its product-count slot");
        DevArray<u64> offs;
        DevArray<u32> pos;
        scan_sizes(ctl, s, nnz_row.ptr, offs, pos);
        u64 sc[3];
        readback(ctl, sc, s.scal.ptr, sizeof(sc));
        const u64 nnz = sc[1];
        const u32 nzr = static_cast<u32>(sc[2]);
        if (nnz > 0xFFFFFFFFull) raise(INVALID_VALUE, "result has more nonzeros than uint32 indices allow");
        if (nnz) {
            clb_buffer_s *cols = buffer_new(ctl, 4ull * nnz);
            try {
                compact_rows(ctl->stream, nrows, nnz, nnz_row.ptr, offs.ptr, temp.ptr, toff.ptr, side_cols,
                             soff.ptr, from_side.ptr, nullptr, nullptr, u32p(cols), nullptr, true);
                assemble(ctl, s, a, nnz_row.ptr, offs.ptr, pos.ptr, nnz, nzr, cols, out);
                sync(ctl);
            } catch (...) {
                settle(ctl);
                if (!out.cols) buffer_release(cols);  // else out's
                clb_dcsr_release(&out);
                throw;
            }
        }
        st.nnz = nnz;
        st.nzr = nzr;
    } catch (...) {
        settle(ctl);
        throw;
    }
}

}  // namespace spg
}  // namespace clb

using namespace clb;

extern "C" {

clb_status clb_dcsr_spgemm_esc(clb_controls ctl, const clb_dcsr *a, const clb_dcsr *b, clb_dcsr *out) {
    return run_guarded(ctl, [&] {
        if (!a || !b || !out) raise(INVALID_ARGUMENT, "null argument");
        clb_spgemm_stats st;
        clb_dcsr r{};
        spg::spgemm_esc(ctl, *a, *b, r, st);
        ctl->last = st;
        *out = r;
    });
}

}  // extern "C"
