// sort.hip -- device sort and deduplication of (row, col) pairs.
//
// Replaces coo::sort_arrays (src/coo/coo_initialization.cpp:6-32, a bitonic
// network over round_to_power2(n) padded pairs, src/cl/coo_bitonic_sort.cl)
// and reduce_duplicates2 (src/core/matrix_coo.cpp:117-170).  Pairs are sorted
// as 64-bit keys row << 32 | col by a stable LSD radix sort over only the bits
// the matrix needs.  Deduplication counts the kept keys per tile, scans the counts and places
// them.
#include "radix.hpp"
#include "sort.hpp"

namespace clb {

// Sort of pairs (hi, lo) as keys hi << 32 | lo: a stable LSD radix sort.  Bit
// p of the sorted value is bit p of lo for p < lo_bits and bit p - lo_bits of
// hi above, so a digit may hold bits of both halves and no pass is spent on
// bits the shape leaves zero.  A pass is three kernels:
//  * k_radix_hist counts the digits of every tile of RX_TILE keys; a workgroup
//    takes a group of consecutive tiles and keeps the counts before each tile
//    of the group and the group's sums;
//  * k_radix_scan turns the groups' sums into prefixes (a workgroup per digit);
//  * k_radix_pass ranks a tile's keys (per wave, by ballots over the digit's
//    bits and a counter per digit in LDS), orders the tile in LDS and writes
//    each digit's run.
// What bounds it: HBM at 24 bytes per key and pass.  Runs of 16 keys (128
// bytes) on average leave each tile; the sort it replaces scattered single
// keys from registers with five barriers per 256 keys and scanned a count per
// tile and digit in three launches.  A single kernel per pass whose tiles
// gather the counts of the tiles before them (no counting read) was slower:
// with a thousand tiles resident at once each reads hundreds of others' 256
// counts (16.1 million keys, 7-bit digits: 121 us a pass; here 24 + 8 + 64,
// 4.0 TB/s in the last kernel; the sort before this one: 53 + 18 + 63, and six
// passes where the transpose of a 2^20 x 2^20 matrix needs three).
// Keys as an array of 64-bit keys, or as two arrays of halves (keys == nullptr).
struct KeysIn {
    const u64 *keys;
    const u32 *hi, *lo;
    __device__ __forceinline__ u64 operator[](u64 i) const {
        return keys ? keys[i] : ((u64)hi[i] << 32) | lo[i];
    }
};
struct KeysOut {
    u64 *keys;
    u32 *hi, *lo;
    __device__ __forceinline__ void put(u64 i, u64 k) const {
        if (keys) {
            keys[i] = k;
        } else {
            hi[i] = (u32)(k >> 32);
            lo[i] = (u32)k;
        }
    }
};

__device__ __forceinline__ u32 radix_digit(u64 key, int lo_bits, int shift, u32 mask) {
    const u64 v = ((key >> 32) << lo_bits) | (u32)key;
    return (u32)(v >> shift) & mask;
}

__global__ void k_pack_pairs(const u32 *__restrict__ rows, const u32 *__restrict__ cols, u64 n,
                             u64 *__restrict__ keys) {
    const u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) keys[i] = ((u64)rows[i] << 32) | cols[i];
}

__global__ void k_copy_pairs(const u32 *__restrict__ rows, const u32 *__restrict__ cols, u64 n,
                             u32 *__restrict__ out_rows, u32 *__restrict__ out_cols) {
    const u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        out_rows[i] = rows[i];
        out_cols[i] = cols[i];
    }
}

// Digit counts of tiles [g * per, (g + 1) * per) for workgroup g: before[t][d]
// = keys of digit d in the group's tiles before t, sums[g][d] = in all of
// them.
__global__ __launch_bounds__(RX_WG) void k_radix_hist(KeysIn in, u64 n, int lo_bits, int shift, int digit_bits,
                                                      u32 per, u32 tiles, u32 *__restrict__ before,
                                                      u32 *__restrict__ sums) {
    static_assert(RX_WG == RX_RADIX, "a thread per digit");
    __shared__ u32 h[RX_RADIX * RX_COPIES];
    const u32 mask = (1u << digit_bits) - 1u;
    const u32 copy = (u32)dev::lane() % RX_COPIES;
    uint4 *mine = reinterpret_cast<uint4 *>(&h[threadIdx.x * RX_COPIES]);
    *mine = make_uint4(0, 0, 0, 0);
    __syncthreads();
    const u32 t0 = blockIdx.x * per, t1 = tiles - t0 < per ? tiles : t0 + per;
    u32 run = 0;
    for (u32 t = t0; t < t1; ++t) {
        const u64 base = (u64)t * RX_TILE + threadIdx.x;
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            u64 k[RX_ITEMS / 2];
#pragma unroll
            for (int q = 0; q < RX_ITEMS / 2; ++q) {
                const u64 i = base + (u64)(half * (RX_ITEMS / 2) + q) * RX_WG;
                k[q] = i < n ? in[i] : 0ull;
            }
#pragma unroll
            for (int q = 0; q < RX_ITEMS / 2; ++q) {
                const u64 i = base + (u64)(half * (RX_ITEMS / 2) + q) * RX_WG;
                radix_count(radix_digit(k[q], lo_bits, shift, mask), i < n, h, copy);
            }
        }
        __syncthreads();
        before[(u64)t * RX_RADIX + threadIdx.x] = run;
        const uint4 v = *mine;
        run = v.x + v.y + v.z + v.w;  // the counters run on over the group
        __syncthreads();
    }
    sums[(u64)blockIdx.x * RX_RADIX + threadIdx.x] = run;
}

// Workgroup d: exclusive prefix of digit d over the groups, in place, and its
// total.
__global__ __launch_bounds__(RX_WG) void k_radix_scan(u32 *__restrict__ sums, u32 groups, u32 *__restrict__ totals) {
    __shared__ u32 red[RX_WG / dev::WAVE + 1];
    u32 carry = 0;
    for (u32 g0 = 0; g0 < groups; g0 += RX_WG) {
        const u32 g = g0 + threadIdx.x;
        u32 *p = sums + (u64)g * RX_RADIX + blockIdx.x;
        u32 all;
        const u32 x = dev::block_excl_scan<u32, RX_WG>(g < groups ? *p : 0u, red, all);
        if (g < groups) *p = carry + x;
        carry += all;
    }
    if (threadIdx.x == 0) totals[blockIdx.x] = carry;
}

__global__ __launch_bounds__(RX_WG) void k_radix_pass(KeysIn in, KeysOut out, u64 n, int lo_bits, int shift,
                                                     int digit_bits, u32 per, const u32 *__restrict__ before,
                                                     const u32 *__restrict__ sums, const u32 *__restrict__ totals) {
    constexpr int NW = RX_WG / dev::WAVE;
    constexpr u32 WKEYS = RX_TILE / NW;
    __shared__ u64 skey[RX_TILE];
    __shared__ u32 wcnt[NW][RX_RADIX];
    __shared__ u32 gbase[RX_RADIX];
    __shared__ u32 red[NW + 1];
    const int l = dev::lane(), w = dev::wave_id();
    const u32 mask = (1u << digit_bits) - 1u;
    const u32 tile = blockIdx.x;
    const u64 t0 = (u64)tile * RX_TILE;
    const u32 cnt = n - t0 < RX_TILE ? (u32)(n - t0) : RX_TILE;
    // wave w holds keys [w * WKEYS, (w + 1) * WKEYS) of the tile, 64 per item
    u64 key[RX_ITEMS];
    const u32 o0 = (u32)w * WKEYS + (u32)l;
    if (cnt == RX_TILE) {
#pragma unroll
        for (int q = 0; q < RX_ITEMS; ++q) key[q] = in[t0 + o0 + q * dev::WAVE];
    } else {
#pragma unroll
        for (int q = 0; q < RX_ITEMS; ++q) {
            const u32 o = o0 + q * dev::WAVE;
            key[q] = o < cnt ? in[t0 + o] : 0ull;
        }
    }
    // thread d: where digit d's keys of this tile go
    const u32 d = threadIdx.x;
    const u32 of_all = totals[d];
    const u32 prior = sums[(u64)(tile / per) * RX_RADIX + d] + before[(u64)tile * RX_RADIX + d];
    u32 total;
    const u32 place = dev::block_excl_scan<u32, RX_WG>(of_all, red, total) + prior;
    radix_tile(key, cnt, digit_bits, place, skey, wcnt, gbase, red,
               [&](u64 k) { return radix_digit(k, lo_bits, shift, mask); });
#pragma unroll
    for (int q = 0; q < RX_ITEMS; ++q) {
        const u32 o = q * RX_WG + threadIdx.x;
        if (o < cnt) {
            const u64 k = skey[o];
            out.put((u32)(gbase[radix_digit(k, lo_bits, shift, mask)] + o), k);
        }
    }
}

static int bits_for(u64 maxv) {
    int b = 0;
    while (b < 32 && (1ull << b) <= maxv) ++b;
    return b;
}

// Sorts by bits [from_bit, hi_bits + lo_bits) of the value hi << lo_bits | lo.
// `in` holds halves and is only read; the result goes to the halves of `out`
// (which may be the same), or to its keys.
static void radix_sort(clb_controls_s *ctl, KeysIn in, u64 n, int hi_bits, int lo_bits, int from_bit, KeysOut out) {
    if (!n) return;
    if (n > 0xFFFFFFFFull) raise(INVALID_VALUE, "sort of more than 2^32 - 1 keys");
    const int bits = hi_bits + lo_bits - from_bit;
    if (n == 1 || bits <= 0) {  // in order as it is
        if (out.keys) {
            k_pack_pairs<<<div_up(n, 256), 256, 0, ctl->stream>>>(in.hi, in.lo, n, out.keys);
            CLB_LAUNCHED("pack_pairs");
        } else if (in.hi != out.hi) {
            k_copy_pairs<<<div_up(n, 256), 256, 0, ctl->stream>>>(in.hi, in.lo, n, out.hi, out.lo);
            CLB_LAUNCHED("copy_pairs");
        }
        return;
    }
    // digits of equal width; a sort takes at least one pass, which also turns
    // halves into keys or back
    const int passes = bits > 8 ? (bits + 7) / 8 : 1;
    const int digit_bits = bits > passes ? (bits + passes - 1) / passes : 1;
    const u32 tiles = div_up(n, RX_TILE);
    // intermediate passes alternate over two buffers; with keys as the result
    // one of them is the result's, taken in turn so that the last pass ends there
    const bool halves = out.keys == nullptr;
    const bool alias = halves && in.hi == out.hi;
    DevArray<u64> tmp0, tmp1;
    if (passes > 1 || (alias && passes == 1)) tmp0.reset(ctl, n);
    if (halves && passes > 2) tmp1.reset(ctl, n);
    u64 *other = halves ? tmp1.ptr : out.keys;
    // groups of tiles per counting workgroup: one tile until every CU has
    // four, then as many as keep about 1024 groups to scan
    const u32 per = tiles > 1024 ? (tiles + 1023) / 1024 : 1;
    const u32 groups = div_up(tiles, per);
    DevArray<u32> before(ctl, (u64)tiles * RX_RADIX), sums(ctl, (u64)groups * RX_RADIX), totals(ctl, RX_RADIX);
    KeysIn src = in;
    if (alias && passes == 1) {  // the one pass reads a copy
        k_pack_pairs<<<div_up(n, 256), 256, 0, ctl->stream>>>(in.hi, in.lo, n, tmp0.ptr);
        CLB_LAUNCHED("pack_pairs");
        src = KeysIn{tmp0.ptr, nullptr, nullptr};
    }
    for (int p = 0; p < passes; ++p) {
        const bool last = p + 1 == passes;
        // counted from the end: the last pass writes the result, the one before it tmp0, ...
        u64 *buf = ((passes - 1 - p) & 1) ? tmp0.ptr : other;
        const KeysOut dst = last ? out : KeysOut{buf, nullptr, nullptr};
        const int shift = from_bit + p * digit_bits;
        k_radix_hist<<<groups, RX_WG, 0, ctl->stream>>>(src, n, lo_bits, shift, digit_bits, per, tiles, before.ptr,
                                                        sums.ptr);
        CLB_LAUNCHED("radix_hist");
        k_radix_scan<<<RX_RADIX, RX_WG, 0, ctl->stream>>>(sums.ptr, groups, totals.ptr);
        CLB_LAUNCHED("radix_scan");
        k_radix_pass<<<tiles, RX_WG, 0, ctl->stream>>>(src, dst, n, lo_bits, shift, digit_bits, per, before.ptr,
                                                       sums.ptr, totals.ptr);
        CLB_LAUNCHED("radix_pass");
        src = KeysIn{buf, nullptr, nullptr};
    }
}

void sort_pairs_to_keys(clb_controls_s *ctl, const u32 *rows, const u32 *cols, u64 n, u32 max_row, u32 max_col,
                        u64 *keys) {
    radix_sort(ctl, KeysIn{nullptr, rows, cols}, n, bits_for(max_row), bits_for(max_col), 0,
               KeysOut{keys, nullptr, nullptr});
}

void sort_pairs(clb_controls_s *ctl, const u32 *rows, const u32 *cols, u64 n, u32 max_row, u32 max_col,
                bool by_row_only, u32 *out_rows, u32 *out_cols) {
    const int cb = bits_for(max_col);
    radix_sort(ctl, KeysIn{nullptr, rows, cols}, n, bits_for(max_row), cb, by_row_only ? cb : 0,
               KeysOut{nullptr, out_rows, out_cols});
}

// Largest row and column: a maximum per workgroup, so the two words see one
// atomic per workgroup (one per wave took 1.41 ms on 4.0 million pairs, this
// reads them at 8 bytes a pair).
__global__ __launch_bounds__(256) void k_pair_max(const u32 *__restrict__ rows, const u32 *__restrict__ cols, u64 n,
                                                  u32 *__restrict__ mx) {
    __shared__ u32 red[2][4];
    u32 r = 0, c = 0;
    const u64 stride = (u64)gridDim.x * 256;
    for (u64 i = (u64)blockIdx.x * 256 + threadIdx.x; i < n; i += stride) {
        const u32 x = rows[i], y = cols[i];
        r = x > r ? x : r;
        c = y > c ? y : c;
    }
    r = dev::wave_max(r);
    c = dev::wave_max(c);
    if (dev::lane() == 0) {
        red[0][dev::wave_id()] = r;
        red[1][dev::wave_id()] = c;
    }
    __syncthreads();
    if (threadIdx.x < 2) {
        u32 m = 0;
        for (int v = 0; v < 4; ++v) m = red[threadIdx.x][v] > m ? red[threadIdx.x][v] : m;
        if (m) atomicMax(&mx[threadIdx.x], m);
    }
}

void pair_bounds(clb_controls_s *ctl, const u32 *rows, const u32 *cols, u64 n, u32 *max_row, u32 *max_col) {
    DevArray<u32> mx(ctl, 2);
    fill_u32(ctl, mx.ptr, 2, 0);
    if (n) {
        const u32 cap = ctl->cu_count * 8;
        const u32 grid = div_up(n, 256 * 8) < cap ? div_up(n, 256 * 8) : cap;
        k_pair_max<<<grid, 256, 0, ctl->stream>>>(rows, cols, n, mx.ptr);
        CLB_LAUNCHED("pair_max");
    }
    u32 h[2];
    readback(ctl, h, mx.ptr, 8);
    *max_row = h[0];
    *max_col = h[1];
}

// Sorted keys -> distinct keys, in tiles of KT_TILE keys.  Key i is kept
// when it differs from key i - 1.  A count pass gives each tile's kept keys,
// their scan each tile's output offset, and the scatter pass places every kept
// key by its rank inside the tile (ballots per wave and item, counts exchanged
// in LDS).  Loads are striped (item it of thread t is key it * KT_WG + t of
// the tile), so every load and every run of stores is coalesced.
constexpr int KT_WG = 256, KT_ITEMS = 16;
constexpr u64 KT_TILE = (u64)KT_WG * KT_ITEMS;

__device__ __forceinline__ bool key_kept(const u64 *__restrict__ keys, u64 i, u64 k) {
    return i == 0 || keys[i - 1] != k;
}

__global__ __launch_bounds__(KT_WG) void k_keys_count(const u64 *__restrict__ keys, u64 n, u32 *__restrict__ kept) {
    __shared__ u32 red[KT_WG / dev::WAVE + 1];
    const u64 base = (u64)blockIdx.x * KT_TILE;
    u32 c = 0;
#pragma unroll 4
    for (int it = 0; it < KT_ITEMS; ++it) {
        const u64 i = base + (u64)it * KT_WG + threadIdx.x;
        if (i < n) c += key_kept(keys, i, keys[i]);
    }
    const u32 sum = dev::block_sum<u32, KT_WG>(c, red);
    if (threadIdx.x == 0) kept[blockIdx.x] = sum;
}

// cols[p], rows[p] = column and row of the p-th kept key.
__global__ __launch_bounds__(KT_WG) void k_keys_scatter(const u64 *__restrict__ keys, u64 n,
                                                        const u32 *__restrict__ koff, u32 *__restrict__ cols,
                                                        u32 *__restrict__ rows) {
    constexpr int NW = KT_WG / dev::WAVE;
    __shared__ u32 cu[KT_ITEMS][NW];
    const u64 base = (u64)blockIdx.x * KT_TILE;
    const u64 *kt = keys + base;  // the tile, indexed by 32-bit offsets
    const u32 nt = n - base < KT_TILE ? (u32)(n - base) : (u32)KT_TILE;
    const u32 w = dev::wave_id();
    u32 fl = 0;  // bit it: kept
    // pass 1: flags; per wave and item the counts go to LDS
#pragma unroll 4
    for (int it = 0; it < KT_ITEMS; ++it) {
        const u32 o = (u32)it * KT_WG + threadIdx.x;
        const bool f = o < nt && key_kept(keys, base + o, kt[o]);
        fl |= (f ? 1u : 0u) << it;
        const u64 m = __ballot(f);
        if (dev::lane() == 0) cu[it][w] = (u32)__popcll(m);
    }
    __syncthreads();
    // pass 2: ranks; the kept keys are read again (from cache)
    u32 at = koff[blockIdx.x];
#pragma unroll 4
    for (int it = 0; it < KT_ITEMS; ++it) {
        u32 before = 0, all = 0;
#pragma unroll
        for (int v = 0; v < NW; ++v) {
            const u32 x = cu[it][v];
            all += x;
            before += (u32)v < w ? x : 0u;
        }
        const bool kept = (fl >> it) & 1u;
        const u64 m = __ballot(kept);
        if (kept) {
            const u64 k = kt[(u32)it * KT_WG + threadIdx.x];
            const u32 p = at + before + dev::lanes_below(m);
            cols[p] = (u32)k;
            rows[p] = (u32)(k >> 32);
        }
        at += all;
    }
}

void pack_pairs(clb_controls_s *ctl, const u32 *rows, const u32 *cols, u64 n, u64 *keys) {
    if (!n) return;
    k_pack_pairs<<<div_up(n, 256), 256, 0, ctl->stream>>>(rows, cols, n, keys);
    CLB_LAUNCHED("pack_pairs");
}

// Sorted keys -> deduplicated (rows, cols) buffers.
u32 unique_keys_to_pairs(clb_controls_s *ctl, const u64 *keys, u64 n, clb_buffer_s **rows_out,
                         clb_buffer_s **cols_out) {
    *rows_out = *cols_out = nullptr;
    if (n == 0) {
        *rows_out = buffer_new(ctl, 4);
        *cols_out = buffer_new(ctl, 4);
        return 0;
    }
    if (n >= 0xFFFFFFFFull) raise(INVALID_VALUE, "more keys than uint32 indices allow");
    const u32 tiles = (u32)((n + KT_TILE - 1) / KT_TILE);
    DevArray<u32> koff(ctl, (u64)tiles + 1);
    k_keys_count<<<tiles, KT_WG, 0, ctl->stream>>>(keys, n, koff.ptr);
    CLB_LAUNCHED("keys_count");
    exclusive_scan_u32(ctl, koff.ptr, koff.ptr, tiles, koff.ptr + tiles);
    u32 m = 0;
    readback(ctl, &m, koff.ptr + tiles, 4);
    *rows_out = buffer_new(ctl, 4ull * (m ? m : 1));
    try {
        *cols_out = buffer_new(ctl, 4ull * (m ? m : 1));
    } catch (...) {
        buffer_release(*rows_out);
        *rows_out = nullptr;
        throw;
    }
    k_keys_scatter<<<tiles, KT_WG, 0, ctl->stream>>>(keys, n, koff.ptr, u32p(*cols_out), u32p(*rows_out));
    CLB_LAUNCHED("keys_scatter");
    return m;
}

// COO construction: matrix_coo.cpp:17-47 (sort if !sorted, dedup if
// !noDuplicates).  rows/cols are consumed (their references move to out).
void coo_finish(clb_controls_s *ctl, clb_buffer_s *rows, clb_buffer_s *cols, u32 nrows, u32 ncols, u32 nnz,
                bool sorted, bool nodup, clb_coo &out) {
    out = clb_coo{};
    out.nrows = nrows;
    out.ncols = ncols;
    out.rows = rows;
    out.cols = cols;
    out.nnz = nnz;
    if (nnz == 0 || (sorted && nodup)) return;
    u32 mr = 0, mc = 0;
    if (!sorted) pair_bounds(ctl, u32p(rows), u32p(cols), nnz, &mr, &mc);
    if (nodup) {
        sort_pairs(ctl, u32p(rows), u32p(cols), nnz, mr, mc, false, u32p(rows), u32p(cols));
        sync(ctl);
        return;
    }
    DevArray<u64> keys(ctl, nnz);
    if (sorted) pack_pairs(ctl, u32p(rows), u32p(cols), nnz, keys.ptr);
    else sort_pairs_to_keys(ctl, u32p(rows), u32p(cols), nnz, mr, mc, keys.ptr);
    clb_buffer_s *nr = nullptr, *nc = nullptr;
    const u32 m = unique_keys_to_pairs(ctl, keys.ptr, nnz, &nr, &nc);
    sync(ctl);
    buffer_release(rows);
    buffer_release(cols);
    out.rows = nr;
    out.cols = nc;
    out.nnz = m;
}

}  // namespace clb

using namespace clb;

extern "C" {

clb_status clb_coo_from_host(clb_controls ctl, const uint32_t *rows, const uint32_t *cols, uint32_t nrows,
                             uint32_t ncols, uint32_t nnz, int sorted, int no_duplicates, clb_coo *out) {
    return run_guarded(ctl, [&] {
        clb_coo r{};
        r.nrows = nrows;
        r.ncols = ncols;
        if (nnz == 0) {  // matrix_coo.cpp:29
            *out = r;
            return;
        }
        clb_buffer_s *rb = buffer_new(ctl, 4ull * nnz);
        clb_buffer_s *cbuf = nullptr;
        try {
            cbuf = buffer_new(ctl, 4ull * nnz);
            CLB_HIP(hipMemcpyAsync(rb->ptr, rows, 4ull * nnz, hipMemcpyHostToDevice, ctl->stream), WRITE_BUFFER_ERROR);
            CLB_HIP(hipMemcpyAsync(cbuf->ptr, cols, 4ull * nnz, hipMemcpyHostToDevice, ctl->stream),
                    WRITE_BUFFER_ERROR);
            sync(ctl);
        } catch (...) {
            buffer_release(rb);
            buffer_release(cbuf);
            throw;
        }
        coo_finish(ctl, rb, cbuf, nrows, ncols, nnz, sorted != 0, no_duplicates != 0, r);
        *out = r;
    });
}

clb_status clb_coo_from_buffers(clb_controls ctl, uint32_t nrows, uint32_t ncols, uint32_t nnz, clb_buffer rows,
                                clb_buffer cols, int sorted, int no_duplicates, clb_coo *out) {
    return run_guarded(ctl, [&] {
        clb_coo r{};
        if (nnz && (!rows || !cols || rows->bytes < 4ull * nnz || cols->bytes < 4ull * nnz))
            raise(INVALID_ARGUMENT, "matrix_coo: buffers smaller than nnz");
        // matrix_coo.cpp:59: the matrix shares the given buffers
        buffer_retain(rows);
        buffer_retain(cols);
        if (!sorted && nnz) {  // sorting happens in place, as coo::sort_arrays does
            u32 mr, mc;
            pair_bounds(ctl, u32p(rows), u32p(cols), nnz, &mr, &mc);
            sort_pairs(ctl, u32p(rows), u32p(cols), nnz, mr, mc, false, u32p(rows), u32p(cols));
            sync(ctl);
        }
        coo_finish(ctl, nnz ? rows : nullptr, nnz ? cols : nullptr, nrows, ncols, nnz, true, no_duplicates != 0, r);
        if (!nnz) {
            buffer_release(rows);
            buffer_release(cols);
        }
        *out = r;
    });
}

clb_status clb_coo_sort_arrays(clb_controls ctl, clb_buffer rows, clb_buffer cols, uint32_t n) {
    return run_guarded(ctl, [&] {
        if (n == 0) return;
        if (!rows || !cols || rows->bytes < 4ull * n || cols->bytes < 4ull * n)
            raise(INVALID_ARGUMENT, "sort_arrays: buffers smaller than n");
        u32 mr, mc;
        pair_bounds(ctl, u32p(rows), u32p(cols), n, &mr, &mc);
        sort_pairs(ctl, u32p(rows), u32p(cols), n, mr, mc, false, u32p(rows), u32p(cols));
        sync(ctl);
    });
}

}  // extern "C"
