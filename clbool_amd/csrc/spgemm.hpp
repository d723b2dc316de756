// spgemm.hpp -- host-side pieces of the SpGEMM shared by the plain, learned
// and batched drivers.
#pragma once

#include "spgemm_kernels.hpp"

namespace clb {
namespace spg {

// Per-call device state: the B row map, per-row product counts and a few
// device scalars ([1] nnz, [2] nzr, [3] overflow flag, ...).
struct Setup {
    u32 nrows = 0, row0 = 0, mapn = 0;
    DevArray<uint2> brange;
    DevArray<u32> bpres;  // presence bits of B rows (hypersparse B only)
    // A without the nonzeros that have no B row (filter_a): a bit per nonzero
    // and their number per tile of `ftile`, then the matrix itself with columns
    // renumbered (bidx) to B's stored rows, whose ranges are crange.
    DevArray<u32> fmask, foffs, bidx, f_rpt, f_cols;
    DevArray<uint2> crange;
    u32 ftile = 0, a_nnz = 0;
    bool filtered = false;
    DevArray<u32> prod;
    DevArray<u64> scal;
    DevArray<u32> ctr;  // row counters of persistent launches (zeroed per launch)
    DevArray<u32> splits;  // per-slice B row ranges (Mats::splits) when ncols spans several windows
    DevArray<u32> packs;  // packed B (Mats::b_packs)
    DevArray<uint2> prange;
    DevArray<u32> psplits;
    bool pack_tried = false;
    // no scratch that only saves time (kept bitmaps, packed B, filtered A, slots
    // of all but the densest dumped rows): there was no room for it
    bool lean = false;
    Mats g{};
    BinCfg cfg{};
    clb_dcsr b{};  // the B operand (its buffers stay owned by the caller)
    u64 bin_products[NBINS] = {};  // of the last binning read back (read_bins)
    u64 bin_work = 0;              // its products, and A nonzeros at 4 each
    u32 *P = nullptr;  // products per row of the block: prod.ptr, or a plan's array
};

// What a plan (plan.hip) hands to one row block's run: the block's slices of
// the per-row arrays computed over all of A at planning time, and the B row
// map and split table built once for all blocks.
struct PlanRows {
    const Setup *shared;  // B row map, presence bits, split table, bin config
    u32 *prod;            // products of the block's rows
    u32 *size;            // plain: exact row sizes; learned / bound: capacities
    const float *pred;    // learned: predicted sizes (nullptr otherwise)
    u64 products;         // sum of prod over the block
    u64 bound;            // one pass: a result above this many nonzeros is not
                          // assembled; the exact row sizes are written to
                          // `size` and *replan is set instead
    bool *replan;
    Store keep;           // plain: bitmaps kept by the plan's symbolic pass, slot_of from the block's first row
};

// HIP-event timing of individual kernel launches, grouped by family
// (CLB_KF(pass, kind) of clbool_c.h).  Disabled unless the caller asked for timing.
struct LaunchTimer {
    bool on = false;
    struct Rec { int family; hipEvent_t a, b; };
    std::vector<Rec> recs;
    hipEvent_t pending = nullptr;
    void begin(hipStream_t st);
    void end(int family, hipStream_t st);
    void collect(clb_spgemm_stats &st);  // after the streams are synchronised
    ~LaunchTimer();
};

constexpr u32 SCALARS = 8;  // Setup::scal
// What a binning leaves in the controls' pinned memory.
struct BinTotals {
    u32 rows[NBINS];
    u64 sums[3 * NBINS];  // products, A nonzeros, key (output nnz)
    u64 scal[SCALARS];    // the product's scalars when the rows were placed
};
// Per-row statistics besides the products (k_row_stats; null: not wanted).
struct RowFeat {
    u32 *mn, *mx, *fc, *lc;
};
// Host copy of the binning: off[b]..off[b+1] is bin b's range of perm.
struct BinHost {
    u32 off[NBINS + 1];
    u64 products[NBINS], a_nnz[NBINS], out_nnz[NBINS];
    u64 total;          // products of all bins
    u64 scal[SCALARS];
};

// Scratch of the dense-bitmap path (see Dump in spgemm_kernels.hpp).
struct DumpBufs {
    bool on = false;
    u32 nbm = 0, nch = 0, words = 0, slots = 0, slice_words = 0;
    DevArray<uint4> store;
    DevArray<u32> cnt, list, count, isdense, fmt;
};
// Buffers of the bitmaps a symbolic pass keeps (see Store).
struct StoreBufs {
    DevArray<uint4> words;
    DevArray<u32> chunks, fmt, slot_of;
    Store keep{};
    void drop() {
        words.free_();
        chunks.free_();
        fmt.free_();
        slot_of.free_();
        keep = Store{};
    }
};
// Below this many products in the bitmap rows their bitmaps are not kept: the
// buffers cost more than the second gather (98 thousand products: 343 us
// kept, 315 not; R-MAT 2^16, 400 million: 1.09 ms kept, 1.60 not).
constexpr u64 KEEP_MIN_PRODUCTS = 1ull << 20;
// Room for the bitmaps (windows of 2^bits words) of the bitmap rows of `h`
// that are worth keeping and fit (keep.words == nullptr: none).
void setup_store(clb_controls_s *ctl, const Setup &s, const BinHost &h, u32 bits, StoreBufs &b);
// Expands rows perm[0 .. n) of a store at their offsets.
void emit_stored(hipStream_t st, const u32 *perm, u32 n, const Store &keep, const u64 *off, u32 *cols);
// Allocates the dense-bitmap scratch for the bitmap bin of `h` (nothing when
// the window is below 2^14 words, the knob disables it or it would not fit)
// and fills o.dump.  With perm and key (the rows' capacities or exact
// sizes), slots only for the rows likely to be dumped; else one per bitmap row.
void setup_dump(clb_controls_s *ctl, const Setup &s, const BinHost &h, DumpBufs &d, Out &o, bool one_pass,
                const u32 *perm = nullptr, const u32 *key = nullptr);
// Expands the dumped rows into cols at the exact row offsets `off`.
void emit_dense(clb_controls_s *ctl, const u32 *perm, const BinHost &h, DumpBufs &d, const u64 *off, u32 *cols,
                LaunchTimer *lt, int pass, clb_spgemm_stats *st);
// The same in two steps: the count and the chunk prefix into gpre on the
// controls' stream (returns the number of dumped rows), then the emission
// kernel on stream `es` (which must be ordered after the prefix).
u32 emit_prepare(clb_controls_s *ctl, DumpBufs &d, DevArray<u64> &gpre, clb_spgemm_stats *st);
void emit_launch(hipStream_t es, u32 count, const u32 *perm, const BinHost &h, const DumpBufs &d, const u64 *gpre,
                 const u64 *off, u32 *cols, LaunchTimer *lt, int pass);

BinCfg make_bincfg(const clb_controls_s *ctl, u32 ncols);
// Where B stores under one row in 16 and the split table over its row ids would
// have this many entries, bitmap rows make the product run over a filtered A,
// whose columns are B's stored rows: the table is then as long as B has rows,
// and no row kernel meets a nonzero without a B row.  Measured filtered against
// not (ms), squares with Zipf columns, bound / plain: 2^24 ids of which 1% are
// stored 1.11 / 1.94 and 1.18 / 2.64, 3% 7.7 / 14.8 and 10.0 / 24.7; 2^22, 1%
// 0.60 / 0.83 and 0.49 / 0.95; 2^21, 3% (6 million entries) 0.84 / 1.05 and
// 0.83 / 1.36.  Small tables cost more launches than they save (30 us), and
// rows of one window gain nothing: 16 million nonzeros, 30 a row, 0.996 /
// 0.963.
constexpr u64 FILTER_MIN_ENTRIES = 1ull << 18;
void ensure_splits(clb_controls_s *ctl, Setup &s, const BinHost &h);
// B packed by groups of 16 columns (Mats::b_packs) for the bitmap rows of `h`,
// after ensure_splits.  Packing costs two passes over B and a read-back, so it
// needs rows that read B often, and columns that share groups: a pack is as
// long as a column index.  Measured packed against not (ms; packs per 100
// nonzeros where they decide): R-MAT 2^16 x 16, plain 0.97 / 1.07; 2^18, plain
// blocks 5.89 / 6.75; 2^20, one pass 41.2 / 46.3; uniform 100 per row of 10^5
// columns (99) 4.30 / 4.43, 600 per row of 10^6 (99) 3.16 / 3.04, 100 per row
// of 20000 (96) 0.77 / 0.79; below 2^24 products the passes cost more than
// they save: R-MAT 20000 vertices, 160000 edges 0.328 / 0.318, uniform 60 per
// row of 3000 0.284 / 0.264.
constexpr u64 PACK_MIN_PRODUCTS = 1ull << 24;
constexpr u32 PACK_MIN_READS = 8;  // products of the bitmap rows per nonzero of B
constexpr u32 PACK_MAX_PCT = 95;   // packs per 100 nonzeros of B
constexpr bool pack_pays(u64 products, u32 b_nnz) {
    return products >= PACK_MIN_PRODUCTS && products >= (u64)PACK_MIN_READS * b_nnz;
}
void ensure_packed(clb_controls_s *ctl, Setup &s, const BinHost &h);
// Gives packed B back; it is not packed again.
void drop_packed(Setup &s);
// B row map, kernel arguments and (stats) per-row products, with `feat` also
// the other statistics.  With `shared`, the B row map, split table and bin
// config are taken from it (a plan's Setup) instead of being built.
void prepare(clb_controls_s *ctl, const clb_dcsr &a, const clb_dcsr &b, u32 row_begin, u32 nrows, Setup &s,
             bool stats = true, const Setup *shared = nullptr, const RowFeat *feat = nullptr);
// Bins the rows of the block by (P, key) into perm (device only, no sync); the
// totals and the scalars as they are then go to pinned memory.
void bin_rows(clb_controls_s *ctl, const Setup &s, const u32 *key, u32 *nnz_row_zero, DevArray<u32> &perm,
              const u32 *slot_of = nullptr);
// Takes the totals of the last bin_rows (synchronises the stream).
void read_bins(clb_controls_s *ctl, Setup &s, BinHost &h);
// Per-bin sums of nnz_row over the rows of each nonempty bin's range of perm
// (rows marked FAILED count 0); the result is read back into out[NBINS].
void sum_by_bin(clb_controls_s *ctl, const u32 *perm, const BinHost &h, u32 nrows, const u32 *nnz_row,
                u64 out[NBINS]);
// Launches the row kernels of every nonempty bin in `mode` (SYM, NUM or ONE)
// on several streams.  family < 0 times launches as sym_* / num_* by mode.
// The controls' stream waits for them at the end, unless `defer` is given:
// then the end of each side stream's work is recorded in defer[k] (NSIDE
// events, made by the caller) for join_deferred.  one_stream: every kernel
// on the controls' stream instead (no side streams).  open: no join, the
// caller joins later (join_side).
// Up to ONE_STREAM_WORK products (an A nonzero counts as four: rows of nonzeros
// without a B row take long without products) the pass is on one stream.
// Measured on one / on several (us): uniform 1024 x 1024 with 98 thousand
// products 102 / 170, 3000 x 3000 with 0.3 million 112 / 178, 30000 x 30000 with
// 0.75 million 161 / 215; at several million products and up there is no
// difference, and 4194 rows of 98 nonzeros, most without a B row, 365 / 319.
constexpr u64 ONE_STREAM_WORK = 3u << 19;
void launch_bins(clb_controls_s *ctl, const Setup &s, const u32 *perm, const u32 off[NBINS + 1], int mode,
                 const Out &o, LaunchTimer *lt, int family, hipEvent_t *defer = nullptr, bool one_stream = false,
                 bool open = false);
// Bitmap rows perm[r0 .. r0 + n) with windows of 2^bits words, by the usual or
// the widest workgroup (bitmap_sym.hip, bitmap_num.hip, bitmap_one.hip).
void launch_bitmap_sym(clb_controls_s *ctl, hipStream_t st, const Setup &s, const u32 *perm, u32 r0, u32 n, u32 bits,
                       bool wide, const Out &o);
void launch_bitmap_num(clb_controls_s *ctl, hipStream_t st, const Setup &s, const u32 *perm, u32 r0, u32 n, u32 bits,
                       bool wide, const Out &o);
void launch_bitmap_one(clb_controls_s *ctl, hipStream_t st, const Setup &s, const u32 *perm, u32 r0, u32 n, u32 bits,
                       bool wide, const Out &o);
// Threads of the bitmap kernels' workgroups and how many of the usual ones a
// CU holds (waves and LDS).
constexpr u32 bitmap_wg(u32 bits) { return bits <= 8 ? 64 : (bits <= 11 ? 256 : (bits <= 14 ? 512 : 1024)); }
constexpr u32 bitmap_wide(u32 bits) { return bits >= 10 ? 1024 : (64u << (bits - 6)); }
constexpr u32 bitmap_resident(u32 bits) {
    const u32 waves = 2048 / bitmap_wg(bits), lds = (160u << 10) / ((4u << bits) + 16 * bitmap_wg(bits));
    return waves < lds ? waves : lds;
}
// The controls' stream waits for the work recorded by a deferred launch_bins.
void join_deferred(clb_controls_s *ctl, const hipEvent_t *defer);
void scan_sizes(clb_controls_s *ctl, Setup &s, const u32 *nnz_row, DevArray<u64> &off, DevArray<u32> &pos);
void assemble(clb_controls_s *ctl, const Setup &s, const clb_dcsr &a, const u32 *nnz_row, const u64 *off,
              const u32 *pos, u64 nnz, u32 nzr, clb_buffer_s *cols, clb_dcsr &out);
void check_dims(const clb_dcsr &a, const clb_dcsr &b);

// pr != nullptr: the block of a plan (the count and symbolic pass were run
// over all rows at planning time; pr->size holds the exact row sizes).
void spgemm_plain(clb_controls_s *ctl, const clb_dcsr &a, const clb_dcsr &b, u32 row_begin, u32 row_end,
                  bool timing, clb_dcsr &out, clb_spgemm_stats &st, const PlanRows *pr = nullptr, bool lean = false);
// Planning passes over all stored rows of A (s from prepare over all rows):
// exact row sizes by the symbolic pass (plain) into size.
void plan_sizes_plain(clb_controls_s *ctl, Setup &s, u32 *size, StoreBufs &store);
// learned.hip.  bound_only: capacities min(P, ncols) for every row, no
// predictor (CLB_SPGEMM_BOUND).
void spgemm_learned(clb_controls_s *ctl, const clb_dcsr &a, const clb_dcsr &b, u32 row_begin, u32 row_end,
                    bool timing, clb_dcsr &out, clb_spgemm_stats &st, bool bound_only = false,
                    const PlanRows *pr = nullptr, bool lean = false);
// The one pass of one block in two halves: start runs everything up to the
// tail (compaction and dense-row emission), which it leaves running on the
// controls' tail streams; finish waits for it and hands over the result.  A
// block that exceeded a plan's bound (one_pass_replan) has no result.
// start is itself launch (binning, and the row kernels left running on the
// side streams) followed by post (the rest, from the overflow count on), so
// that a caller can launch the next block before posting this one: its row
// kernels then queue behind this block's on the side streams and start as
// soon as they end, while the host posts this block.
struct OnePass;
struct OnePassDeleter {
    void operator()(OnePass *p) const;  // waits for the block's kernels first
};
using OnePassPtr = std::unique_ptr<OnePass, OnePassDeleter>;
OnePassPtr one_pass_start(clb_controls_s *ctl, const clb_dcsr &a, const clb_dcsr &b, u32 row_begin, u32 row_end,
                          bool timing, bool bound_only, const PlanRows *pr, bool lean);
OnePassPtr one_pass_launch(clb_controls_s *ctl, const clb_dcsr &a, const clb_dcsr &b, u32 row_begin, u32 row_end,
                           bool timing, bool bound_only, const PlanRows *pr, bool lean);
void one_pass_post(OnePass &p);
bool one_pass_replan(const OnePass &p);
u64 one_pass_bytes(const OnePass &p);  // device memory the block holds
void one_pass_finish(OnePass &p, clb_dcsr &out, clb_spgemm_stats &st);
// Planning pass of the one pass: s prepared over all rows (products in s.P
// afterwards), capacities into size, predictions into pred (learned only).
void plan_sizes_learned(clb_controls_s *ctl, const clb_dcsr &a, const clb_dcsr &b, Setup &s, u32 *size,
                        float *pred, bool bound_only);
// Copies every row r with nnz_row[r] != 0 to cols + off[r] (off: exact
// offsets, off[nrows] = nnz): from side + soff[r] when key2[r] != 0, else
// from temp + toff[r]; rows with isdense[r] are skipped (written elsewhere).
// With pred, accumulates |log2(1 + pred[r]) - log2(1 + nnz_row[r])| into
// *err.  by_tiles: workgroups take equal tiles of output columns instead of
// one row each.  (learned.hip)
void compact_rows(hipStream_t st, u32 nrows, u64 nnz, const u32 *nnz_row, const u64 *off, const u32 *temp,
                  const u64 *toff, const u32 *side, const u64 *soff, const u32 *key2, const u32 *isdense,
                  const float *pred, u32 *cols, double *err, bool by_tiles);
// esc.hip: the expand-sort-compress SpGEMM (dcsr::matrix_multiplication)
void spgemm_esc(clb_controls_s *ctl, const clb_dcsr &a, const clb_dcsr &b, clb_dcsr &out, clb_spgemm_stats &st);
void spgemm_dispatch(clb_controls_s *ctl, const clb_dcsr &a, const clb_dcsr &b, const clb_spgemm_opts &o,
                     clb_dcsr &out, clb_spgemm_stats &st);

}  // namespace spg
}  // namespace clb
