// closure.hip -- batched closure step of CFPQ/RPQ evaluation: X_t |= Y_t * Z_t
// for a set of triples t over label matrices that share one vertex set.
//
// clBool itself has no closure driver: its user (spbla) calls
// dcsr::matrix_multiplication_hash and an addition once per triple.  The
// per-triple loop is kept here as the baseline (mode CLB_CLOSURE_PER_TRIPLE).
// The batched mode runs all products of a step as ONE SpGEMM on stacked
// operands: Y' = [Y_0 | Y_1 | ...] (row block t holds Y_t, its columns shifted
// by t * n) times Z' = [Z_0; Z_1; ...] (row block t holds Z_t) gives row block
// t of the result = Y_t * Z_t, so every kernel launch of the SpGEMM covers the
// rows of all products.  The product is taken in row blocks of Y' whose
// output bound (sum over rows of min(products, n)) stays below 2^32, so each
// block's result fits uint32 indices however large the step grows.  Each X's
// union merges sorted key segments -- its own keys and, per triple that
// targets it, that triple's product rows (already sorted: a product block is
// canonical DCSR) -- and drops duplicates.  Every step of both modes is
// bit-exact: the products
// and unions are exact set operations, only the launch structure differs.
#include "expand.hpp"
#include "sort.hpp"
#include "spgemm.hpp"

#include <algorithm>
#include <chrono>

namespace clb {

// One matrix of a stacked operand.
struct Seg {
    const u32 *rpt, *rows, *cols;
    u32 nzr, nnz;
    u32 row_shift, col_shift;  // added to row ids and to column ids
    u32 nzr_off, nnz_off;      // position of the block in the stack
};

// Copies the blocks' rows (ids shifted) and row pointers (offset by the
// block's nonzero position) into the stack; one thread per stored row.
__global__ void k_stack_rows(const Seg *__restrict__ segs, u32 nseg, u32 total_nzr, u32 *__restrict__ rpt,
                             u32 *__restrict__ rows, u32 total_nnz) {
    const u32 g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g == 0) rpt[total_nzr] = total_nnz;
    if (g >= total_nzr) return;
    u32 lo = 0, hi = nseg;  // last segment with nzr_off <= g
    while (hi - lo > 1) {
        const u32 mid = (lo + hi) / 2;
        if (segs[mid].nzr_off <= g) lo = mid;
        else hi = mid;
    }
    while (lo + 1 < nseg && segs[lo + 1].nzr_off <= g) ++lo;  // skip empty segments
    const Seg &s = segs[lo];
    const u32 i = g - s.nzr_off;
    rows[g] = s.rows[i] + s.row_shift;
    rpt[g] = s.rpt[i] + s.nnz_off;
}

// Copies the blocks' columns (shifted); one thread per nonzero.
__global__ void k_stack_cols(const Seg *__restrict__ segs, u32 nseg, u32 total_nnz, u32 *__restrict__ cols) {
    const u32 e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= total_nnz) return;
    u32 lo = 0, hi = nseg;
    while (hi - lo > 1) {
        const u32 mid = (lo + hi) / 2;
        if (segs[mid].nnz_off <= e) lo = mid;
        else hi = mid;
    }
    while (lo + 1 < nseg && segs[lo + 1].nnz_off <= e) ++lo;
    const Seg &s = segs[lo];
    cols[e] = s.cols[e - s.nnz_off] + s.col_shift;
}

// Keys (row << 32 | col) of many pieces of DCSR matrices in one launch.
struct KeySeg {
    const u32 *rpt, *rows, *cols;
    u32 r_lo, r_hi;    // the piece's stored rows: nonzeros [rpt[r_lo], rpt[r_hi])
    u32 e_lo, e_hi;
    u32 row_shift;     // added to row ids (modulo 2^32)
    u32 tile0;         // its first tile of the launch
    u64 *keys;         // the piece's first key
};

// One tile of EX_TILE nonzeros per workgroup.  The piece is found by one
// probe per thread, the tile's first and last rows by rounds of a 256-way
// split: dependent loads, but no launch of its own per piece, and a closure's
// pieces are many and mostly small.
__global__ __launch_bounds__(EX_WG) void k_keys_segs(const KeySeg *__restrict__ segs, u32 nseg) {
    __shared__ u32 srpt[EX_TILE], srow[EX_TILE];
    u32 s = 0;  // last piece with tile0 <= this tile (pieces are not empty)
    for (u32 b = 0; b < nseg; b += EX_WG) {
        const u32 k = b + threadIdx.x;
        s += (u32)__syncthreads_count(k < nseg && segs[k].tile0 <= blockIdx.x);
    }
    const KeySeg g = segs[s - 1];
    const u64 e0 = (u64)g.e_lo + (u64)(blockIdx.x - g.tile0) * EX_TILE;
    const u64 e1 = e0 + EX_TILE < g.e_hi ? e0 + EX_TILE : g.e_hi;
    // last row in [lo, hi) that starts at or before e
    auto row_of = [&](u32 lo, u32 hi, u64 e) {
        while (hi - lo > 1) {
            const u32 step = (hi - lo + EX_WG - 1) / EX_WG;
            const u64 c = (u64)lo + (u64)threadIdx.x * step;
            const u32 cnt = (u32)__syncthreads_count(c < hi && g.rpt[c] <= e);
            lo += (cnt - 1) * step;
            hi = hi - lo < step ? hi : lo + step;
        }
        return lo;
    };
    const u32 r0 = row_of(g.r_lo, g.r_hi, e0);
    // at most EX_TILE rows, unless some stored rows are empty
    const bool near = g.r_hi - r0 > EX_TILE && g.rpt[r0 + EX_TILE] >= e1;
    const u32 nr = row_of(r0, near ? r0 + EX_TILE : g.r_hi, e1 - 1) - r0 + 1;
    const bool staged = nr <= EX_TILE;
    if (staged)
        for (u32 j = threadIdx.x; j < nr; j += EX_WG) {
            srpt[j] = g.rpt[r0 + j];
            srow[j] = g.rows[r0 + j];
        }
    __syncthreads();
#pragma unroll
    for (u32 q = 0; q < EX_ITEMS; ++q) {
        const u64 e = e0 + q * EX_WG + threadIdx.x;
        if (e >= e1) break;
        u32 a = 0, b = nr;
        while (b - a > 1) {
            const u32 m = (a + b) >> 1;
            if ((staged ? srpt[m] : g.rpt[r0 + m]) <= e) a = m;
            else b = m;
        }
        const u32 id = staged ? srow[a] : g.rows[r0 + a];
        g.keys[e - g.e_lo] = ((u64)(id + g.row_shift) << 32) | g.cols[e];
    }
}

// The output bound of a stored row of Y': min(its products, n).
struct RowBound {
    const u32 *prod;
    u32 n;
    __device__ __forceinline__ u64 operator()(u64 r) const { return prod[r] < n ? prod[r] : n; }
};

__global__ void k_row_bounds(RowBound f, u32 nzr, u64 *__restrict__ bound) {
    const u32 r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r < nzr) bound[r] = f(r);
}

// Their sum; at most RB_GRID workgroups, since each adds to one word.
constexpr u32 RB_GRID = 128;
__global__ __launch_bounds__(256) void k_bound_sum(RowBound f, u32 nzr, u64 *__restrict__ sum) {
    __shared__ u64 red[256 / dev::WAVE + 1];
    u64 v = 0;
    for (u64 r = (u64)blockIdx.x * 256 + threadIdx.x; r < nzr; r += (u64)gridDim.x * 256) v += f(r);
    v = dev::block_sum<u64, 256>(v, red);
    if (threadIdx.x == 0 && v) atomicAdd(reinterpret_cast<unsigned long long *>(sum), (unsigned long long)v);
}

// cuts[b] = first stored row whose exclusive bound prefix is >= b * step
// (pre holds nzr + 1 entries, pre[nzr] = the total).  Every row's bound is at
// most n, so with step = lim - n + 1 a block [cuts[b], cuts[b+1]) has bound
// pre[cuts[b+1]] - pre[cuts[b]] < (b+1)*step + n - b*step, i.e. at most lim.
// bbound[b] receives that block bound.
__global__ void k_cuts(const u64 *__restrict__ pre, u32 nzr, u64 step, u32 nb, u32 *__restrict__ cuts) {
    const u32 b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b > nb) return;
    if (b == nb) {
        cuts[b] = nzr;
        return;
    }
    const u64 target = (u64)b * step;
    u32 lo = 0, hi = nzr;
    while (lo < hi) {
        const u32 mid = lo + (hi - lo) / 2;
        if (pre[mid] < target) lo = mid + 1;
        else hi = mid;
    }
    cuts[b] = lo;
}

__global__ void k_block_bounds(const u64 *__restrict__ pre, const u32 *__restrict__ cuts, u32 nb,
                               u64 *__restrict__ bbound) {
    const u32 b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b < nb) bbound[b] = pre[cuts[b + 1]] - pre[cuts[b]];
}

// For row blocks t = 0..nt of a product (row ids t*n + i): out[2t] = first
// stored row with id >= t*n, out[2t+1] = its position in cols.
__global__ void k_row_splits(const u32 *__restrict__ rpt, const u32 *__restrict__ rows, u32 nzr, u32 n, u32 nt,
                             u32 *__restrict__ out) {
    const u32 t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t > nt) return;
    const u64 target = (u64)t * n;
    u32 lo = 0, hi = nzr;
    while (lo < hi) {
        const u32 mid = lo + (hi - lo) / 2;
        if ((u64)rows[mid] < target) lo = mid + 1;
        else hi = mid;
    }
    out[2 * t] = lo;
    out[2 * t + 1] = rpt[lo];
}

// Output bound of one stacked row block: the caller's block_bound (0 or
// above 2^32 - 1: 2^32 - 1), raised to 2n when smaller (one row's bound is up
// to n, and cuts need room for at least one row).
static u64 closure_block_limit(u32 block_bound, u32 n) {
    u64 lim = block_bound ? block_bound : 0xFFFFFFFFull;
    if (lim < 2ull * n) lim = 2ull * n;
    return lim < 0xFFFFFFFFull ? lim : 0xFFFFFFFFull;
}

// Builds the stack of the given matrices on the device; segs stays as it is
// until the controls' stream has been waited for.
static clb_dcsr stack(clb_controls_s *ctl, std::vector<Seg> &segs, u32 nrows, u32 ncols) {
    u64 nzr = 0, nnz = 0;
    for (auto &s : segs) {
        s.nzr_off = (u32)nzr;
        s.nnz_off = (u32)nnz;
        nzr += s.nzr;
        nnz += s.nnz;
    }
    if (nnz > 0xFFFFFFFFull) raise(INVALID_VALUE, "stacked operand exceeds uint32 nonzeros");
    clb_dcsr m{};
    m.nrows = nrows;
    m.ncols = ncols;
    if (!nnz) return m;
    DevArray<Seg> dseg(ctl, segs.size());
    CLB_HIP(hipMemcpyAsync(dseg.ptr, segs.data(), segs.size() * sizeof(Seg), hipMemcpyHostToDevice, ctl->stream),
            WRITE_BUFFER_ERROR);
    m.rpt = buffer_new(ctl, 4 * (nzr + 1));
    m.rows = buffer_new(ctl, 4 * nzr);
    m.cols = buffer_new(ctl, 4 * nnz);
    k_stack_rows<<<div_up(nzr + 1, 256), 256, 0, ctl->stream>>>(dseg.ptr, (u32)segs.size(), (u32)nzr, u32p(m.rpt),
                                                                 u32p(m.rows), (u32)nnz);
    CLB_LAUNCHED("stack_rows");
    k_stack_cols<<<div_up(nnz, 256), 256, 0, ctl->stream>>>(dseg.ptr, (u32)segs.size(), (u32)nnz, u32p(m.cols));
    CLB_LAUNCHED("stack_cols");
    m.nnz = (u32)nnz;
    m.nzr = (u32)nzr;
    return m;
}

static Seg seg_of(const clb_dcsr &m, u32 row_shift, u32 col_shift) {
    return Seg{u32p(m.rpt), u32p(m.rows), u32p(m.cols), m.nzr, m.nnz, row_shift, col_shift, 0, 0};
}

// X |= its products for every distinct X of the step.  A batch of X
// matrices is united at once: their keys are stacked (matrix x in rows
// [x * n, (x + 1) * n)) into one sorted list, and so are, for r = 0, 1, ..., the
// products of each one's r-th triple (a product's parts in consecutive row
// blocks follow each other in row order).  The products' lists are merged
// pairwise into one, which the union then meets the matrices' list with.  A
// batch holds at most UNITE_KEYS keys (or one matrix), which bounds its
// memory; where there is no room for that either, it is one matrix.  United
// one by one, the 17 matrices of a 32-rule step took 4.0 ms, mostly launches and
// read-backs, for 6.1 million keys.
constexpr u64 UNITE_KEYS = 1ull << 27;

// One batch: matrices xs[batch[i]], `total` keys in all and `base` their own.
static void unite_batch(clb_controls_s *ctl, clb_dcsr *mats, const std::vector<u32> &xs,
                        const std::vector<std::vector<u32>> &of, const std::vector<size_t> &batch, u64 total, u64 base,
                        u32 n, const std::vector<clb_dcsr> &prods, const std::vector<std::vector<u32>> &splits) {
    auto part = [&](size_t q, u32 t) -> u64 { return splits[q][2 * t + 3] - splits[q][2 * t + 1]; };
    DevArray<u64> keys(ctl, total), tmp(ctl, total - base);  // matrices | products; tmp: products
    std::vector<KeySeg> segs;
    u32 tiles = 0;
    auto piece = [&](const clb_dcsr &m, u32 r_lo, u32 r_hi, u32 e_lo, u32 e_hi, u32 shift, u64 at) {
        if (e_hi == e_lo) return;
        segs.push_back(KeySeg{u32p(m.rpt), u32p(m.rows), u32p(m.cols), r_lo, r_hi, e_lo, e_hi, shift, tiles,
                              keys.ptr + at});
        tiles += div_up((u64)e_hi - e_lo, EX_TILE);
    };
    u64 pos = 0;
    size_t rounds = 0;
    for (size_t i = 0; i < batch.size(); ++i) {
        const clb_dcsr &x = mats[xs[batch[i]]];
        piece(x, 0, x.nzr, 0, x.nnz, (u32)i * n, pos);
        pos += x.nnz;
        rounds = std::max(rounds, of[batch[i]].size());
    }
    std::vector<std::pair<u64, u64>> lists;  // (start, length) after the matrices' keys
    for (size_t r = 0; r < rounds; ++r) {
        const u64 start = pos;
        for (size_t i = 0; i < batch.size(); ++i) {
            if (r >= of[batch[i]].size()) continue;
            const u32 t = of[batch[i]][r];
            for (size_t q = 0; q < prods.size(); ++q) {
                const std::vector<u32> &hs = splits[q];
                // rows t * n + row -> i * n + row
                piece(prods[q], hs[2 * t], hs[2 * t + 2], hs[2 * t + 1], hs[2 * t + 3], ((u32)i - t) * n, pos);
                pos += part(q, t);
            }
        }
        lists.push_back({start - base, pos - start});
    }
    DevArray<KeySeg> dsegs(ctl, segs.size());
    CLB_HIP(hipMemcpyAsync(dsegs.ptr, segs.data(), segs.size() * sizeof(KeySeg), hipMemcpyHostToDevice,
                           ctl->stream),
            WRITE_BUFFER_ERROR);
    k_keys_segs<<<tiles, EX_WG, 0, ctl->stream>>>(dsegs.ptr, (u32)segs.size());
    CLB_LAUNCHED("keys");
    u64 *cur = keys.ptr + base, *nxt = tmp.ptr;
    while (lists.size() > 1) {
        std::vector<std::pair<u64, u64>> next;
        for (size_t i = 0; i < lists.size(); i += 2) {
            const auto &la = lists[i];
            if (i + 1 == lists.size()) {  // odd one out: copied to the other buffer
                CLB_HIP(hipMemcpyAsync(nxt + la.first, cur + la.first, 8 * la.second, hipMemcpyDeviceToDevice,
                                       ctl->stream),
                        COPY_BUFFER_ERROR);
                next.push_back(la);
                continue;
            }
            const auto &lb = lists[i + 1];  // adjacent
            merge_keys(ctl, cur + la.first, la.second, cur + lb.first, lb.second, nxt + la.first);
            next.push_back({la.first, la.second + lb.second});
        }
        lists.swap(next);
        std::swap(cur, nxt);
    }
    std::vector<clb_dcsr> united;
    for (size_t i : batch) united.push_back(mats[xs[i]]);
    union_keys_to_matrices(ctl, keys.ptr, base, cur, total - base, n, united);
    for (size_t i = 0; i < batch.size(); ++i) {
        clb_dcsr &x = mats[xs[batch[i]]];
        if (united[i].cols == x.cols) continue;  // unchanged
        clb_dcsr_release(&x);
        x = united[i];
    }
}

static void unite_products(clb_controls_s *ctl, clb_dcsr *mats, const std::vector<u32> &xs, const u32 *triples,
                           u32 ntriples, u32 n, const std::vector<clb_dcsr> &prods,
                           const std::vector<std::vector<u32>> &splits) {
    auto part = [&](size_t q, u32 t) -> u64 { return splits[q][2 * t + 3] - splits[q][2 * t + 1]; };
    std::vector<std::vector<u32>> of(xs.size());  // each X's triples with products
    std::vector<u64> add(xs.size(), 0);           // their nonzeros
    for (u32 t = 0; t < ntriples; ++t) {
        u64 len = 0;
        for (size_t q = 0; q < prods.size(); ++q) len += part(q, t);
        if (!len) continue;
        const size_t k = std::lower_bound(xs.begin(), xs.end(), triples[3 * t]) - xs.begin();
        of[k].push_back(t);
        add[k] += len;
    }
    size_t k0 = 0;
    u64 most = UNITE_KEYS;
    while (k0 < xs.size()) {
        if (of[k0].empty()) {
            ++k0;
            continue;
        }
        std::vector<size_t> batch;
        u64 total = 0, base = 0;  // keys in all, and of the matrices themselves
        size_t k1 = k0;
        for (; k1 < xs.size(); ++k1) {
            if (of[k1].empty()) continue;
            const u64 mine = mats[xs[k1]].nnz + add[k1];
            if (mine >= 0xFFFFFFFFull) raise(INVALID_VALUE, "a closure union exceeds uint32 nonzeros");
            if (!batch.empty() && total + mine > most) break;
            batch.push_back(k1);
            total += mine;
            base += mats[xs[k1]].nnz;
        }
        try {
            unite_batch(ctl, mats, xs, of, batch, total, base, n, prods, splits);
        } catch (const Error &e) {
            if (!no_room(e) || batch.size() == 1) throw;
            make_room(ctl);
            most = 0;
            continue;
        }
        k0 = k1;
    }
}

}  // namespace clb

using namespace clb;

extern "C" {

clb_status clb_closure_step(clb_controls ctl, clb_dcsr *mats, uint32_t nmats, const uint32_t *triples,
                            uint32_t ntriples, const clb_closure_opts *opts, clb_closure_stats *stats) {
    return run_guarded(ctl, [&] {
        clb_closure_opts o{};
        if (opts) o = *opts;
        clb_closure_stats st{};
        auto t0 = std::chrono::steady_clock::now();
        if (!nmats) raise(INVALID_ARGUMENT, "no matrices");
        const u32 n = mats[0].nrows;
        for (u32 k = 0; k < nmats; ++k)
            if (mats[k].nrows != n || mats[k].ncols != n)
                raise(INVALID_ARGUMENT, "closure matrices must share one square vertex set");
        for (u32 t = 0; t < 3 * ntriples; ++t)
            if (triples[t] >= nmats) raise(INVALID_ARGUMENT, "triple names an unknown matrix");
        std::vector<u64> before(nmats);
        for (u32 k = 0; k < nmats; ++k) before[k] = mats[k].nnz;
        // distinct X matrices of the step
        std::vector<u32> xs;
        for (u32 t = 0; t < ntriples; ++t) xs.push_back(triples[3 * t]);
        std::sort(xs.begin(), xs.end());
        xs.erase(std::unique(xs.begin(), xs.end()), xs.end());
        clb_spgemm_opts so{};
        so.mode = o.spgemm_mode;
        auto t_prod = t0;  // end of the products phase

        if (o.mode == CLB_CLOSURE_PER_TRIPLE) {
            // the reference-style loop: products from the step's start values,
            // then one union per triple
            std::vector<clb_dcsr> prods(ntriples);
            try {
                for (u32 t = 0; t < ntriples; ++t) {
                    clb_spgemm_stats ss;
                    spg::spgemm_dispatch(ctl, mats[triples[3 * t + 1]], mats[triples[3 * t + 2]], so, prods[t], ss);
                    st.products += ss.products;
                    st.fallback_rows += ss.fallback_rows;
                    st.dense_rows += ss.dense_rows;
                    ++st.spgemm_calls;
                }
                sync(ctl);
                t_prod = std::chrono::steady_clock::now();
                for (u32 t = 0; t < ntriples; ++t) {
                    clb_dcsr &x = mats[triples[3 * t]];
                    clb_dcsr u{};
                    const clb_status rc = clb_dcsr_addition(ctl, &x, &prods[t], &u);
                    if (rc != CLB_SUCCESS) raise(static_cast<Status>(rc - 1), clb_last_error());
                    clb_dcsr_release(&x);
                    x = u;
                }
            } catch (...) {
                settle(ctl);
                for (auto &p : prods) clb_dcsr_release(&p);
                throw;
            }
            for (auto &p : prods) clb_dcsr_release(&p);
        } else {
            if ((u64)ntriples * n > 0xFFFFFFFFull || n > (1u << 31))
                raise(INVALID_VALUE, "stacked operands exceed uint32 indices");
            // Y' (row block t = Y_t, columns shifted by t*n) and Z' (row block t = Z_t)
            std::vector<Seg> ys, zs;
            for (u32 t = 0; t < ntriples; ++t) {
                ys.push_back(seg_of(mats[triples[3 * t + 1]], t * n, t * n));
                zs.push_back(seg_of(mats[triples[3 * t + 2]], t * n, 0));
            }
            std::vector<clb_dcsr> prods;  // row blocks of Y' * Z'
            std::vector<std::vector<u32>> splits;
            auto release_all = [&] {
                for (auto &p : prods) clb_dcsr_release(&p);
            };
            clb_dcsr Y = stack(ctl, ys, ntriples * n, ntriples * n);
            clb_dcsr Z{};
            try {
                Z = stack(ctl, zs, ntriples * n, n);
                if (Y.nnz && Z.nnz) {
                    // row blocks of Y' with output bound below 2^32 each; one
                    // block when the sum of its rows' bounds says so
                    const u64 lim = closure_block_limit(o.block_bound, n);
                    const u64 step = lim - n + 1;
                    std::vector<u32> hc{0, Y.nzr};
                    std::vector<u64> hb(1);
                    u32 nb = 0;
                    {
                        spg::Setup ps;
                        ps.lean = true;  // the products per row are all it is for
                        spg::prepare(ctl, Y, Z, 0, Y.nzr, ps, true);
                        const RowBound rb{ps.P, n};
                        const u32 grid = div_up(Y.nzr, 256) < RB_GRID ? div_up(Y.nzr, 256) : RB_GRID;
                        k_bound_sum<<<grid, 256, 0, ctl->stream>>>(rb, Y.nzr, ps.scal.ptr);
                        CLB_LAUNCHED("bound_sum");
                        u64 total = 0;
                        readback(ctl, &total, ps.scal.ptr, 8);
                        nb = (u32)((total + step - 1) / step);
                        if (nb == 1) {
                            hb[0] = total;
                        } else if (nb > 1) {
                            DevArray<u64> pre(ctl, (u64)Y.nzr + 1);
                            k_row_bounds<<<div_up(Y.nzr, 256), 256, 0, ctl->stream>>>(rb, Y.nzr, pre.ptr);
                            CLB_LAUNCHED("row_bounds");
                            exclusive_scan_u64(ctl, pre.ptr, pre.ptr, Y.nzr, pre.ptr + Y.nzr);
                            DevArray<u32> cuts(ctl, (u64)nb + 1);
                            DevArray<u64> bb(ctl, nb);
                            k_cuts<<<div_up(nb + 1, 256), 256, 0, ctl->stream>>>(pre.ptr, Y.nzr, step, nb, cuts.ptr);
                            CLB_LAUNCHED("cuts");
                            k_block_bounds<<<div_up(nb, 256), 256, 0, ctl->stream>>>(pre.ptr, cuts.ptr, nb, bb.ptr);
                            CLB_LAUNCHED("block_bounds");
                            hc.resize((size_t)nb + 1);
                            hb.resize(nb);
                            readback(ctl, hc.data(), cuts.ptr, 4ull * (nb + 1));
                            readback(ctl, hb.data(), bb.ptr, 8ull * nb);
                        }
                    }
                    for (u32 k = 0; k < nb; ++k) {
                        if (hb[k] > lim) raise(RUN_KERNEL_FAILURE, "closure row block exceeds its output bound");
                        if (hb[k] > st.max_block_bound) st.max_block_bound = hb[k];
                    }
                    DevArray<u32> sp(ctl, 2ull * (ntriples + 1));
                    auto absorb = [&](clb_dcsr &T, const clb_spgemm_stats &ss) {
                        st.products += ss.products;
                        st.fallback_rows += ss.fallback_rows;
                        st.dense_rows += ss.dense_rows;
                        ++st.spgemm_calls;
                        if (!T.nnz) {
                            clb_dcsr_release(&T);
                            return;
                        }
                        prods.push_back(T);
                        // where each product block t starts in T
                        k_row_splits<<<div_up(ntriples + 1, 256), 256, 0, ctl->stream>>>(
                            u32p(T.rpt), u32p(T.rows), T.nzr, n, ntriples, sp.ptr);
                        CLB_LAUNCHED("row_splits");
                        std::vector<u32> hs(2 * (ntriples + 1));
                        readback(ctl, hs.data(), sp.ptr, 4ull * hs.size());
                        splits.push_back(hs);
                    };
                    const bool one_pass = so.mode == CLB_SPGEMM_LEARNED || so.mode == CLB_SPGEMM_BOUND;
                    if (!one_pass) {
                        for (u32 k = 0; k < nb; ++k) {
                            if (hc[k + 1] <= hc[k]) continue;
                            clb_spgemm_opts bo = so;
                            bo.row_begin = hc[k];
                            bo.row_end = hc[k + 1];
                            clb_spgemm_stats ss;
                            clb_dcsr T{};
                            spg::spgemm_dispatch(ctl, Y, Z, bo, T, ss);
                            absorb(T, ss);
                        }
                    } else {
                        // one-pass blocks overlap: block k + 1's passes start while
                        // block k's compaction and dense-row emission still run,
                        // and its row kernels are launched before block k is
                        // posted, so that they follow block k's on the device
                        // (each when device memory allows)
                        spg::OnePassPtr pend, cur, nxt;
                        auto finish_pending = [&]() {
                            clb_dcsr T{};
                            clb_spgemm_stats ss;
                            spg::one_pass_finish(*pend, T, ss);
                            pend.reset();
                            absorb(T, ss);
                        };
                        auto avail = [&]() -> u64 {
                            size_t free_b = 0, total_b = 0;
                            if (hipMemGetInfo(&free_b, &total_b) != hipSuccess) (void)hipGetLastError();
                            return free_b + pool_for(ctl->device).cached_bytes();
                        };
                        bool lean = false;
                        auto launch = [&](u32 k) {
                            const bool bound_only = so.mode == CLB_SPGEMM_BOUND;
                            return spg::one_pass_launch(ctl, Y, Z, hc[k], hc[k + 1], false, bound_only, nullptr, lean);
                        };
                        auto nonempty = [&](u32 k) {  // the first block from k with rows
                            while (k < nb && hc[k + 1] <= hc[k]) ++k;
                            return k;
                        };
                        for (u32 k = nonempty(0); k < nb;) try {
                            if (!cur) {
                                if (pend && avail() < 3 * spg::one_pass_bytes(*pend)) finish_pending();
                                cur = launch(k);
                            }
                            const u32 k2 = nonempty(k + 1);
                            if (k2 < nb) {
                                const u64 mine = spg::one_pass_bytes(*cur) + 4 * hb[k];
                                const u64 need = std::max<u64>(pend ? spg::one_pass_bytes(*pend) : 0, mine);
                                if (avail() >= 2 * need) nxt = launch(k2);
                            }
                            spg::one_pass_post(*cur);
                            if (pend) finish_pending();
                            pend = std::move(cur);
                            cur = std::move(nxt);
                            k = k2;
                        } catch (const Error &e) {
                            // block k (or the one after it) again, alone and lean
                            if (!no_room(e) || lean) throw;
                            nxt.reset();
                            cur.reset();
                            if (pend) finish_pending();
                            make_room(ctl);
                            lean = true;
                        }
                        if (pend) finish_pending();
                    }
                }
            } catch (...) {
                settle(ctl);
                release_all();
                clb_dcsr_release(&Y);
                clb_dcsr_release(&Z);
                throw;
            }
            clb_dcsr_release(&Y);
            clb_dcsr_release(&Z);
            sync(ctl);
            t_prod = std::chrono::steady_clock::now();
            try {
                unite_products(ctl, mats, xs, triples, ntriples, n, prods, splits);
                sync(ctl);
            } catch (...) {
                settle(ctl);
                release_all();
                throw;
            }
            release_all();
        }
        for (u32 k = 0; k < nmats; ++k)
            if (mats[k].nnz != before[k]) {
                ++st.changed;
                st.added += mats[k].nnz - before[k];
            }
        sync(ctl);
        const auto t1 = std::chrono::steady_clock::now();
        st.ms = std::chrono::duration<double, std::milli>(t1 - t0).count();
        st.ms_products = std::chrono::duration<double, std::milli>(t_prod - t0).count();
        st.ms_unions = std::chrono::duration<double, std::milli>(t1 - t_prod).count();
        if (stats) *stats = st;
    });
}

}  // extern "C"
