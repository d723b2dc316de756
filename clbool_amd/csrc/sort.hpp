// sort.hpp -- pair-key sort and union helpers shared by the COO/CSR/DCSR
// operations.
#pragma once

#include "clb_internal.hpp"

namespace clb {

// Stable sorts of pairs (row, col), over only the bits that the largest row
// and column need.  sort_pairs_to_keys: two arrays to sorted keys.
// sort_pairs: two arrays to two arrays (which may be the same), by_row_only:
// stable by row alone.
void sort_pairs_to_keys(clb_controls_s *ctl, const u32 *rows, const u32 *cols, u64 n, u32 max_row, u32 max_col,
                        u64 *keys);
void sort_pairs(clb_controls_s *ctl, const u32 *rows, const u32 *cols, u64 n, u32 max_row, u32 max_col,
                bool by_row_only, u32 *out_rows, u32 *out_cols);
void pack_pairs(clb_controls_s *ctl, const u32 *rows, const u32 *cols, u64 n, u64 *keys);
void pair_bounds(clb_controls_s *ctl, const u32 *rows, const u32 *cols, u64 n, u32 *max_row, u32 *max_col);
// Sorted keys -> new deduplicated (rows, cols) buffers; returns their length.
u32 unique_keys_to_pairs(clb_controls_s *ctl, const u64 *keys, u64 n, clb_buffer_s **rows_out,
                         clb_buffer_s **cols_out);
// Merge of two ascending key lists into out[0, na + nb) (merge path, kept
// duplicates).
void merge_keys(clb_controls_s *ctl, const u64 *a, u64 na, const u64 *b, u64 nb, u64 *out);
// Union of two ascending key lists that hold the rows of mats.size() n x n
// matrices, matrix x in rows [x * n, (x + 1) * n): mats[x] (what the first
// list was made from; only its nnz is read) is replaced by a new matrix when
// the union has more nonzeros, and left alone otherwise.  The caller releases
// what was replaced.
void union_keys_to_matrices(clb_controls_s *ctl, const u64 *ka, u64 na, const u64 *kb, u64 nb, u32 n,
                            std::vector<clb_dcsr> &mats);
void coo_finish(clb_controls_s *ctl, clb_buffer_s *rows, clb_buffer_s *cols, u32 nrows, u32 ncols, u32 nnz,
                bool sorted, bool nodup, clb_coo &out);

// COO rows -> DCSR rpt/rows (create_rows_pointers, matrices_conversions.cpp:7-37).
void rows_to_dcsr(clb_controls_s *ctl, const u32 *rows, u32 nnz, clb_buffer_s **rpt_out, clb_buffer_s **rows_out,
                  u32 *nzr_out);
// DCSR rpt/rows -> per-nonzero row ids (dscr_to_coo.cl:8-23).
void dcsr_expand_rows(clb_controls_s *ctl, const u32 *rpt, const u32 *rows, u32 nzr, u32 nnz, u32 *out_rows);

}  // namespace clb
