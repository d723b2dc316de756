// bitmap_launch.hpp -- launches of the bitmap kernels in one mode.  Each mode
// has a source file of its own (bitmap_sym.hip, bitmap_num.hip,
// bitmap_one.hip): the instantiations compile side by side.
#pragma once

#include "spgemm.hpp"

namespace clb {
namespace spg {

// Packed B serves a window when its groups tell the window's columns: always
// up to 2^20 columns, above through slices no wider than the window.
static bool use_packs(const Mats &g, u32 bits) {
    return g.b_packs && (g.ncols <= (1u << 20) || (g.psplits && bits >= g.split_bits));
}

// One workgroup per row, or (tuning.bitmap_persistent) a persistent grid that
// takes rows from a counter.
template <int WBITS, int WG, int MODE, bool COMB>
static void launch_bitmap_c(clb_controls_s *ctl, hipStream_t st, const Setup &s, const u32 *perm, u32 r0, u32 n,
                            const Out &o) {
    if (!ctl->tuning.bitmap_persistent) {
        if constexpr (!COMB) {
            if (use_packs(s.g, WBITS)) {
                k_bitmap<WBITS, WG, MODE, false, true><<<n, WG, 0, st>>>(s.g, perm, r0, o);
                return;
            }
        }
        k_bitmap<WBITS, WG, MODE, COMB, false><<<n, WG, 0, st>>>(s.g, perm, r0, o);
        return;
    }
    int per_cu = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_bitmap_persist<WBITS, WG, MODE, COMB>, WG, 0) !=
            hipSuccess ||
        per_cu < 1) {
        (void)hipGetLastError();
        per_cu = 1;
    }
    const u64 fit = (u64)ctl->cu_count * (u64)per_cu;
    u32 *ctr = s.ctr.ptr + MODE;  // one counter per pass of the SpGEMM
    fill_u32_on(st, ctr, 1, 0u);
    k_bitmap_persist<WBITS, WG, MODE, COMB><<<(u32)(n < fit ? n : fit), WG, 0, st>>>(s.g, perm, n, ctr, o);
}

template <int WBITS, int MODE>
static void launch_bitmap_w(clb_controls_s *ctl, hipStream_t st, const Setup &s, const u32 *perm, u32 r0, u32 n,
                            bool wide, const Out &o) {
    constexpr int WG = (int)bitmap_wg(WBITS), WIDE = (int)bitmap_wide(WBITS);
    if constexpr (WIDE > WG) {
        if (wide) {
            if (use_packs(s.g, WBITS)) k_bitmap<WBITS, WIDE, MODE, false, true><<<n, WIDE, 0, st>>>(s.g, perm, r0, o);
            else k_bitmap<WBITS, WIDE, MODE, false, false><<<n, WIDE, 0, st>>>(s.g, perm, r0, o);
            return;
        }
    }
    if (s.g.combine) launch_bitmap_c<WBITS, WG, MODE, true>(ctl, st, s, perm, r0, n, o);
    else launch_bitmap_c<WBITS, WG, MODE, false>(ctl, st, s, perm, r0, n, o);
}

template <int MODE>
static void launch_bitmap_mode(clb_controls_s *ctl, hipStream_t st, const Setup &s, const u32 *perm, u32 r0, u32 n,
                               u32 bits, bool wide, const Out &o) {
    switch (bits) {
        case 6: launch_bitmap_w<6, MODE>(ctl, st, s, perm, r0, n, wide, o); break;
        case 7: launch_bitmap_w<7, MODE>(ctl, st, s, perm, r0, n, wide, o); break;
        case 8: launch_bitmap_w<8, MODE>(ctl, st, s, perm, r0, n, wide, o); break;
        case 9: launch_bitmap_w<9, MODE>(ctl, st, s, perm, r0, n, wide, o); break;
        case 10: launch_bitmap_w<10, MODE>(ctl, st, s, perm, r0, n, wide, o); break;
        case 11: launch_bitmap_w<11, MODE>(ctl, st, s, perm, r0, n, wide, o); break;
        case 12: launch_bitmap_w<12, MODE>(ctl, st, s, perm, r0, n, wide, o); break;
        case 13: launch_bitmap_w<13, MODE>(ctl, st, s, perm, r0, n, wide, o); break;
        case 14: launch_bitmap_w<14, MODE>(ctl, st, s, perm, r0, n, wide, o); break;
        case 15: launch_bitmap_w<15, MODE>(ctl, st, s, perm, r0, n, wide, o); break;
    }
}

}  // namespace spg
}  // namespace clb
