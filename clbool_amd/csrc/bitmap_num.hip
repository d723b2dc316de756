// bitmap_num.hip -- the bitmap kernels of the SpGEMM in numeric (columns at exact places) mode.
#include "bitmap_launch.hpp"

namespace clb {
namespace spg {

void launch_bitmap_num(clb_controls_s *ctl, hipStream_t st, const Setup &s, const u32 *perm, u32 r0, u32 n, u32 bits,
                       bool wide, const Out &o) {
    launch_bitmap_mode<NUM>(ctl, st, s, perm, r0, n, bits, wide, o);
}

}  // namespace spg
}  // namespace clb
