// bitmap_sym.hip -- the bitmap kernels of the SpGEMM in symbolic (sizes) mode.
#include "bitmap_launch.hpp"

namespace clb {
namespace spg {

void launch_bitmap_sym(clb_controls_s *ctl, hipStream_t st, const Setup &s, const u32 *perm, u32 r0, u32 n, u32 bits,
                       bool wide, const Out &o) {
    launch_bitmap_mode<SYM>(ctl, st, s, perm, r0, n, bits, wide, o);
}

}  // namespace spg
}  // namespace clb
