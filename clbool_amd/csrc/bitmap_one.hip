// bitmap_one.hip -- the bitmap kernels of the SpGEMM in one-pass (columns in slots of given capacity) mode.
#include "bitmap_launch.hpp"

namespace clb {
namespace spg {

void launch_bitmap_one(clb_controls_s *ctl, hipStream_t st, const Setup &s, const u32 *perm, u32 r0, u32 n, u32 bits,
                       bool wide, const Out &o) {
    launch_bitmap_mode<ONE>(ctl, st, s, perm, r0, n, bits, wide, o);
}

}  // namespace spg
}  // namespace clb
