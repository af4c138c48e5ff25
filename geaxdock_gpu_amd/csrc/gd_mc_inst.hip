// gd_mc_inst.hip -- the MC kernel instances of one atoms-per-lane count,
// GD_MC_APL (set by the build: this file is compiled once per count, so the
// instances build in parallel). Each instance keeps only the registers its
// lane shape needs.
#include "gd_mc.h"

namespace gd {

// Host handle of gd_mc_kernel<GD_MC_APL, da, ...>: da 0 plain MC and pose
// evaluation, 1 delayed acceptance with the network per atom, 2 with its
// tabulated outputs, 3 and 4 the same with the receptor split's groups
// sharing the surrogate's KDE and MCS sums, DA_TREE plain MC by a tree of
// energies, DA_POSES poses with fewer lanes than the complex's shape; DA_NEAR
// added: without the distance tests; rec: the receptor resident in LDS by
// chunks, streamed through LDS tiles, or resident with unit lists.
template <>
const void *mc_kernel_handle<GD_MC_APL>(int da, int rec) {
  if (da & DA_NEAR) {
    switch (rec == REC_CHUNKS ? da : rec == REC_TILED && da == DA_NEAR ? -1 : -2) {
      case DA_NEAR: return (const void *)gd_mc_kernel<GD_MC_APL, DA_NEAR, false, false>;
      case DA_NEAR + 2: return (const void *)gd_mc_kernel<GD_MC_APL, DA_NEAR + 2, false, false>;
      case DA_NEAR + 4: return (const void *)gd_mc_kernel<GD_MC_APL, DA_NEAR + 4, false, false>;
      case -1: return (const void *)gd_mc_kernel<GD_MC_APL, DA_NEAR, true, false>;
      default: da &= ~DA_NEAR;
    }
  }
  if (rec == REC_TILED) {
    switch (da) {
      case 1: return (const void *)gd_mc_kernel<GD_MC_APL, 1, true, false>;
      case 2: return (const void *)gd_mc_kernel<GD_MC_APL, 2, true, false>;
      case 3: return (const void *)gd_mc_kernel<GD_MC_APL, 3, true, false>;
      case 4: return (const void *)gd_mc_kernel<GD_MC_APL, 4, true, false>;
      case DA_TREE: return (const void *)gd_mc_kernel<GD_MC_APL, DA_TREE, true, false>;
#if GD_MC_APL == 2 || GD_MC_APL == 3
      case DA_POSES: return (const void *)gd_mc_kernel<GD_MC_APL, DA_POSES, true, false>;
#endif
#if GD_MC_APL == 3
      case DA_POSES2: return (const void *)gd_mc_kernel<GD_MC_APL, DA_POSES2, true, false>;
#endif
      default: return (const void *)gd_mc_kernel<GD_MC_APL, 0, true, false>;
    }
  }
  if (rec == REC_FLAT) {
    switch (da) {
      case 0: return (const void *)gd_mc_kernel<GD_MC_APL, 0, false, true>;
      case 2: return (const void *)gd_mc_kernel<GD_MC_APL, 2, false, true>;
      case 4: return (const void *)gd_mc_kernel<GD_MC_APL, 4, false, true>;
      case DA_TREE: return (const void *)gd_mc_kernel<GD_MC_APL, DA_TREE, false, true>;
#if GD_MC_APL == 2 || GD_MC_APL == 3
      case DA_POSES: return (const void *)gd_mc_kernel<GD_MC_APL, DA_POSES, false, true>;
#endif
#if GD_MC_APL == 3
      case DA_POSES2: return (const void *)gd_mc_kernel<GD_MC_APL, DA_POSES2, false, true>;
#endif
      default: return nullptr;
    }
  }
  switch (da) {
    case 1: return (const void *)gd_mc_kernel<GD_MC_APL, 1, false, false>;
    case 2: return (const void *)gd_mc_kernel<GD_MC_APL, 2, false, false>;
    case 3: return (const void *)gd_mc_kernel<GD_MC_APL, 3, false, false>;
    case 4: return (const void *)gd_mc_kernel<GD_MC_APL, 4, false, false>;
    case DA_TREE: return (const void *)gd_mc_kernel<GD_MC_APL, DA_TREE, false, false>;
    default: return (const void *)gd_mc_kernel<GD_MC_APL, 0, false, false>;
  }
}

}  // namespace gd
