// D3Q27 cumulant collision for cumulant sets other than the default polynomial one (the relaxation as linear
// maps from the method table), FP32 arithmetic: the sweep kernels of this family and compute type for every streaming
// pattern (templates in sweep_kernel.h and sweep_eso_kernel.h).
#include "sweep_eso_kernel.h"
#include "sweep_kernel.h"

namespace lbm355 {

void* pick_sweep_cumulant_general_f32(int stencil, int store, int pat, bool walls, int mode) {
  if (stencil != LBM355_D3Q27) return nullptr;
  return pick_store<D3Q27, FAMILY_CUMULANT_GENERAL, float>(store, pat, walls, mode);
}

void* eso_pick_cumulant_general_f32(int stencil, int store, int pat, int mode) {
  if (stencil != LBM355_D3Q27) return nullptr;
  return eso_pick_store<D3Q27, FAMILY_CUMULANT_GENERAL, float>(store, pat, mode);
}

}  // namespace lbm355
