// D3Q27 cumulant collision with Galilean / fourth-order corrections, FP32 arithmetic: the sweep kernels of this family and compute type for every streaming pattern
// (templates in sweep_kernel.h and sweep_eso_kernel.h).
#include "sweep_eso_kernel.h"
#include "sweep_kernel.h"

namespace lbm355 {

void* pick_sweep_cumulant_corrected_f32(int stencil, int store, int pat, bool walls, int mode) {
  if (stencil != LBM355_D3Q27) return nullptr;
  return pick_store<D3Q27, FAMILY_CUMULANT_CORRECTED, float>(store, pat, walls, mode);
}

void* eso_pick_cumulant_corrected_f32(int stencil, int store, int pat, int mode) {
  if (stencil != LBM355_D3Q27) return nullptr;
  return eso_pick_store<D3Q27, FAMILY_CUMULANT_CORRECTED, float>(store, pat, mode);
}

}  // namespace lbm355
