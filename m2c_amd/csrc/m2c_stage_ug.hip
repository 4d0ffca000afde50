// The stage kernel of tiles of one material, reconstruction in conservative
// or characteristic variables (one tile shape, kTiles[kGenTile]).
#include <hip/hip_runtime.h>
#include "m2c_stage_launch.h"
#include "m2c_stage_u.h"

namespace m2c {

template <bool HLLC>
static void launch(const StageArgs& a, int mode, hipStream_t st) {
  constexpr int X = kTiles[kGenTile].bx, Y = kTiles[kGenTile].by, Z = kTiles[kGenTile].bz, NT = X * Y * Z;
  const dim3 grid = stage_grid(stage_tiles(a.g, X, Y, Z));
  switch (mode) {
    case MODE_RESIDUAL: k_stage_u<MODE_RESIDUAL, X, Y, Z, HLLC, true><<<grid, NT, 0, st>>>(a); break;
    case MODE_STAGE1: k_stage_u<MODE_STAGE1, X, Y, Z, HLLC, true><<<grid, NT, 0, st>>>(a); break;
    case MODE_RK2_FINAL: k_stage_u<MODE_RK2_FINAL, X, Y, Z, HLLC, true><<<grid, NT, 0, st>>>(a); break;
    case MODE_RK3_STAGE2: k_stage_u<MODE_RK3_STAGE2, X, Y, Z, HLLC, true><<<grid, NT, 0, st>>>(a); break;
    case MODE_RK3_FINAL: k_stage_u<MODE_RK3_FINAL, X, Y, Z, HLLC, true><<<grid, NT, 0, st>>>(a); break;
    case MODE_FE: k_stage_u<MODE_FE, X, Y, Z, HLLC, true><<<grid, NT, 0, st>>>(a); break;
  }
}

void ustage_launch_gen(const StageArgs& a, int mode, hipStream_t st) {
  if (a.s.flux == M2CX_FLUX_HLLC) launch<true>(a, mode, st);
  else launch<false>(a, mode, st);
}
hipError_t ustage_set_materials_gen(int slot, const DevMats& m) {
  return hipMemcpyToSymbol(HIP_SYMBOL(c_mats), &m, sizeof(DevMats), slot * sizeof(DevMats));
}

}  // namespace m2c
