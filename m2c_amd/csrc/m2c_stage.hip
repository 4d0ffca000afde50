// Launches of the general stage kernel.
#include <hip/hip_runtime.h>
#include "m2c_stage.h"
#include "m2c_stage_launch.h"

namespace m2c {

template <int V>
struct Tile {
  static constexpr int X = kTiles[V].bx, Y = kTiles[V].by, Z = kTiles[V].bz, NT = X * Y * Z;
};

template <int V, bool GEN>
static void launch(const StageArgs& a, int mode, hipStream_t st) {
  using T = Tile<V>;
  const dim3 grid = stage_grid(stage_tiles(a.g, T::X, T::Y, T::Z));
  switch (mode) {
    case MODE_RESIDUAL: k_stage<MODE_RESIDUAL, T::X, T::Y, T::Z, GEN><<<grid, T::NT, 0, st>>>(a); break;
    case MODE_STAGE1: k_stage<MODE_STAGE1, T::X, T::Y, T::Z, GEN><<<grid, T::NT, 0, st>>>(a); break;
    case MODE_RK2_FINAL: k_stage<MODE_RK2_FINAL, T::X, T::Y, T::Z, GEN><<<grid, T::NT, 0, st>>>(a); break;
    case MODE_RK3_STAGE2: k_stage<MODE_RK3_STAGE2, T::X, T::Y, T::Z, GEN><<<grid, T::NT, 0, st>>>(a); break;
    case MODE_RK3_FINAL: k_stage<MODE_RK3_FINAL, T::X, T::Y, T::Z, GEN><<<grid, T::NT, 0, st>>>(a); break;
    case MODE_FE: k_stage<MODE_FE, T::X, T::Y, T::Z, GEN><<<grid, T::NT, 0, st>>>(a); break;
  }
}

template <int V>
static void launch_multi(const StageArgs* tab, const int* toff, int nm, int ntiles, int mode, hipStream_t st) {
  using T = Tile<V>;
  const dim3 grid = stage_grid(ntiles);
  switch (mode) {
    case MODE_STAGE1: k_stage_multi<MODE_STAGE1, T::X, T::Y, T::Z><<<grid, T::NT, 0, st>>>(tab, toff, nm); break;
    case MODE_RK2_FINAL: k_stage_multi<MODE_RK2_FINAL, T::X, T::Y, T::Z><<<grid, T::NT, 0, st>>>(tab, toff, nm); break;
    case MODE_RK3_STAGE2: k_stage_multi<MODE_RK3_STAGE2, T::X, T::Y, T::Z><<<grid, T::NT, 0, st>>>(tab, toff, nm); break;
    case MODE_RK3_FINAL: k_stage_multi<MODE_RK3_FINAL, T::X, T::Y, T::Z><<<grid, T::NT, 0, st>>>(tab, toff, nm); break;
  }
}

void stage_launch(const StageArgs& a, int mode, int variant, hipStream_t st) {
  switch (variant) {
    case 1: launch<1, false>(a, mode, st); break;
    case 2: launch<2, false>(a, mode, st); break;
    case 3: launch<3, false>(a, mode, st); break;
    default: launch<0, false>(a, mode, st); break;
  }
}

void stage_launch_gen(const StageArgs& a, int mode, hipStream_t st) { launch<kGenTile, true>(a, mode, st); }

void stage_launch_multi(const StageArgs* tab, const int* toff, int nm, int ntiles, int mode, int variant,
                        hipStream_t st) {
  switch (variant) {
    case 1: launch_multi<1>(tab, toff, nm, ntiles, mode, st); break;
    case 2: launch_multi<2>(tab, toff, nm, ntiles, mode, st); break;
    case 3: launch_multi<3>(tab, toff, nm, ntiles, mode, st); break;
    default: launch_multi<0>(tab, toff, nm, ntiles, mode, st); break;
  }
}

hipError_t stage_set_materials(int slot, const DevMats& m, hipStream_t st) {
  return hipMemcpyToSymbolAsync(HIP_SYMBOL(c_mats), &m, sizeof(DevMats), slot * sizeof(DevMats), hipMemcpyHostToDevice,
                                st);
}

}  // namespace m2c
