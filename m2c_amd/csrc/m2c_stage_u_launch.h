// Launches of the stage kernel of tiles of one material, for a translation
// unit that compiles it for HLLC or for the other fluxes.
#pragma once
#include "m2c_stage_launch.h"
#include "m2c_stage_u.h"

namespace m2c {

template <int V>
struct Tile {
  static constexpr int X = kTiles[V].bx, Y = kTiles[V].by, Z = kTiles[V].bz, NT = X * Y * Z;
};

template <int V, bool HLLC>
static void launch(const StageArgs& a, int mode, hipStream_t st) {
  using T = Tile<V>;
  const dim3 grid = stage_grid(stage_tiles(a.g, T::X, T::Y, T::Z));
  switch (mode) {
    case MODE_RESIDUAL: k_stage_u<MODE_RESIDUAL, T::X, T::Y, T::Z, HLLC, false><<<grid, T::NT, 0, st>>>(a); break;
    case MODE_STAGE1: k_stage_u<MODE_STAGE1, T::X, T::Y, T::Z, HLLC, false><<<grid, T::NT, 0, st>>>(a); break;
    case MODE_RK2_FINAL: k_stage_u<MODE_RK2_FINAL, T::X, T::Y, T::Z, HLLC, false><<<grid, T::NT, 0, st>>>(a); break;
    case MODE_RK3_STAGE2: k_stage_u<MODE_RK3_STAGE2, T::X, T::Y, T::Z, HLLC, false><<<grid, T::NT, 0, st>>>(a); break;
    case MODE_RK3_FINAL: k_stage_u<MODE_RK3_FINAL, T::X, T::Y, T::Z, HLLC, false><<<grid, T::NT, 0, st>>>(a); break;
    case MODE_FE: k_stage_u<MODE_FE, T::X, T::Y, T::Z, HLLC, false><<<grid, T::NT, 0, st>>>(a); break;
  }
}

template <int V, bool HLLC>
static void launch_multi(const StageArgs* tab, const int* toff, int nm, int ntiles, int mode, hipStream_t st) {
  using T = Tile<V>;
  const dim3 grid = stage_grid(ntiles);
  switch (mode) {
    case MODE_STAGE1: k_stage_u_multi<MODE_STAGE1, T::X, T::Y, T::Z, HLLC, false><<<grid, T::NT, 0, st>>>(tab, toff, nm); break;
    case MODE_RK2_FINAL: k_stage_u_multi<MODE_RK2_FINAL, T::X, T::Y, T::Z, HLLC, false><<<grid, T::NT, 0, st>>>(tab, toff, nm); break;
    case MODE_RK3_STAGE2: k_stage_u_multi<MODE_RK3_STAGE2, T::X, T::Y, T::Z, HLLC, false><<<grid, T::NT, 0, st>>>(tab, toff, nm); break;
    case MODE_RK3_FINAL: k_stage_u_multi<MODE_RK3_FINAL, T::X, T::Y, T::Z, HLLC, false><<<grid, T::NT, 0, st>>>(tab, toff, nm); break;
  }
}

template <bool HLLC>
static void launch_shape(const StageArgs& a, int mode, int variant, hipStream_t st) {
  switch (variant) {
    case 1: launch<1, HLLC>(a, mode, st); break;
    case 2: launch<2, HLLC>(a, mode, st); break;
    case 3: launch<3, HLLC>(a, mode, st); break;
    default: launch<0, HLLC>(a, mode, st); break;
  }
}

template <bool HLLC>
static void launch_shape_multi(const StageArgs* tab, const int* toff, int nm, int ntiles, int mode, int variant,
                               hipStream_t st) {
  switch (variant) {
    case 1: launch_multi<1, HLLC>(tab, toff, nm, ntiles, mode, st); break;
    case 2: launch_multi<2, HLLC>(tab, toff, nm, ntiles, mode, st); break;
    case 3: launch_multi<3, HLLC>(tab, toff, nm, ntiles, mode, st); break;
    default: launch_multi<0, HLLC>(tab, toff, nm, ntiles, mode, st); break;
  }
}

}  // namespace m2c
