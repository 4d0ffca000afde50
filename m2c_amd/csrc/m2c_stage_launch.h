// Launches of the fused stage kernels, which have translation units of their
// own (m2c_stage.hip: the general kernel; m2c_stage_u.hip, m2c_stage_ur.hip,
// m2c_stage_ug.hip: tiles of one material), so that they build beside the rest
// of the library.  `variant`: tile shape, an index of kTiles.
#pragma once
#include "m2c_stage.h"

namespace m2c {

// Tile shapes the autotuner chooses from (all 256 threads).
struct TileVariant {
  int bx, by, bz;
};
constexpr int kNumTiles = M2CX_NUM_TILES;
constexpr TileVariant kTiles[kNumTiles] = {{16, 4, 4}, {32, 4, 2}, {8, 8, 4}, {16, 8, 2}};
// the shape for reconstruction in conservative or characteristic variables: the
// one with the fewest cells around a tile
constexpr int kGenTile = 2;

// one work-group per tile, padded to a multiple of the XCD count (xcd_tile)
inline dim3 stage_grid(long ntiles) { return dim3((unsigned)((ntiles + NXCD - 1) / NXCD * NXCD)); }
inline long stage_tiles(const DevGrid& g, int bx, int by, int bz) {
  return (long)((g.NX + bx - 1) / bx) * ((g.NY + by - 1) / by) * ((g.NZ + bz - 1) / bz);
}

// the general kernel: primitive variables, or (gen) any, on kTiles[kGenTile]
void stage_launch(const StageArgs& a, int mode, int variant, hipStream_t st);
void stage_launch_gen(const StageArgs& a, int mode, hipStream_t st);
// the members of an ensemble: argument table and prefix sums of their tiles
void stage_launch_multi(const StageArgs* tab, const int* toff, int nm, int ntiles, int mode, int variant,
                        hipStream_t st);
// slot of the material tables in each unit's constant memory (enqueued on st)
hipError_t stage_set_materials(int slot, const DevMats& m, hipStream_t st);

// tiles of one material (those that a.tflag, when given, does not mark), for
// the HLLC flux and for the others
void ustage_launch_hllc(const StageArgs& a, int mode, int variant, hipStream_t st);
void ustage_launch_other(const StageArgs& a, int mode, int variant, hipStream_t st);
void ustage_launch_multi_hllc(const StageArgs* tab, const int* toff, int nm, int ntiles, int mode, int variant,
                              hipStream_t st);
void ustage_launch_multi_other(const StageArgs* tab, const int* toff, int nm, int ntiles, int mode, int variant,
                               hipStream_t st);
// reconstruction in conservative or characteristic variables
void ustage_launch_gen(const StageArgs& a, int mode, hipStream_t st);
// the marks of k_recon_flags on the tiles of one material
void recon_flags_launch_u(const StageArgs& a, unsigned char* flag, hipStream_t st);
hipError_t ustage_set_materials_gen(int slot, const DevMats& m, hipStream_t st);
hipError_t ustage_set_materials_hllc(int slot, const DevMats& m, hipStream_t st);
hipError_t ustage_set_materials_other(int slot, const DevMats& m, hipStream_t st);

}  // namespace m2c
