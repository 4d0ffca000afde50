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

// k_recon_flags on the tiles of one material of a uniform mesh: the general
// code takes each neighbour's material from memory and handles its equation of
// state at run time, at 112 B of scratch per lane; here there is one material
// and a copy of the code per type of equation of state (191x97x61 water,
// conservative-characteristic: 171 -> 106 us, bound by the FP64 arithmetic).
// Three waves per SIMD at five spilled registers; two without: 118 us.
__device__ __forceinline__ void recon_flag(const StageArgs& a, const DevEos E, int i, int j, int k,
                                           unsigned char* __restrict__ flag) {
  const Scheme& s = a.s;
  const long c = gidx(a.g, i, j, k);
  double v[5];
  load5(a.Vin, c, v);
  bool fails = false, ok = true;
#pragma unroll 1
  for (int D = 0; D < 3; D++) {
    const long st = axis_stride(a.g, D);
    double vm[5], vp[5], q0[5], h[5], f[5];
    load5(a.Vin, c - st, vm);
    load5(a.Vin, c + st, vp);
    ok = slopes_in_vars(E, s, D, v, vm, vp, q0, h) && ok;
    face_from_vars(E, s, q0, h, true, f);
    fails = fails || eos_check5(E, f);
    face_from_vars(E, s, q0, h, false, f);
    fails = fails || eos_check5(E, f);
  }
  flag[c] = fails ? 1 : 0;
  if (!ok) atomicOr(&a.cnt->error, 1);
}
template <int BX, int BY, int BZ>
__global__ void __launch_bounds__(BX * BY * BZ, 3) k_recon_flags_u(StageArgs a, unsigned char* __restrict__ flag) {
  const DevGrid& g = a.g;
  const int ntx = (g.NX + BX - 1) / BX, nty = (g.NY + BY - 1) / BY, ntiles = ntx * nty * ((g.NZ + BZ - 1) / BZ);
  const int tile = xcd_tile(ntiles);
  if (tile >= ntiles || (a.tflag && a.tflag[tile])) return;
  const int t = threadIdx.x, ib = (tile % ntx) * BX, jb = ((tile / ntx) % nty) * BY, kb = (tile / (ntx * nty)) * BZ;
  const int i = ib + t % BX, j = jb + (t / BX) % BY, k = kb + t / (BX * BY);
  if (i >= g.NX || j >= g.NY || k >= g.NZ) return;
  const int id = __builtin_amdgcn_readfirstlane((int)a.ID[gidx(g, ib, jb, kb)]);
  const DevEos E = c_mats[a.s.mset].m[id];
  if (E.type == M2CX_EOS_SG) recon_flag(a, E, i, j, k, flag);
  else if (E.type == M2CX_EOS_NASG) recon_flag(a, E, i, j, k, flag);
  else recon_flag(a, E, i, j, k, flag);
}
void recon_flags_launch_u(const StageArgs& a, unsigned char* flag, hipStream_t st) {
  constexpr int X = kTiles[kGenTile].bx, Y = kTiles[kGenTile].by, Z = kTiles[kGenTile].bz;
  k_recon_flags_u<X, Y, Z><<<stage_grid(stage_tiles(a.g, X, Y, Z)), X * Y * Z, 0, st>>>(a, flag);
}
hipError_t ustage_set_materials_gen(int slot, const DevMats& m, hipStream_t st) {
  return hipMemcpyToSymbolAsync(HIP_SYMBOL(c_mats), &m, sizeof(DevMats), slot * sizeof(DevMats), hipMemcpyHostToDevice,
                                st);
}

}  // namespace m2c
