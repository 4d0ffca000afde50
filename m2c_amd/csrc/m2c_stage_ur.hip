// The stage kernel of tiles of one material, Roe and LLF fluxes.
#include <hip/hip_runtime.h>
#include "m2c_stage_u_launch.h"

namespace m2c {

void ustage_launch_other(const StageArgs& a, int mode, int variant, hipStream_t st) {
  launch_shape<false>(a, mode, variant, st);
}
void ustage_launch_multi_other(const StageArgs* tab, const int* toff, int nm, int ntiles, int mode, int variant,
                              hipStream_t st) {
  launch_shape_multi<false>(tab, toff, nm, ntiles, mode, variant, st);
}
hipError_t ustage_set_materials_other(int slot, const DevMats& m, hipStream_t st) {
  return hipMemcpyToSymbolAsync(HIP_SYMBOL(c_mats), &m, sizeof(DevMats), slot * sizeof(DevMats), hipMemcpyHostToDevice,
                                st);
}

}  // namespace m2c
