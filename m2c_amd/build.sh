#!/bin/bash
# Builds libm2c_amd.so (gfx950) in-tree.  No FMA contraction and no fast-math:
# results must match the reference's non-contracted x86-64 arithmetic bit for
# bit.  Packed-FP32 instructions are disabled: some of their forms have given
# wrong results on this hardware.
set -e
cd "$(dirname "$0")"
HIPCC=${HIPCC:-/opt/rocm/bin/hipcc}
FLAGS="--offload-arch=gfx950 -O3 -std=c++17 -fPIC -ffp-contract=off -fno-fast-math
  -Xclang -target-feature -Xclang -packed-fp32-ops
  -Wall -Wno-unused-variable -Wno-unused-but-set-variable -Wno-unused-value -Wno-unused-result
  -Wno-bitwise-instead-of-logical -I../include"
mkdir -p build
pids=()
UNITS="m2c_capi m2c_stage m2c_stage_u m2c_stage_ur m2c_stage_ug"
for unit in $UNITS; do
  $HIPCC $FLAGS -c -o build/$unit.o csrc/$unit.hip "$@" &
  pids+=($!)
done
for p in "${pids[@]}"; do wait "$p"; done
$HIPCC --offload-arch=gfx950 -fPIC -shared -o libm2c_amd.so.tmp $(printf 'build/%s.o ' $UNITS)
# replace the library in one step, so that a reader never sees a partial file
mv -f libm2c_amd.so.tmp libm2c_amd.so
# C++ facades with the reference's SpaceVariable3D / SpaceOperator /
# TimeIntegrator signatures over the C ABI (host code only), and the test
# driver that runs the reference's time loop through them.
CXX=${CXX:-g++}
$CXX -O2 -std=c++17 -fPIC -shared -Wall -Wextra -I../include -o libm2c_amd_facade.so.tmp facade/m2c_facade.cpp \
  -L. -lm2c_amd -Wl,-rpath,'$ORIGIN'
mv -f libm2c_amd_facade.so.tmp libm2c_amd_facade.so
$CXX -O2 -std=c++17 -fPIC -shared -Wall -Wextra -I../include -o ../tests/libfacade_driver.so.tmp \
  ../tests/facade_driver.cpp -L. -lm2c_amd_facade -lm2c_amd -Wl,-rpath,'$ORIGIN/../m2c_amd'
mv -f ../tests/libfacade_driver.so.tmp ../tests/libfacade_driver.so
# the quotients and roots of m2c_exactdiv.h over arrays, for their test
$HIPCC $FLAGS -shared -o ../tests/libexactdiv.so.tmp ../tests/exactdiv_driver.hip
mv -f ../tests/libexactdiv.so.tmp ../tests/libexactdiv.so
