// Kernels of the explicit step around the fused stage (gfx950): cell flags,
// boundary fill, clipping, time step, transposes.  See m2c_grid.h for the
// layout.
#pragma once
#include "m2c_stage.h"

namespace m2c {

// Cells whose reconstruction in the scheme's variable type fails CheckState
// on one of their six faces; they are reconstructed in primitive variables
// instead (Reconstructor.cpp:722-778).  c0^2 < 0 in a characteristic
// transform is the reference's abort (FluxFcnBase.h:315-320).
__global__ void k_recon_flags(DevGrid g, Scheme s, CF5 V, const unsigned char* __restrict__ ID,
                              unsigned char* __restrict__ flag, DevCounters* cnt,
                              const unsigned char* __restrict__ mixed, int BX, int BY, int BZ) {
  const DevMats& M = c_mats[s.mset];
  const long n = (long)g.NX * g.NY * g.NZ;
  for (long q = blockIdx.x * (long)blockDim.x + threadIdx.x; q < n; q += (long)gridDim.x * blockDim.x) {
    int i, j, k;
    cell_ijk(g, q, i, j, k);
    if (mixed && !mixed[i / BX + ((g.NX + BX - 1) / BX) * (j / BY + ((g.NY + BY - 1) / BY) * (k / BZ))]) continue;
    const long c = gidx(g, i, j, k);
    const int myid = ID[c];
    if (myid == s.inactive) {
      flag[c] = 0;
      continue;
    }
    const DevEos& E = M.m[myid];
    double v[5];
    load5(V, c, v);
    bool fails = false, ok = true;
#pragma unroll 1
    for (int D = 0; D < 3; D++) {
      double q0[5], sig[5], f[5];
      ok = recon_slope(g, s, M, V, ID, s.var_type, D, i, j, k, v, q0, sig) && ok;
      recon_face(E, s.var_type, v, q0, sig, 0, f);
      fails = fails || eos_check5(E, f);
      recon_face(E, s.var_type, v, q0, sig, 1, f);
      fails = fails || eos_check5(E, f);
    }
    flag[c] = fails ? 1 : 0;
    if (!ok) atomicOr(&cnt->error, 1);
  }
}

// tflag[tile] = 1 where the tile's cells and the two cells around them along
// each axis (the reach of the stage's stencil) do not all hold one active
// material.  One wave per tile; the IDs change once per time step at most, so
// this runs once per step.
__global__ void __launch_bounds__(256) k_tile_mixed(DevGrid g, int inactive, const unsigned char* __restrict__ ID,
                                                    unsigned char* __restrict__ tflag, int BX, int BY, int BZ,
                                                    int ntiles) {
  const int tile = (int)(blockIdx.x * 4 + threadIdx.x / 64), lane = threadIdx.x % 64;
  if (tile >= ntiles) return;
  const int ntx = (g.NX + BX - 1) / BX, nty = (g.NY + BY - 1) / BY;
  const int ib = (tile % ntx) * BX, jb = ((tile / ntx) % nty) * BY, kb = (tile / (ntx * nty)) * BZ;
  const int id0 = ID[gidx(g, ib, jb, kb)];
  bool mixed = id0 == inactive;
  // box D: the tile widened by two cells along axis D, cut to the ghosted brick
#pragma unroll 1
  for (int D = 0; D < 3; D++) {
    const int i0 = D == 0 ? max(ib - 2, -1) : ib, j0 = D == 1 ? max(jb - 2, -1) : jb, k0 = D == 2 ? max(kb - 2, -1) : kb;
    const int i1 = D == 0 ? min(ib + BX + 2, g.NX + 1) : min(ib + BX, g.NX);
    const int j1 = D == 1 ? min(jb + BY + 2, g.NY + 1) : min(jb + BY, g.NY);
    const int k1 = D == 2 ? min(kb + BZ + 2, g.NZ + 1) : min(kb + BZ, g.NZ);
    const int nx = i1 - i0, nxy = nx * (j1 - j0), n = nxy * (k1 - k0);
    for (int q = lane; q < n; q += 64) {
      const int kk = q / nxy, r = q - kk * nxy, jj = r / nx, ii = r - jj * nx;
      mixed = mixed || ID[gidx(g, i0 + ii, j0 + jj, k0 + kk)] != id0;
    }
  }
  const bool any = __any(mixed);
  if (lane == 0) tflag[tile] = any ? 1 : 0;
}

// U = P2C(V) on interior cells, only if the preceding stage clipped a cell
// (TimeIntegrator.cpp:569-572, 622-625).
__global__ void k_resync(DevGrid g, int mset, CF5 V, F5 U, const unsigned char* __restrict__ ID, const DevCounters* cnt) {
  if (cnt->stage_clipped == 0) return;
  long n = (long)g.NX * g.NY * g.NZ;
  for (long q = blockIdx.x * (long)blockDim.x + threadIdx.x; q < n; q += (long)gridDim.x * blockDim.x) {
    int i, j, k;
    cell_ijk(g, q, i, j, k);
    long c = gidx(g, i, j, k);
    double v[5], u[5];
    load5(V, c, v);
    eos_p2c(c_mats[mset].m[ID[c]], v, u);
    store5(U, c, u);
  }
}

__global__ void k_reset_stage(DevCounters* cnt) { cnt->stage_clipped = 0; }
__global__ void k_reset_error(DevCounters* cnt) { cnt->error = 0; }

// SpaceOperator::ApplyBoundaryConditions on a state field (face ghosts)
__global__ void k_apply_bc(DevGrid g, F5 V) {
  long n = (long)g.NX * g.NY * g.NZ;
  for (long q = blockIdx.x * (long)blockDim.x + threadIdx.x; q < n; q += (long)gridDim.x * blockDim.x) {
    int i, j, k;
    cell_ijk(g, q, i, j, k);
    if (i != 0 && i != g.NX - 1 && j != 0 && j != g.NY - 1 && k != 0 && k != g.NZ - 1) continue;
    double v[5];
    CF5 cv{V.b, V.cs};
    load5(cv, gidx(g, i, j, k), v);
    write_ghosts(g, V, i, j, k, v);
  }
}

// ClipDensityAndPressure on interior cells (SpaceOperator.cpp:646-693)
__global__ void k_clip(DevGrid g, int mset, F5 V, const unsigned char* __restrict__ ID, DevCounters* cnt) {
  long n = (long)g.NX * g.NY * g.NZ;
  for (long q = blockIdx.x * (long)blockDim.x + threadIdx.x; q < n; q += (long)gridDim.x * blockDim.x) {
    int i, j, k;
    cell_ijk(g, q, i, j, k);
    long c = gidx(g, i, j, k);
    double v[5];
    for (int p = 0; p < 5; p++) v[p] = V(p, c);
    const DevEos& E = c_mats[mset].m[ID[c]];
    if (eos_clip(E, v)) {
      atomicAdd(&cnt->clipped, 1ull);
      atomicAdd(&cnt->stage_clipped, 1ull);
      for (int p = 0; p < 5; p++) V(p, c) = v[p];
    }
    if (eos_check5(E, v)) atomicOr(&cnt->error, 1);
  }
}

// ---------------------------------------------------------------------------
// Time step (SpaceOperator.cpp:1223-1330 and the loop of Main.cpp:653-712):
// dt = cfl * min over cells and active axes of d_a/(|u_a|+c).  Block minima
// go to `part`; the last block to finish reduces them and, when `advance`,
// clamps dt at MaxTime and moves t, like the driver loop.
// ---------------------------------------------------------------------------
__device__ __forceinline__ double nmin(double a, double b) { return (b < a) ? b : a; }  // std::min(a,b)

__device__ __forceinline__ double wave_min(double m) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) m = nmin(m, __shfl_xor(m, off, 64));
  return m;
}

// Launched with DT_BLOCKS blocks of 256 (grid-stride over the cells): few
// enough partial minima that the last block reduces them in one pass.
constexpr int DT_BLOCKS = 2048;
__global__ void __launch_bounds__(256) k_dt(DevGrid g, Scheme s, CF5 V, const unsigned char* __restrict__ ID,
                                            double* part, DevCounters* cnt, int advance) {
  __shared__ double red[4];
  __shared__ bool last;
  double m = DBL_MAX;
  const long n = (long)g.NX * g.NY * g.NZ;
  const double* dxs = g_axis(g, 3);
  const double* dys = g_axis(g, 4);
  const double* dzs = g_axis(g, 5);
  for (long q = blockIdx.x * (long)blockDim.x + threadIdx.x; q < n; q += (long)gridDim.x * blockDim.x) {
    int i, j, k;
    cell_ijk(g, q, i, j, k);
    long c = gidx(g, i, j, k);
    int id = ID[c];
    if (id == s.inactive) continue;
    const DevEos& E = c_mats[s.mset].m[id];
    double v[5];
    load5(V, c, v);
    double e = eos_e(E, v[0], v[4]);
    double c2 = eos_c2(E, v[0], e);
    if (c2 < 0) atomicOr(&cnt->error, 1);
    double cc = sqrt(c2);
    double lf = fabs(v[1]) + cc, lg = fabs(v[2]) + cc, lh = fabs(v[3]) + cc;
    if (g.NX > 1) m = nmin(m, dxs[i + 1] / lf);
    if (g.NY > 1) m = nmin(m, dys[j + 1] / lg);
    if (g.NZ > 1) m = nmin(m, dzs[k + 1] / lh);
  }
  // min is exact and order-independent: any reduction order gives the same dt
  m = wave_min(m);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    part[blockIdx.x] = nmin(nmin(red[0], red[1]), nmin(red[2], red[3]));
    __threadfence();
    unsigned int tk = atomicAdd(&cnt->dt_ticket, 1u);
    last = (tk == gridDim.x - 1);
  }
  __syncthreads();
  if (!last) return;
  __threadfence();
  double mm = DBL_MAX;
  for (int b = threadIdx.x; b < (int)gridDim.x; b += blockDim.x) mm = nmin(mm, ((volatile double*)part)[b]);
  mm = wave_min(mm);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = mm;
  __syncthreads();
  if (threadIdx.x == 0) red[0] = nmin(nmin(red[0], red[1]), nmin(red[2], red[3]));
  if (threadIdx.x == 0) {
    cnt->dt_ticket = 0;
    double cfl, dt;
    if (s.time_step > 0) {  // Time.TimeStep (SpaceOperator.cpp:1315-1321)
      dt = s.time_step;
      cfl = dt / red[0];
    } else {
      cfl = s.cfl;
      dt = cfl * red[0];
    }
    if (advance) {
      double t = cnt->t, tmax = cnt->tmax;
      if (t + dt > tmax) {
        cfl *= (tmax - t) / dt;
        dt = tmax - t;
      }
      cnt->dts = dt;
      cnt->t = t + dt;
      cnt->time_step += 1;
      cnt->steps += 1;
    }
    cnt->dt = dt;
    cnt->cfl = cfl;
  }
}

// ---------------------------------------------------------------------------
// AoS (reference layout) <-> SoA transposes for upload/download
// ---------------------------------------------------------------------------
__global__ void k_aos_to_soa(const double* __restrict__ src, F5 dst, int dof, long n) {
  for (long c = blockIdx.x * (long)blockDim.x + threadIdx.x; c < n; c += (long)gridDim.x * blockDim.x)
    for (int p = 0; p < dof; p++) dst(p, c) = src[c * dof + p];
}
__global__ void k_soa_to_aos(CF5 src, double* __restrict__ dst, int dof, long n) {
  for (long c = blockIdx.x * (long)blockDim.x + threadIdx.x; c < n; c += (long)gridDim.x * blockDim.x)
    for (int p = 0; p < dof; p++) dst[c * dof + p] = src(p, c);
}
// `seen` becomes `upload`, the number of this field, if a cell holds the
// material `inactive`
__global__ void k_i32_to_u8(const int* __restrict__ src, unsigned char* __restrict__ dst, long n, int inactive,
                            int* seen, int upload) {
  bool any = false;
  for (long c = blockIdx.x * (long)blockDim.x + threadIdx.x; c < n; c += (long)gridDim.x * blockDim.x) {
    dst[c] = (unsigned char)src[c];
    any |= (int)(unsigned char)src[c] == inactive;
  }
  if (any) *seen = upload;
}
__global__ void k_u8_to_i32(const unsigned char* __restrict__ src, int* __restrict__ dst, long n) {
  for (long c = blockIdx.x * (long)blockDim.x + threadIdx.x; c < n; c += (long)gridDim.x * blockDim.x)
    dst[c] = src[c];
}

// Batched numerical flux (FluxFcnBase::ComputeNumericalFluxAtCellInterface)
__global__ void k_flux_batch(Scheme s, int n, int d, const double* Vm, const double* Vp, const int* id, double* F,
                             DevCounters* cnt) {
  int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= n) return;
  int err = 0;
  flux_num(c_mats[s.mset].m[id[q]], s.flux, s.del, d, Vm + 5 * q, Vp + 5 * q, F + 5 * q, err);
  if (err) atomicOr(&cnt->error, 1);
}

}  // namespace m2c
