// Quotients and roots of m2c_exactdiv.h over arrays, for the test that compares
// them with IEEE division and square root.
#include "../m2c_amd/csrc/m2c_exactdiv.h"

__global__ void k_quot(const double* a, const double* b, double* q, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) q[i] = m2c::Recip(b[i]).quot(a[i]);
}
__global__ void k_root(const double* x, double* r, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) r[i] = m2c::root_in_range(x[i]);
}

// b null: roots of a; host arrays of n
extern "C" int exactdiv(const double* a, const double* b, double* out, int n) {
  double *da = nullptr, *db = nullptr, *dq = nullptr;
  const size_t bytes = (size_t)n * 8;
  int rc = 0;
  auto ok = [&rc](hipError_t e) { if (e != hipSuccess && !rc) rc = (int)e; return !rc; };
  if (ok(hipMalloc(&da, bytes)) && ok(hipMalloc(&db, bytes)) && ok(hipMalloc(&dq, bytes)) &&
      ok(hipMemcpy(da, a, bytes, hipMemcpyHostToDevice)) &&
      (!b || ok(hipMemcpy(db, b, bytes, hipMemcpyHostToDevice)))) {
    if (b) k_quot<<<(n + 255) / 256, 256>>>(da, db, dq, n);
    else k_root<<<(n + 255) / 256, 256>>>(da, dq, n);
    if (ok(hipGetLastError())) ok(hipMemcpy(out, dq, bytes, hipMemcpyDeviceToHost));
  }
  (void)hipFree(da); (void)hipFree(db); (void)hipFree(dq);
  return rc;
}
