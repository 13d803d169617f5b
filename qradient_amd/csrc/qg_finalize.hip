// Deterministic final reduction of the partial rows written by the passes,
// and the pass-kernel dispatch used by the host planner.
#include <hip/hip_runtime.h>

#include "qg_internal.h"

namespace qg {

hipError_t launch_pass_c64(int R, bool two, int phase, bool post, const PassDesc* d, int K, int grid, int batch,
                           int threads, bool big, hipStream_t st, int* occ, int tab);
hipError_t launch_pass_c128(int R, bool two, int phase, bool post, const PassDesc* d, int K, int grid, int batch,
                            int threads, bool big, hipStream_t st, int* occ, int tab);
hipError_t launch_pass_c64x(int R, bool two, int phase, bool post, const PassDesc* d, int K, int grid, int batch,
                            int threads, bool big, hipStream_t st, int* occ, int tab);
hipError_t set_attributes_c64();
hipError_t set_attributes_c128();
hipError_t set_attributes_c64x();

// out[i] = sum over the rows (r, cnt) of output i of sum_{w < cnt} part[r*stride + w];
// with ndot, out[0] = the sum of dot[0, ndot).  One workgroup per output; each thread sums a fixed
// strided subset, then a fixed-shape tree: the result does not depend on
// scheduling.  The table and the outputs may lie in host memory.
__global__ __launch_bounds__(256) void k_finalize(int nout, const int* __restrict__ ptr, const int2* __restrict__ rows,
                                                  const double* __restrict__ part, int stride,
                                                  const double* __restrict__ dot, int ndot, double* __restrict__ out) {
  __shared__ double red[256];
  const int i = blockIdx.x;
  if (i >= nout) return;
  double s = 0.0;
  for (int k = ptr[i]; k < ptr[i + 1]; ++k) {
    const int2 r = rows[k];
    for (int w = threadIdx.x; w < r.y; w += blockDim.x) s += part[(size_t)r.x * stride + w];
  }
  if (i == 0)
    for (int w = threadIdx.x; w < ndot; w += blockDim.x) s += dot[w];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int h = blockDim.x / 2; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h) red[threadIdx.x] += red[threadIdx.x + h];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[i] = red[0];
}

hipError_t launch_finalize(int nout, const int* ptr, const int2* rows, const double* part, int stride,
                           const double* dot, int ndot, double* out, hipStream_t st) {
  if (nout <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_finalize, dim3(nout), dim3(256), 0, st, nout, ptr, rows, part, stride, dot, ndot, out);
  return hipGetLastError();
}

hipError_t set_pass_attributes() {
  hipError_t e = set_attributes_c64();
  if (e == hipSuccess) e = set_attributes_c128();
  if (e == hipSuccess) e = set_attributes_c64x();
  return e;
}

// dtype 1: complex64 storage, 0: complex128, 2: complex64 storage with FP64
// LDS tiles (phase-free passes only).  post: an adjoint pass of the general
// form.  With occ != NULL the pass is not launched: *occ
// receives the workgroups per CU.  tab: bytes of the table the pass stages in
// LDS.
hipError_t launch_pass(int dtype, int R, bool two, int phase, bool post, const PassDesc* d, int K, int grid,
                       int batch, int threads, int n, hipStream_t st, int* occ, int tab) {
  // byte offsets of a 2^n state: 32-bit addressing below 4 GiB
  const bool big = (n + (dtype == 0 ? 4 : 3)) > 32;
  if (dtype == 1) return launch_pass_c64(R, two, phase, post, d, K, grid, batch, threads, big, st, occ, tab);
  if (dtype == 2) return launch_pass_c64x(R, two, phase, post, d, K, grid, batch, threads, big, st, occ, tab);
  return launch_pass_c128(R, two, phase, post, d, K, grid, batch, threads, big, st, occ, tab);
}

}  // namespace qg
