// Instantiations of the multi-layer passes: complex64 (FP32 or FP64 LDS tiles)
// and complex128.
#include "qg_sweep.hpp"

namespace qg {

// dtype as in launch_pass: 0 complex128, 1 complex64, 2 complex64 with FP64 LDS tiles.
hipError_t launch_sweep(int dtype, bool two, const SweepDesc* d, int K, int grid, int batch, int n, hipStream_t st,
                        int* occ, int tab) {
  if (K < kSweepMinK || K > kSweepMaxK || K > n) return hipErrorInvalidValue;
  const bool big = (n + (dtype == 0 ? 4 : 3)) > 32;
  switch (dtype * 2 + (two ? 1 : 0)) {
    case 0: return launch_sweep_t<double, false>(d, K, grid, batch, big, st, occ, tab);
    case 1: return launch_sweep_t<double, true>(d, K, grid, batch, big, st, occ, tab);
    case 2: return launch_sweep_t<float, false>(d, K, grid, batch, big, st, occ, tab);
    case 3: return launch_sweep_t<float, true>(d, K, grid, batch, big, st, occ, tab);
    case 4: return launch_sweep_t<F32L64, false>(d, K, grid, batch, big, st, occ, tab);
    case 5: return launch_sweep_t<F32L64, true>(d, K, grid, batch, big, st, occ, tab);
  }
  return hipErrorInvalidValue;
}

hipError_t set_sweep_attributes() {
  hipError_t e = set_sweep_attr_t<double, false>();
  if (e == hipSuccess) e = set_sweep_attr_t<double, true>();
  if (e == hipSuccess) e = set_sweep_attr_t<float, false>();
  if (e == hipSuccess) e = set_sweep_attr_t<float, true>();
  if (e == hipSuccess) e = set_sweep_attr_t<F32L64, false>();
  if (e == hipSuccess) e = set_sweep_attr_t<F32L64, true>();
  return e;
}

}  // namespace qg
