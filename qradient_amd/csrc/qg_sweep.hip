// Instantiations of the multi-layer passes: complex64 (FP32 or FP64 LDS tiles)
// and complex128.
#include "qg_sweep.hpp"

namespace qg {

namespace {

// Calls f with the kernel variant's template arguments.
template <class F>
hipError_t sweep_variant(int dtype, bool two, bool big, bool obs, F&& f) {
  auto with_mode = [&](auto s, auto b) {
    if (!two) return f(s, std::false_type{}, b, std::false_type{});
    return obs ? f(s, std::true_type{}, b, std::true_type{}) : f(s, std::true_type{}, b, std::false_type{});
  };
  auto with_big = [&](auto s) { return big ? with_mode(s, std::true_type{}) : with_mode(s, std::false_type{}); };
  return dtype == 0 ? with_big(double{}) : dtype == 1 ? with_big(float{}) : with_big(F32L64{});
}

}  // namespace

// dtype as in launch_pass: 0 complex128, 1 complex64, 2 complex64 with FP64
// LDS tiles.  obs: an adjoint pass that forms lambda.
hipError_t launch_sweep(int dtype, bool two, bool obs, const SweepDesc* d, int K, int grid, int batch, int n,
                        hipStream_t st, int* occ, int tab) {
  if (K < kSweepMinK || K > kSweepMaxK || K > n) return hipErrorInvalidValue;
  return sweep_variant(dtype, two, (n + (dtype == 0 ? 4 : 3)) > 32, obs, [&](auto s, auto tw, auto b, auto o) {
    return launch_sweep_t<decltype(s), decltype(tw)::value, decltype(b)::value, decltype(o)::value>(d, K, grid, batch,
                                                                                                   st, occ, tab);
  });
}

hipError_t set_sweep_attributes() {
  hipError_t e = hipSuccess;
  for (int v = 0; v < 24 && e == hipSuccess; ++v)
    e = sweep_variant(v / 8, v & 1, v & 2, v & 4, [](auto s, auto tw, auto b, auto o) {
      return set_sweep_attr_t<decltype(s), decltype(tw)::value, decltype(b)::value, decltype(o)::value>();
    });
  return e;
}

}  // namespace qg
