// Instantiations of the QAOA turning passes: complex64 and complex128.
#include "qg_turn.hpp"

namespace qg {

namespace {

// Calls f with the kernel variant's template arguments.
template <class F>
hipError_t turn_variant(int dtype, bool two, int ph, bool big, F&& f) {
  auto with_big = [&](auto s, auto tw, auto p) {
    return big ? f(s, tw, p, std::true_type{}) : f(s, tw, p, std::false_type{});
  };
  auto with_ph = [&](auto s, auto tw) {
    return ph == TP_LUT      ? with_big(s, tw, ic<TP_LUT>{})
           : ph == TP_SINCOS ? with_big(s, tw, ic<TP_SINCOS>{})
                             : with_big(s, tw, ic<TP_LARGE>{});
  };
  auto with_two = [&](auto s) { return two ? with_ph(s, std::true_type{}) : with_ph(s, std::false_type{}); };
  return dtype == 0 ? with_two(double{}) : with_two(float{});
}

}  // namespace

// dtype: 0 complex128, 1 complex64.
hipError_t launch_turn(int dtype, bool two, int ph, const TurnDesc* d, int K, int grid, int batch, int n,
                       hipStream_t st, int* occ, int tab) {
  if (K < kSweepMinK || K > kSweepMaxK || K > n) return hipErrorInvalidValue;
  return turn_variant(dtype, two, ph, (n + (dtype == 0 ? 4 : 3)) > 32, [&](auto s, auto tw, auto p, auto b) {
    return launch_turn_t<decltype(s), decltype(tw)::value, decltype(p)::value, decltype(b)::value>(d, K, grid, batch,
                                                                                                  st, occ, tab);
  });
}

hipError_t set_turn_attributes() {
  hipError_t e = hipSuccess;
  for (int v = 0; v < 24 && e == hipSuccess; ++v)
    e = turn_variant(v & 1, v & 2, v / 8, v & 4, [](auto s, auto tw, auto p, auto b) {
      return set_turn_attr_t<decltype(s), decltype(tw)::value, decltype(p)::value, decltype(b)::value>();
    });
  return e;
}

}  // namespace qg
