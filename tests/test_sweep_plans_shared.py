"""Plans of multi-layer passes shared between a context's plans (SweepPlans in
csrc/qg_sweep_plan.hpp), compiled for the host: the same passes as a fresh
planner's whatever was asked before, from several threads, within the bounds."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), '..', 'qradient_amd', 'csrc')

SOURCE = r'''
#include <cstdio>
#include <random>
#include <thread>
#include "qg_sweep_plan.hpp"
using namespace qg;
static bool same(const std::vector<PlanPass>& a, const std::vector<PlanPass>& b) {
  if (a.size() != b.size()) return false;
  for (size_t i = 0; i < a.size(); ++i) {
    if (a[i].lo != b[i].lo || a[i].hi != b[i].hi || a[i].c != b[i].c || a[i].rounds.size() != b[i].rounds.size())
      return false;
    for (size_t r = 0; r < a[i].rounds.size(); ++r) {
      const PlanRound &x = a[i].rounds[r], &y = b[i].rounds[r];
      if (x.lo != y.lo || x.b1 != y.b1 || x.b2 != y.b2) return false;
      for (int k = 0; k < 4; ++k)
        if (x.bit[k] != y.bit[k] || x.layer[k] != y.layer[k]) return false;
    }
  }
  return true;
}
int main() {
  SweepPlans shared;
  bool ok[8];
  std::vector<std::thread> threads;
  for (int t = 0; t < 8; ++t)
    threads.emplace_back([&shared, &ok, t] {
      std::mt19937 rng(t);
      ok[t] = true;
      for (int i = 0; i < 300; ++i) {
        const int n = 14 + (int)(rng() % 14), K = 10 + (int)(rng() % 4), c = 1 + (int)(rng() % 4);
        const SweepKey k = {n, 1 + (int)(rng() % 6), (int)(rng() % 2), K, c, rng() % 2 ? 6 : 4};
        ok[t] = ok[t] && same(shared.get(k), SweepPlanner(k[0], k[1], k[2] != 0, k[3], k[4]).plan(k[5]));
      }
    });
  for (auto& th : threads) th.join();
  bool all = true;
  for (bool o : ok) all = all && o;
  const bool few = shared.plans() <= SweepPlans::kPlans && shared.rounds() <= SweepPlans::kRounds;
  for (int n = 14; n < 30; ++n) shared.get({n, 1000, 0, 12, 3, 4});  // long circuits: bounded by their rounds
  const bool small = shared.rounds() <= SweepPlans::kRounds && shared.plans() < 16;
  shared.get({30, 30000, 0, 12, 3, 4});  // more rounds than are kept
  std::printf("%d %d %d %d\n", all, few, small, shared.rounds() <= SweepPlans::kRounds);
}
'''


def test_shared_plans_equal_fresh_ones(tmp_path):
    (tmp_path / 'plans.cpp').write_text(SOURCE)
    subprocess.run(['g++', '-O2', '-std=c++17', '-pthread', '-I', CSRC, str(tmp_path / 'plans.cpp'), '-o',
                    str(tmp_path / 'plans')], check=True)
    out = subprocess.run([str(tmp_path / 'plans')], check=True, capture_output=True, text=True).stdout
    assert out.split() == ['1', '1', '1', '1']
