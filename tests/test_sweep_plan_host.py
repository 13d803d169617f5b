"""The planner of the multi-layer passes (csrc/qg_sweep_plan.hpp), compiled for
the host: the number of rounds of every default tile stays within the bound that
sizes a plan's tables, and the bound grows with the shape."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), '..', 'qradient_amd', 'csrc')

# prints "n L dtype-size entangler passes rounds bound" of every shape; the tile
# rule is that of plan_sweeps in qg_api.cpp
SOURCE = r'''
#include <cstdio>
#include "qg_sweep_plan.hpp"
int main() {
  for (int bytes = 8; bytes <= 16; bytes += 8)
    for (int cz = 0; cz < 2; ++cz)
      for (int L = 1; L <= 100; L += L < 24 ? 1 : 7)
        for (int n = 14; n <= 32; ++n) {
          const bool cached = ((size_t)bytes << n) <= ((size_t)64 << 20);
          const int K = n < 20 ? 11 : 12, c = cached ? 2 : 3, steps = n >= 20 && cached ? 6 : 4;
          const auto plan = qg::SweepPlanner(n, L, cz, K, c).plan(steps);
          int rounds = 0;
          for (const auto& p : plan) rounds += (int)p.rounds.size();
          std::printf("%d %d %d %d %d %d %d\n", n, L, bytes, cz, (int)plan.size(), rounds, qg::sweep_round_bound(n, L));
        }
}
'''


@pytest.fixture(scope='module')
def shapes(tmp_path_factory):
    d = tmp_path_factory.mktemp('sweep_plan')
    (d / 'plan.cpp').write_text(SOURCE)
    subprocess.run(['g++', '-O2', '-std=c++17', '-I', CSRC, str(d / 'plan.cpp'), '-o', str(d / 'plan')], check=True)
    out = subprocess.run([str(d / 'plan')], check=True, capture_output=True, text=True).stdout
    return [tuple(map(int, line.split())) for line in out.splitlines()]


def test_rounds_stay_within_the_bound(shapes):
    assert len(shapes) > 2000
    over = [s for s in shapes if s[5] > s[6]]
    assert not over, over[:5]


def test_bound_grows_with_the_shape(shapes):
    bound = {(s[0], s[1]): s[6] for s in shapes}
    for (n, L), b in bound.items():
        assert b <= bound.get((n + 1, L), b) and b <= bound.get((n, L + 1), b), (n, L)
