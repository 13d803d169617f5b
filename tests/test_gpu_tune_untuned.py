"""tune_mcclean times the untuned plan beside its candidates and keeps it when no
candidate is faster; a circuit with tune=True then runs untuned."""
import numpy as np
import pytest

from oracle import statevector as sv
from tests.conftest import rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('n,L', [(16, 6), (20, 4)])
def test_untuned_plan_is_a_candidate(gpu, tmp_path, monkeypatch, n, L):
    from qradient_amd import autotune
    from qradient_amd.circuit_logic import McClean
    monkeypatch.setenv('QRADIENT_AMD_TUNE_CACHE', str(tmp_path / 'tune.json'))
    # 8 local bits: one layer a pass and several passes a layer, far behind the default
    slow = {'kmax': 8, 'cmin': 4, 'r_fwd': 4, 'r_rev': 4}
    best, results = autotune.tune_mcclean(n, L, 'complex128', shapes=[slow])
    untuned = autotune.untuned_shape(n, 'complex128')
    assert [s for s, _ in results] == [untuned, slow]
    assert best == untuned
    assert autotune.cached('mcclean', n, L, 'complex128', 'cnot') == best
    rs = np.random.RandomState(n)
    axes, angles = sv.mcclean_random_params(L, n, rs)
    obs = sv.zz_chain_observable(n, rs.standard_normal(n - 1))
    out = [McClean(n, obs, L, axes=axes, angles=angles, tune=t).grad_run() for t in (False, True)]
    assert out[0][0] == out[1][0] and np.array_equal(out[0][1], out[1][1])
    assert rel_err(out[1][1], sv.mcclean_grad_run_adjoint(n, axes, angles, obs)[1]) <= 1e-12
