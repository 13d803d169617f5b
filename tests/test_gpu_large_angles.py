"""Rotation angles of many periods.  The oracle takes cosine and sine of half the
angle itself, so 1e-12 holds at any size: an error of the angle's reduction
would be 1.2e-16 per half period, 4e-5 at 1e12."""
import numpy as np
import pytest

from oracle import statevector as sv
from tests.conftest import rel_err

pytestmark = pytest.mark.gpu

TOL = 1e-12


@pytest.mark.parametrize('scale', [1.0, 1e4, 1e8, 1e12])
@pytest.mark.parametrize('n', [4, 10, 13, 15])
def test_mcclean(gpu, n, scale):
    from qradient_amd.circuit_logic import McClean
    rs = np.random.RandomState(n)
    L = 4
    axes, _ = sv.mcclean_random_params(L, n, rs)
    angles = scale * rs.uniform(-8, 8, (L, n))
    obs = sv.zz_chain_observable(n, rs.standard_normal(n - 1))
    c = McClean(n, obs, L, axes=axes, angles=angles)
    E, g = c.grad_run()
    Eo, go = sv.mcclean_grad_run_adjoint(n, axes, angles, obs)
    assert abs(E - Eo) <= TOL * max(1.0, abs(Eo))
    assert rel_err(g, go) <= TOL
    c.run_expec_val()
    assert np.linalg.norm(c.final_state() - sv.mcclean_forward(n, axes, angles)) <= TOL


@pytest.mark.parametrize('scale', [1.0, 1e8])
@pytest.mark.parametrize('n', [5, 12, 15])
def test_qaoa_mixer(gpu, n, scale):
    from qradient_amd.circuit_logic import Qaoa
    rs = np.random.RandomState(n)
    p = 3
    obs = sv.maxcut_observable(n, [(i, i + 1) for i in range(n - 1)])
    b, g = scale * rs.uniform(-4, 4, p), rs.uniform(0.1, 2.0, p)
    E, gr = Qaoa(n, obs, p).grad_run(b, g)
    Eo, go = sv.qaoa_grad_run_adjoint(n, obs, b, g)
    assert abs(E - Eo) <= TOL * max(1.0, abs(Eo))
    assert rel_err(gr, go) <= TOL
