"""The whole-circuit kernel at every qubit number it is built for (its layouts
differ with the number: one thread, part of a wave, one wave, 2, 4 and 8
waves), and each way it forms the QAOA phase: table, reduced sincos, library
sincos.  Oracle in complex128; 1e-12 norm-relative (13 qubits and 3 layers are
some 10^3 roundings of 1e-16 each)."""
import numpy as np
import pytest

from oracle import statevector as sv
from tests.conftest import rel_err

pytestmark = pytest.mark.gpu

TOL = 1e-12


@pytest.mark.parametrize('n', range(1, 14))
@pytest.mark.parametrize('entangler', ['cnot', 'cz'])
def test_mcclean_every_size(gpu, n, entangler):
    from qradient_amd.circuit_logic import McClean
    rs = np.random.RandomState(900 + n)
    L = 3
    axes, angles = sv.mcclean_random_params(L, n, rs)
    angles = angles * 3 - 6  # past one period on both sides: dropped signs
    obs = sv.zz_chain_observable(n, rs.standard_normal(n - 1)) if n > 1 else {}
    for key in ('x', 'y', 'z'):
        obs[key] = np.array([float(rs.standard_normal()) for _ in range(n)], dtype=object)
    c = McClean(n, obs, L, axes=axes, angles=angles, entangler=entangler)
    E, g = c.grad_run()
    Eo, go = sv.mcclean_grad_run_adjoint(n, axes, angles, obs, entangler=entangler)
    assert abs(E - Eo) <= TOL * max(1.0, abs(Eo))
    assert rel_err(g, go) <= TOL
    c.run_expec_val()
    vo = sv.mcclean_forward(n, axes, angles, entangler=entangler)
    assert np.linalg.norm(c.state.vec - vo) <= TOL


@pytest.mark.parametrize('n', range(2, 14))
@pytest.mark.parametrize('phase', ['table', 'sincos', 'large'])
def test_qaoa_every_size(gpu, n, phase):
    from qradient_amd.circuit_logic import Qaoa
    rs = np.random.RandomState(700 + n)
    p = 2
    zz = np.full((n, n), None)
    for i in range(n - 1):
        zz[i, i + 1] = float(rs.randint(1, 4))
    if n > 3:
        zz[0, n - 1] = -2.0
    if phase != 'table':
        # quarters: C(x) is exact, so the phase angle gamma * C(x) is one rounding
        zz[0, 1] = 0.75
    obs = {'zz': zz, 'z': np.array([1.0 if q % 3 == 0 else None for q in range(n)], dtype=object)}
    b = rs.uniform(-4, 4, p)
    g = rs.uniform(0.1, 2.0, p) * (1e8 if phase == 'large' else 1.0)
    c = Qaoa(n, obs, p)
    E, grad = c.grad_run(b, g)
    Eo, go = sv.qaoa_grad_run_adjoint(n, obs, b, g)
    assert abs(E - Eo) <= TOL * max(1.0, abs(Eo))
    assert rel_err(grad, go) <= TOL
    c.run_expec_val(b, g)
    vo = sv.qaoa_forward(n, obs, b, g)
    vo = vo[-1] if isinstance(vo, (tuple, list)) else vo
    assert np.linalg.norm(c.state.vec - vo) <= TOL
