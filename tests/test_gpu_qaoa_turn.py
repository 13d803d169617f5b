"""QAOA turning passes: windows, register windows and phase forms at their edges.

Bars: complex128 within 1e-12 norm-relative of the oracle (some 100 gates at
2^-53 each); complex64 within 1e-6 (FP64 arithmetic, some tens of roundings
to 2^-24 per amplitude, which average out over the state).
"""
import numpy as np
import pytest

from oracle import statevector as sv
from tests.conftest import rel_err

pytestmark = pytest.mark.gpu

TOL = {'complex128': 1e-12, 'complex64': 1e-6}


def _hamiltonian(n, rs, weights):
    """Ring and chords, and one-bit terms on the outermost bits."""
    zz = np.full((n, n), None)
    for i in range(n):
        for k in (1, n // 2):
            a, b = sorted((i, (i + k) % n))
            if a != b:
                zz[a, b] = 1.0 if weights == 'unit' else float(rs.standard_normal())
    z = np.array([1.0 if q in (0, n - 1) else None for q in range(n)], dtype=object)
    return {'zz': zz, 'z': z}


def _check(n, p, dtype, weights, tile=None, scale=1.0, batch=1, ini=None):
    from qradient_amd import _native
    from qradient_amd.batch import QaoaBatch
    rs = np.random.RandomState(n * 100 + p)
    obs = [_hamiltonian(n, rs, weights) for _ in range(batch)]
    betas, gammas = rs.uniform(0, 3, (batch, p)), scale * rs.uniform(-2, 2, (batch, p))
    q = QaoaBatch(n, p, batch, dtype=dtype)
    if tile:
        _native.call('qg_qaoa_tune', q._plan, tile[0], tile[1], 0, 16)
    states = None if ini is None else np.array([ini] * batch)
    E, g = q.grad_run(obs, betas, gammas, ini_states=states)
    E2 = q.expec_val(obs, betas, gammas, ini_states=states)
    for b in range(batch):
        Eo, go = sv.qaoa_grad_run_adjoint(n, obs[b], betas[b], gammas[b], ini_state=ini)
        wsum = sum(abs(float(w)) for m in obs[b].values() for w in m.ravel() if w is not None)
        assert abs(E[b] - Eo) <= TOL[dtype] * wsum, (b, E[b], Eo)
        assert abs(E2[b] - Eo) <= TOL[dtype] * wsum, (b, E2[b], Eo)
        go = np.asarray(go).reshape(-1)
        assert rel_err(np.asarray(g[b]).reshape(-1), go) <= TOL[dtype], (b, rel_err(np.asarray(g[b]).reshape(-1), go))


# two and three windows; the narrowest window (one owned bit), register
# windows that overlap (13 local bits) and that are not full
@pytest.mark.parametrize('n,tile', [(14, (13, 3)), (14, (10, 3)), (15, (10, 1)), (17, (10, 7)), (18, (12, 3)),
                                    (17, (13, 4)), (16, (11, 6))])
@pytest.mark.parametrize('p', [1, 2, 5])
@pytest.mark.parametrize('weights', ['unit', 'real'])
def test_windows(gpu, n, tile, p, weights):
    _check(n, p, 'complex64' if (n + p) % 2 else 'complex128', weights, tile)


@pytest.mark.parametrize('n', [14, 18, 20])
@pytest.mark.parametrize('dtype', ['complex128', 'complex64'])
def test_default_tiles_batched(gpu, n, dtype):
    _check(n, 3, dtype, 'unit', batch=3)


def test_large_angles(gpu):
    """Angles past the range of the kernels' own sincos (2^26)."""
    # gamma D to 2^-53 relative is an absolute phase error of 1e8 * 2^-53 =
    # 1e-8 in the oracle and the kernels alike: the same product, so the same
    # rounded argument up to the summation order of D; compare at 1e-6
    from qradient_amd.batch import QaoaBatch
    n, rs = 14, np.random.RandomState(4)
    obs = _hamiltonian(n, rs, 'unit')
    obs['z'][0] = 0.5  # exactly representable: D is the same in any order
    betas, gammas = rs.uniform(0, 3, (1, 2)), np.array([[1.0e8, -3.0e8]])
    E, g = QaoaBatch(n, 2, 1, dtype='complex128').grad_run([obs], betas, gammas)
    Eo, go = sv.qaoa_grad_run_adjoint(n, obs, betas[0], gammas[0])
    assert abs(E[0] - Eo) <= 1e-6 * 50
    assert rel_err(np.asarray(g[0]).reshape(-1), np.asarray(go).reshape(-1)) <= 1e-6


@pytest.mark.parametrize('p', [1, 4])
def test_ini_states(gpu, p):
    rs = np.random.RandomState(8)
    ini = rs.standard_normal(1 << 15) + 1j * rs.standard_normal(1 << 15)
    ini /= np.linalg.norm(ini)
    _check(15, p, 'complex128', 'real', batch=2, ini=ini)


@pytest.mark.parametrize('n', [2, 9, 10, 11, 12, 13])
def test_large_angles_from_a_table(gpu, n):
    """Whole-circuit runs with integer weights and angles past 2^26: the
    table's arguments are the oracle's products, so the bar is the usual one
    times the libraries' sincos (1e-12 covers both)."""
    from qradient_amd.batch import QaoaBatch
    rs = np.random.RandomState(n)
    zz = np.full((n, n), None)
    for i in range(n - 1):
        zz[i, i + 1] = 1.0
    betas, gammas = rs.uniform(0, 3, (1, 3)), np.array([[1.0e8, -2.5e8, 0.7]])
    E, g = QaoaBatch(n, 3, 1).grad_run([{'zz': zz}], betas, gammas)
    Eo, go = sv.qaoa_grad_run_adjoint(n, {'zz': zz}, betas[0], gammas[0])
    assert abs(E[0] - Eo) <= 1e-12 * n
    assert rel_err(np.asarray(g[0]).reshape(-1), np.asarray(go).reshape(-1)) <= 1e-12
