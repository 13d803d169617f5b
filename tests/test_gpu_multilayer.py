"""Multi-layer McClean passes: tiles, windows and memory modes at their edges.

Bars: complex128 within 1e-12 norm-relative of the oracle (the bar of
test_gpu_mcclean.py: some 100 gates at 2^-53 each); complex64 within 1e-6
(FP64 arithmetic, at most some 50 roundings to 2^-24 per amplitude, which
average out over 2^14 and more of them).
"""
import numpy as np
import pytest

from oracle import statevector as sv
from tests.conftest import rel_err

pytestmark = pytest.mark.gpu

TOL = {'complex128': 1e-12, 'complex64': 1e-6}


def _circuit(n, L, seed, dtype='complex128', entangler='cnot', tile=None, ckpt=0):
    from qradient_amd import _native
    from qradient_amd.circuit_logic import McClean
    rs = np.random.RandomState(seed)
    axes, angles = sv.mcclean_random_params(L, n, rs)
    obs = sv.zz_chain_observable(n, rs.standard_normal(n - 1))
    c = McClean(n, obs, L, axes=axes, angles=angles, dtype=dtype, entangler=entangler, ckpt_every=ckpt)
    if tile:
        _native.call('qg_plan_tune', c._get_plan(), tile[0], tile[1], 4, 4)
    return c, axes, angles, obs


def _check(c, axes, angles, obs, dtype, entangler, ini=None):
    n = angles.shape[1]
    E, g = c.grad_run(ini_state=ini)
    E2 = c.run_expec_val(ini_state=ini)
    Eo, go = sv.mcclean_grad_run_adjoint(n, axes, angles, obs, entangler=entangler, ini_state=ini)
    wsum = sum(abs(float(w)) for w in obs['zz'].ravel() if w is not None)
    assert abs(E - Eo) <= TOL[dtype] * wsum, (E, Eo)
    assert abs(E2 - Eo) <= TOL[dtype] * wsum, (E2, Eo)
    assert rel_err(g, go) <= TOL[dtype], rel_err(g, go)


# the smallest and largest tiles, the narrowest and widest windows above the
# contiguous bits, a window that ends at the top qubit and one short of it
@pytest.mark.parametrize('tile', [(10, 1), (10, 6), (11, 2), (12, 3), (12, 5), (13, 4), (13, 9)])
@pytest.mark.parametrize('n,L', [(14, 1), (14, 9), (15, 4), (17, 3)])
@pytest.mark.parametrize('entangler', ['cnot', 'cz'])
def test_tiles(gpu, tile, n, L, entangler):
    dtype = 'complex64' if (n + L + tile[0]) % 2 else 'complex128'
    c, *args = _circuit(n, L, 100 * n + L, dtype, entangler, tile)
    _check(c, *args, dtype, entangler)


@pytest.mark.parametrize('n,L', [(14, 5), (19, 3), (20, 3), (21, 2)])
@pytest.mark.parametrize('ckpt', [1, 2, 64])
@pytest.mark.parametrize('dtype', ['complex128', 'complex64'])
def test_checkpoints(gpu, n, L, ckpt, dtype):
    c, *args = _circuit(n, L, n + ckpt, dtype, 'cz' if ckpt == 2 else 'cnot', ckpt=ckpt)
    _check(c, *args, dtype, c.entangler)


@pytest.mark.parametrize('lds64', [1, 2])
def test_fp64_tiles(gpu, lds64):
    from qradient_amd import _native
    c, *args = _circuit(16, 6, 7, 'complex64')
    _native.call('qg_plan_set_lds64', c._get_plan(), lds64)
    _check(c, *args, 'complex64', 'cnot')


@pytest.mark.parametrize('ckpt', [0, 2])
def test_ini_state(gpu, ckpt):
    rs = np.random.RandomState(3)
    ini = rs.standard_normal(1 << 15) + 1j * rs.standard_normal(1 << 15)
    ini /= np.linalg.norm(ini)
    c, *args = _circuit(15, 4, 11, ckpt=ckpt)
    _check(c, *args, 'complex128', 'cnot', ini)


@pytest.mark.parametrize('dtype,n', [('complex128', 28), ('complex64', 29)])
def test_wide_offsets(gpu, dtype, n):
    """States of 4 GiB take 64-bit addresses; the same circuit in single-layer
    passes (tiles of 2^9) is the reference."""
    c, *_ = _circuit(n, 2, 5, dtype, ckpt=2)
    E, g = c.grad_run()
    del c
    c, *_ = _circuit(n, 2, 5, dtype, tile=(9, 3), ckpt=2)
    E0, g0 = c.grad_run()
    assert abs(E - E0) <= TOL[dtype] * n
    assert rel_err(g, g0) <= TOL[dtype], rel_err(g, g0)
