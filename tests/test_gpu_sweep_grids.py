"""Every tile of the multi-layer passes is launched on a grid that the partial
rows hold, whatever the variants' occupancies: the forward passes, which hold
one state, may be resident in greater number than the adjoint ones.  The
circuit is trivial (two layers of RZ by 2 pi, which is minus the identity, on
the RY(pi/4) product state, each after a ladder of CZ), so <Z_0> = cos(pi/4) and the
gradient vanishes: 48 gates leave 1e-12 in complex128, and single roundings of
2^-24 stay below 1e-6."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('tile', [(10, 1), (10, 6), (11, 2), (11, 7), (12, 3), (13, 3)])
@pytest.mark.parametrize('dtype,lds64', [('complex128', 0), ('complex64', 0), ('complex64', 1), ('complex64', 2)])
def test_grids_fit_the_rows(gpu, tile, dtype, lds64):
    from qradient_amd import _native
    from qradient_amd.circuit_logic import McClean
    n, L = 24, 2
    z = np.full(n, None)
    z[0] = 1.0
    c = McClean(n, {'z': z}, L, axes=np.full((L, n), 2), angles=np.full((L, n), 2 * np.pi), dtype=dtype,
                entangler='cz')
    if lds64:
        _native.call('qg_plan_set_lds64', c._get_plan(), lds64)
    _native.call('qg_plan_tune', c._get_plan(), tile[0], tile[1], 4, 4)
    E, g = c.grad_run()
    tol = 1e-12 if dtype == 'complex128' else 1e-6
    assert abs(E - np.cos(np.pi / 4)) <= tol
    assert np.linalg.norm(g) <= tol
