"""The basis sampler's search at the edges of its two levels: states smaller
than a wave and than a block, one block, several rounds of the block prefix
(more than 1024 blocks), shot counts that do not fill a workgroup, long runs of
zero probability, and draws that no position reaches."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('n,shots', [(1, 1), (5, 3), (9, 5), (10, 64), (11, 7), (17, 1001), (21, 130)])
@pytest.mark.parametrize('dtype', ['complex128', 'complex64'])
@pytest.mark.parametrize('holes', [False, True])
def test_draws_are_the_inverse_cdf(gpu, n, shots, dtype, holes):
    from qradient_amd.physical_components import State
    N = 2 ** n
    rs = np.random.RandomState(10 * n + shots)
    v = rs.standard_normal(N) + 1j * rs.standard_normal(N)
    if holes and N > 2:
        v[N // 4:N - max(1, N // 8)] = 0.0
    v /= np.linalg.norm(v)
    st = State(n, dtype=dtype)
    st.vec = v
    p = np.abs(st.vec) ** 2
    cdf = np.cumsum(p)
    u = rs.uniform(0.0, 0.999, size=shots)
    u[0] = 0.0
    got = st.sample_basis(u)
    want = np.searchsorted(cdf, u, side='left')
    # equal up to draws within rounding of a boundary (sums of 2^21 terms: < 1e-12)
    lo = np.where(got > 0, cdf[np.maximum(got, 1) - 1], 0.0)
    assert np.all((got == want) | ((lo - 1e-12 <= u) & (u <= cdf[got] + 1e-12) & (np.abs(cdf[want] - u) < 1e-12)))


def test_draws_past_the_total_mass_give_position_zero(gpu):
    from qradient_amd.physical_components import State
    n = 12
    v = np.zeros(2 ** n, dtype=complex)
    v[100:200] = 0.05  # total mass 0.25
    st = State(n)
    st.vec = v
    got = st.sample_basis(np.array([0.3, 0.9, 0.1]))
    assert got[0] == 0 and got[1] == 0 and 100 <= got[2] < 200
