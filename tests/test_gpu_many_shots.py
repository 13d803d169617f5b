"""More shots than a launch of one wave per shot could hold (2^32 threads), drawn
in turn by the waves of a bounded grid, on states of one sampling block and of
several.  The uniform state makes the expected position a floor."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('n,shots', [(3, 2 ** 26 + 5), (11, 2 ** 26 + 5), (3, 32771), (7, 100003), (10, 32770), (12, 131075)])
@pytest.mark.parametrize('dtype', ['complex64', 'complex128'])
def test_every_shot_is_drawn(gpu, n, shots, dtype):
    from qradient_amd.physical_components import State
    N = 2 ** n
    u = np.random.default_rng(n).integers(0, 64 * N, shots)
    st = State(n, '+', dtype=dtype)
    # midway between two of 64 marks per position: 2^-7 of a position from an edge
    got = st.sample_basis((u + 0.5) / (64 * N))
    assert np.array_equal(got, u // 64)
