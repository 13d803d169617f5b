"""Batched shifted circuits and the term measurement behind them, at the edges
of a batch: one circuit, groups cut by the batch bound, shifts out of layer
order, checkpoints with unshifted layers in between, both entanglers; QAOA's
shifted circuits with table and sincos phases on one and two passes a layer."""
import numpy as np
import pytest

from oracle import reference_algorithm as ra
from oracle import statevector as sv

pytestmark = pytest.mark.gpu


def _shifted_probs(n, axes, angles, params, deltas, obs, entangler):
    out = []
    for k, d in zip(params, deltas):
        a = angles.copy()
        a.flat[k] += d
        out.append(sv.term_probs(sv.mcclean_forward(n, axes, a, entangler=entangler), obs)[0])
    return np.array(out)


@pytest.mark.parametrize('n,L,ckpt', [(1, 2, 0), (4, 3, 0), (9, 4, 3), (12, 2, 0), (14, 2, 0), (15, 4, 4), (20, 2, 0)])
@pytest.mark.parametrize('entangler', ['cnot', 'cz'])
def test_mcclean_shift_probs(gpu, n, L, ckpt, entangler):
    from qradient_amd.circuit_logic import McClean
    rs = np.random.RandomState(n)
    axes, angles = sv.mcclean_random_params(L, n, rs)
    obs = sv.zz_chain_observable(n, rs.standard_normal(n - 1)) if n > 1 else {}
    obs['z'] = np.array([0.5 for _ in range(n)], dtype=object)
    obs['x'] = np.array([0.5 if q == 0 else None for q in range(n)], dtype=object)
    c = McClean(n, obs, L, axes=axes, angles=angles, entangler=entangler, ckpt_every=ckpt)
    if n <= 14:
        params = np.concatenate([np.repeat(np.arange(L * n), 2), [L * n - 1, 0, 0]])
    else:
        params = np.array([0, 1, n, n + 1, n + 2, n + 3, n + 4, 2])  # a group of more than the 4 circuits of a launch
    deltas = rs.uniform(-4, 4, params.size)
    got = c.shifted_term_probs(params, deltas, c.observable.terms)
    want = _shifted_probs(n, axes, angles, params, deltas, obs, entangler)
    assert np.max(np.abs(got - want)) <= 1e-12  # probabilities: sums of 2^21 squares, some 10^2 roundings each
    vo = sv.mcclean_forward(n, axes, angles, entangler=entangler)
    assert np.linalg.norm(c.state.vec - vo) <= 1e-12


@pytest.mark.parametrize('n,terms', [(3, 4), (7, 9), (8, 9), (11, 30), (12, 24), (13, 25), (18, 48), (21, 23)])
@pytest.mark.parametrize('dtype,tol', [('complex128', 1e-13), ('complex64', 1e-13)])
def test_term_probs(gpu, n, terms, dtype, tol):
    """Every bit range of the diagonal measurement: thread, wave, block and iteration bits."""
    from qradient_amd.physical_components import Observable, State
    rs = np.random.RandomState(n)
    zz = np.full((n, n), None)
    pairs = [(i, j) for i in range(n) for j in range(i + 1, n)]
    for k in rs.permutation(len(pairs))[:terms]:
        zz[pairs[k]] = 1.0
    obs = {'zz': zz, 'z': np.array([1.0] * n, dtype=object)}
    st = State(n, dtype=dtype)
    v = rs.standard_normal(2 ** n) + 1j * rs.standard_normal(2 ** n)
    st.vec = v / np.linalg.norm(v)
    got = st.term_probs(Observable(obs))
    m = np.abs(st.vec) ** 2  # the stored state: no rounding of its own here
    x = np.arange(2 ** n)
    sign = [1 - 2 * ((x >> (n - 1 - q)) & 1) for q in range(n)]
    want = [0.5 * (m.sum() + (m * sign[q]).sum()) for q in range(n)]
    want += [0.5 * (m.sum() + (m * sign[i] * sign[j]).sum()) for i, j in pairs if zz[i, j] is not None]
    assert np.max(np.abs(got - want)) <= tol


@pytest.mark.parametrize('n,p,weights,dtype', [(2, 1, 'unit', 'complex128'), (6, 3, 'real', 'complex128'),
                                               (6, 2, 'unit', 'complex128'), (7, 2, 'mixed', 'complex128')])
@pytest.mark.parametrize('kmax', [0, 4])
def test_qaoa_shift_sample(gpu, n, p, weights, dtype, kmax):
    """Against the reference's dense formulation; kmax = 4 splits a layer into passes."""
    from qradient_amd import _native
    from qradient_amd.circuit_logic import Qaoa
    rs = np.random.RandomState(n * p)
    zz = np.full((n, n), None)
    for i in range(n - 1):
        zz[i, i + 1] = 1.0 if weights == 'unit' else float(rs.uniform(0.3, 1.5))
    obs = {'zz': zz}
    if weights == 'mixed':
        obs['z'] = np.array([0.4 if q % 2 else None for q in range(n)], dtype=object)
    b, g = rs.uniform(-3, 3, p), rs.uniform(-2, 2, p)
    c = Qaoa(n, obs, p, dtype=dtype)
    if kmax and n > kmax:
        _native.call('qg_qaoa_tune', c._get_plan(), kmax, 2, 0, 16)
    np.random.seed(3)
    E, gr = c.sample_grad_dense(b, g, shot_num=17)
    after = np.random.random_sample()
    np.random.seed(3)
    Eo, go = ra.qaoa_sample_grad_dense(n, obs, b, g, 17)
    assert np.random.random_sample() == after
    assert abs(E - Eo) <= 1e-12
    assert np.max(np.abs(gr - go)) <= 1e-12


def test_qaoa_shift_sample_larger_equals_state_operations(gpu):
    """14 qubits: the copies of a layer against the State API, one gate at a time."""
    import ctypes

    from qradient_amd import _native
    from qradient_amd.circuit_logic import Qaoa
    from qradient_amd.physical_components import State
    n, p, shots = 14, 2, 9
    rs = np.random.RandomState(5)
    edges = sorted({tuple(sorted(rs.choice(n, 2, replace=False))) for _ in range(n)})
    obs = sv.maxcut_observable(n, edges)
    b, g = rs.uniform(0.2, 1, p), rs.uniform(0.2, 1, p)
    c = Qaoa(n, obs, p)
    terms = c.observable.classical_terms()
    arr, k = _native.terms_array(terms)
    u = rs.uniform(size=(p * 2 * (k + n), shots))
    idx = np.empty(u.shape, dtype=np.int32)
    ex = np.empty(k + 1)
    _native.call('qg_qaoa_shift_sample', c._get_plan(), arr, k, _native.dptr(b), _native.dptr(g), None, arr, k,
                 _native.dptr(ex), shots, _native.dptr(u), _native.iptr(idx))
    st = State(n, '+')
    st.gates = c._gates
    row = 2 * (k + n) + 2 * k + 2 * 3  # layer 1, qubit 3, +pi/2
    for i in range(2):
        st.exp_ham_classical(g[i])
        st.xrot_all(b[i])
    st.xrot(np.pi / 2, 3)
    assert np.array_equal(st.sample_basis(u[row]), idx[row])
    st.reset('+')
    st.exp_ham_classical(g[0])
    st.exp_ham_classical_component(-np.pi / 4, 2)  # layer 0, component 2, minus
    st.xrot_all(b[0])
    st.exp_ham_classical(g[1])
    st.xrot_all(b[1])
    assert np.array_equal(st.sample_basis(u[2 * 2 + 1]), idx[2 * 2 + 1])
    assert ctypes.sizeof(ctypes.c_int32) == idx.itemsize
