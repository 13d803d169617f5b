"""Gradient runs whose first adjoint pass forms lambda and E (states of 32 MiB and
more), in batches and replayed as a graph: bitwise the results of single, direct
runs, run after run, with other angles (batches: other weights and term counts) in
between."""
import numpy as np
import pytest

from oracle import statevector as sv

pytestmark = pytest.mark.gpu

SHAPES = [(21, 3, 'complex128'), (22, 3, 'complex64'), (23, 2, 'complex64')]


@pytest.mark.parametrize('n,L,dtype', SHAPES)
@pytest.mark.parametrize('entangler', ['cnot', 'cz'])
def test_batch_equals_single_runs(gpu, n, L, dtype, entangler):
    from qradient_amd.batch import McCleanBatch
    from qradient_amd.circuit_logic import McClean
    B = 3
    rs = np.random.RandomState(n + L)
    mb = McCleanBatch(n, L, B, dtype=dtype, entangler=entangler)
    for terms in (n - 1, 2):
        axes, angles = (3 * rs.rand(B, L, n)).astype(np.int32), 2 * np.pi * rs.rand(B, L, n)
        obs = sv.zz_chain_observable(n, rs.standard_normal(n - 1))
        obs['zz'][terms:] = None
        E, g = mb.grad_run(axes, angles, obs)
        for b in range(B):
            c = McClean(n, obs, L, axes=axes[b], angles=angles[b], dtype=dtype, entangler=entangler)
            Eb, gb = c.grad_run()
            c._destroy_plan()
            assert E[b] == Eb and np.array_equal(g[b], gb), b


@pytest.mark.parametrize('n,L,dtype', SHAPES + [(16, 4, 'complex64')])
@pytest.mark.parametrize('ckpt', [0, 1])
def test_graph_replays_equal_direct_runs(gpu, n, L, dtype, ckpt):
    from qradient_amd.circuit_logic import McClean
    from qradient_amd.physical_components import State
    rs = np.random.RandomState(n * L)
    scratch = State(12)
    w = rs.standard_normal(n - 1)
    replayed = McClean(n, sv.zz_chain_observable(n, w), L, dtype=dtype, ckpt_every=ckpt, graph=True)
    direct = McClean(n, sv.zz_chain_observable(n, w), L, dtype=dtype, ckpt_every=ckpt)
    for rep in range(4):
        axes, angles = sv.mcclean_random_params(L, n, rs)
        for c in (replayed, direct):
            c.axes, c.angles = axes, angles
        E1, g1 = replayed.grad_run()
        scratch.xrot(0.3 * rep, rep % 12)  # other device work between replays
        E0, g0 = direct.grad_run()
        assert E1 == E0 and np.array_equal(g1, g0), rep
