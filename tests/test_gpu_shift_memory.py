"""The scratch of shot-based QAOA gradients: a large circuit's stored states are
given back at the end of the call, so the plan's gradient runs find the memory
they would have without it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('n,p,dtype', [(24, 2, 'complex128'), (25, 2, 'complex64'), (16, 2, 'complex128')])
def test_scratch_is_given_back(gpu, n, p, dtype):
    import torch
    from qradient_amd.circuit_logic import Qaoa
    zz = np.full((n, n), None)
    zz[0, 1] = 1.0
    c = Qaoa(n, {'zz': zz}, p, dtype=dtype)
    c._get_plan()
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info(0)[0]
    b, g = np.array([0.3, 0.5]), np.array([0.4, 0.2])
    for _ in range(2):
        E, gr = c.sample_grad_dense(b, g, shot_num=3)
        # five stored states and a copy are 1.5 GiB at 24 qubits in complex128;
        # what stays is at most 512 MiB and the plan's descriptor tables
        assert free - torch.cuda.mem_get_info(0)[0] <= (512 + 64) << 20
    Eg, gg = c.grad_run(b, g)
    assert abs(E - Eg) <= (1e-12 if dtype == 'complex128' else 1e-6)
