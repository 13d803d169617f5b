"""Device memory of a McClean batch plan's tables: 4096 circuits of 14 qubits and
20 layers took 667 MB while every layer had passes of its own (2 x 20 x 2
descriptors of 1.3 KB and their partial rows a circuit); the multi-layer passes'
descriptors take their place, not more."""
import ctypes

import pytest

pytestmark = pytest.mark.gpu


def test_tables_of_a_large_batch(gpu):
    import torch
    from qradient_amd import _native
    ctx = _native.Context(0)
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info(0)[0]
    h = ctypes.c_void_p()
    _native.call('qg_mcclean_batch_plan', ctx.handle, 14, 20, _native.DTYPES['complex64'], _native.ENTANGLERS['cnot'],
                 4096, ctypes.byref(h))
    try:
        used = free - torch.cuda.mem_get_info(0)[0]
        print('tables {:.0f} MB'.format(used / 1e6), flush=True)
        assert used <= 600e6
    finally:
        _native.call('qg_plan_destroy', h)
