"""Laying a plan out for a smaller shape allocates nothing, also where the
smaller shape takes more multi-layer passes (below 20 qubits the tile is
smaller: at 40 layers 29 passes of 19 qubits against 24 of 22, complex128)."""
import ctypes

import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('dtype', ['complex64', 'complex128'])
@pytest.mark.parametrize('entangler', ['cnot', 'cz'])
def test_smaller_shapes_allocate_nothing(gpu, dtype, entangler):
    import torch
    from qradient_amd import _native
    L = 6000  # tables of many megabytes: an allocation shows in the free memory
    ctx = _native.Context(0)
    plan = ctypes.c_void_p()
    _native.call('qg_mcclean_plan', ctx.handle, 22, L, _native.DTYPES[dtype], _native.ENTANGLERS[entangler], 0,
                 ctypes.byref(plan))
    try:
        free = torch.cuda.mem_get_info(0)[0]
        for n in (21, 20, 19, 17, 16, 15, 14, 22):
            _native.call('qg_plan_reshape', plan, n, L, 0)
            assert torch.cuda.mem_get_info(0)[0] == free, n
    finally:
        _native.call('qg_plan_destroy', plan)
