"""Device blocks above 1 GiB are kept after free, reused by size, and bounded at 8 GiB."""
import ctypes
import gc

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GIB = 1 << 30
LARGE_MAX = 8 * GIB


def _free_bytes(module):
    """Free device memory, from the HIP runtime that the library itself loaded."""
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert module.lib().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def _state(module, n):
    qs = module.create_qubit_states(np.float64)
    qs.processor.initialize_qubit_states(qs, n)
    qs.processor.reset_qubit_states(qs)
    return qs


@pytest.mark.parametrize('sizes', [(27,), (27, 28, 29), (29, 27, 28, 27), (30, 27)])
def test_large_blocks_are_reused_and_bounded(hip_module, sizes):
    """complex128 states of 2^n amplitudes (27: 2 GiB .. 30: 16 GiB, beyond the bound)."""
    gc.collect()
    free_before = None
    for turn in range(2):
        states = [_state(hip_module, n) for n in sizes]
        for qs, n in zip(states, sizes):
            assert qs.processor.calc_probability(qs, n - 1) == 1.
        for qs in states:
            qs.delete()
        free = _free_bytes(hip_module)
        kept = sum(16 << n for n in sizes)
        if turn and kept <= LARGE_MAX:       # the second turn took the first one's blocks
            assert abs(free - free_before) < GIB // 2
        free_before = free
    hip_module.module_finalize()             # everything is given back
    given_back = _free_bytes(hip_module)
    hip_module.module_init()
    assert given_back >= free_before
    assert given_back - free_before <= 2 * LARGE_MAX + GIB
    fits = [16 << n for n in sizes if (16 << n) <= LARGE_MAX]
    assert given_back - free_before >= min(max(fits), LARGE_MAX) - GIB // 2
