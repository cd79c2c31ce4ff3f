"""Device blocks above 1 GiB are kept after free, reused by size, and bounded at 8 GiB."""
import ctypes
import gc
import time

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


@pytest.mark.parametrize('order', ['small first', 'large first'])
def test_one_bound_for_blocks_of_all_sizes(hip_module, order):
    """After 7 GiB of complex128 states of 26 qubits (1 GiB, a power-of-two class) and 6 GiB of 27 and 28
    (large blocks) are freed, all that stays is 8 GiB and 256 MiB; what another allocator may take.
    What was freed last is there again: neither size crowds out the other."""
    gc.collect()
    hip_module.module_finalize()
    hip_module.module_init()
    keep = _state(hip_module, 4)
    before = _free_bytes(hip_module)
    small, large = [_state(hip_module, 26) for _ in range(7)], [_state(hip_module, n) for n in (27, 28)]
    for qs in small + large if order == 'small first' else large + small:
        qs.delete()
    for _ in range(50):                      # the driver takes freed memory back with a delay
        kept = before - _free_bytes(hip_module)
        print(order, kept / GIB)
        if kept <= LARGE_MAX + GIB // 2:
            break
        time.sleep(0.1)
    assert kept <= LARGE_MAX + GIB // 2 and kept >= 7 * GIB - GIB // 2
    again = [_state(hip_module, 28)] if order == 'small first' else [_state(hip_module, 26) for _ in range(4)]
    assert before - _free_bytes(hip_module) <= kept + GIB // 2
    for qs in again + [keep]:
        qs.delete()
