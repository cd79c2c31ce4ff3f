"""Circuits that run in one workgroup: <H>, gradient and final state, alone and in a batch, against
the gate-by-gate path in double precision.

Tolerance: each of N gates rounds the state by at most a few units in the last place, relative to
its norm, so <H> and each gradient term are off by at most about 4 N eps sum |c_k|."""
import math

import numpy as np
import pytest

from qgate_amd.adjoint import PauliSum
from tests import adjoint_checks as ac

pytestmark = pytest.mark.gpu

DTYPES = [np.float64, np.float32]
MAX_BITS = {np.float64: 12, np.float32: 13}


def _case(n, dtype, gates):
    spec = ac.mixed_spec(n, gates, seed=n, n_params=max(4, gates // 3))
    h = ac.random_observable(n, 7, seed=n + 40)
    params = np.random.RandomState(n).uniform(-math.pi, math.pi, spec.n_params)
    tol = 4 * gates * np.finfo(dtype).eps * np.sum(np.abs(h.coefs))
    return spec, h, params, tol


def _reference(spec, params, h):
    circ = spec.build(np.float64).set_fusion('off')
    value, grad = circ.gradient(params, h)
    circ.expectation(params, h)
    return value, grad, circ.state()


# one amplitude unit; below, at and above each width of workgroup; more gradient terms than one
# pass of the sweep holds
@pytest.mark.parametrize('dtype', DTYPES)
@pytest.mark.parametrize('n,gates', [(3, 30), (5, 60), (8, 90), (9, 420), (10, 120), (11, 420), (12, 150), (13, 400),
                                     (14, 60)])
def test_one_workgroup(hip_module, dtype, n, gates):
    from qgate_amd.batch import AdjointBatch
    spec, h, params, tol = _case(n, dtype, gates)
    value, grad, state = _reference(spec, params, h)
    circ = spec.build(dtype)
    v, g = circ.gradient(params, h)
    assert abs(v - value) < tol and np.max(np.abs(g - grad)) < tol
    circ.expectation(params, h)
    assert np.max(np.abs(circ.state() - state)) < 4 * gates * np.finfo(dtype).eps
    # other parameters in the same batch do not mix with these
    batch = AdjointBatch(dtype)
    for k in range(3):
        batch.add(circ, params + 0.1 * (k - 1), h)
    values, grads = batch.run()
    assert abs(values[1] - value) < tol and np.max(np.abs(grads[1] - grad)) < tol
    v0, g0 = circ.gradient(params - 0.1, h)
    assert abs(values[0] - v0) < tol and np.max(np.abs(grads[0] - g0)) < tol
    (group,) = batch.tuning
    bits = 9 if n <= 9 else 11 if n <= 11 else n
    if n <= MAX_BITS[dtype]:
        assert (group['tile_bits'], group['threads']) == (bits, 2 ** bits // 8)


@pytest.mark.parametrize('dtype', DTYPES)
def test_groups_of_every_width_in_one_batch(hip_module, dtype):
    """Groups of one and of many items, in every width and beyond, and new parameters on replay."""
    from qgate_amd.batch import AdjointBatch
    batch = AdjointBatch(dtype)
    cases = []
    for n, items in ((13, 1), (3, 5), (11, 2), (14, 2), (9, 300), (12, 3)):
        spec, h, params, tol = _case(n, dtype, 40)
        circ = spec.build(dtype)
        for k in range(items):
            cases.append((circ, params + 0.01 * k, h, tol))
            batch.add(circ, params + 0.01 * k, h)
    for shift in (0., 0.5, -0.25):
        for i, (circ, params, h, tol) in enumerate(cases):
            batch.set_params(i, params + shift)
        values, grads = batch.run()
        for i in list(range(0, len(cases), 37)) + [0, 1, 6, 8, len(cases) - 1]:
            circ, params, h, tol = cases[i]
            v, g = circ.gradient(params + shift, h)
            assert abs(values[i] - v) < tol and np.max(np.abs(grads[i] - g)) < tol


@pytest.mark.parametrize('dtype', DTYPES)
def test_circuits_without_gates_or_parameters(hip_module, dtype):
    from qgate_amd.adjoint import ParametricCircuit
    from qgate_amd.batch import AdjointBatch
    h = PauliSum([(0.5, {0: 'Z'}), (0.25, {1: 'X'})])
    empty, fixed = ParametricCircuit(2, dtype), ParametricCircuit(2, dtype)
    fixed.gate(np.array([[1, 1], [1, -1]]) / math.sqrt(2), 1)
    batch = AdjointBatch(dtype)
    for circ, want in ((empty, 0.5), (fixed, 0.75)):
        v, g = circ.gradient(np.zeros(0), h)
        assert abs(v - want) < 1e-6 and len(g) == 0
        batch.add(circ, np.zeros(0), h)
    values, grads = batch.run()
    assert np.max(np.abs(values - [0.5, 0.75])) < 1e-6 and all(len(g) == 0 for g in grads)


@pytest.mark.parametrize('dtype', DTYPES)
def test_terms_wider_than_a_tile_stay_refused(hip_module, dtype):
    n = MAX_BITS[dtype]
    spec, h, params, tol = _case(n, dtype, 30)
    wide = PauliSum([(1., {q: 'X' for q in range(n)})])
    circ = spec.build(dtype)
    with pytest.raises(Exception):
        circ.expectation(params, wide)
    v, g = circ.gradient(params, h)
    assert abs(v - _reference(spec, params, h)[0]) < tol
