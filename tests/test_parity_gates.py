"""CX . D . CX with D diagonal on the target runs as one gate on the parity of two lanes: states, <H>
and gradients against the gate-by-gate path, where the pattern is whole, broken by other gates on
its lanes, or overlaps another one, on lanes inside and outside the tiles, alone and in a batch.

Tolerance: 8 N eps per norm, as for the other register ops."""
import math

import numpy as np
import pytest

from qgate_amd.adjoint import ParametricCircuit, PauliSum

pytestmark = pytest.mark.gpu

DTYPES = [np.float64, np.float32]
X = np.array([[0, 1], [1, 0]])
T = np.diag([1, complex(math.cos(0.8), math.sin(0.8))])
BOTH = np.diag([complex(math.cos(0.2), math.sin(0.2)), complex(math.cos(1.1), -math.sin(1.1))])
H = np.array([[1, 1], [1, -1]]) / math.sqrt(2)
N_PARAMS = 9


def _circuit(n, dtype):
    rs = np.random.RandomState(100 + n)
    c, k, gates = ParametricCircuit(n, dtype), 0, n

    def rot(kind, q, controls=()):
        nonlocal k
        getattr(c, kind)(q, k % N_PARAMS, controls=controls)
        k += 1

    for q in range(n):
        c.gate(H, q)
    for step in range(3 * n):
        a, b, d = [int(v) for v in rs.choice(n, 3, replace=False)] if step % 3 else (step % n, (step + 1) % n, (step + 2) % n)
        kind = step % 9
        c.gate(X, b, controls=[a])
        if kind == 1:
            rot('rx', b)            # not diagonal
        if kind == 2:
            rot('ry', a)            # the control changes
        if kind == 3:
            c.gate(X, d, controls=[a])   # the control's lane is used in between
        if kind == 4:
            rot('rz', b, [d])       # controlled
        elif kind == 5:
            c.gate(T, b)
        elif kind == 6:
            c.gate(BOTH, b)
        else:
            rot('rz', b)
        if kind == 7:
            rot('rz', b)            # two in a row
        if kind == 8:
            rot('rx', d)            # on another lane
        c.gate(X, b, controls=[a if kind != 0 or step % 2 else d])
        rot('rx', int(rs.randint(n)))
        gates += 5
    return c, gates


@pytest.mark.parametrize('dtype', DTYPES)
@pytest.mark.parametrize('n', [4, 9, 12, 13, 14, 16])
def test_parity_gates(hip_module, dtype, n):
    from qgate_amd.batch import AdjointBatch
    h = PauliSum([(0.7, {0: 'Z', n - 1: 'Z'}), (-0.4, {1: 'X', n // 2: 'Y'}), (0.3, {n - 2: 'Y'}), (0.2, {3: 'X'})])
    params = np.linspace(-2.9, 2.7, N_PARAMS)
    ref, gates = _circuit(n, np.float64)
    ref.set_fusion('off')
    v0, g0 = ref.gradient(params, h)
    ref.expectation(params, h)
    s0 = ref.state()
    circ, _ = _circuit(n, dtype)
    v1, g1 = circ.gradient(params, h)
    circ.expectation(params, h)
    tol = 8 * gates * np.finfo(dtype).eps
    weight, terms = np.sum(np.abs(h.coefs)), 2 * 3 * n / N_PARAMS
    assert np.linalg.norm(circ.state() - s0) < tol
    assert abs(v1 - v0) < tol * weight and np.max(np.abs(g1 - g0)) < tol * weight * terms
    batch = AdjointBatch(dtype)
    for shift in (0.3, 0.):
        batch.add(circ, params + shift, h)
    values, grads = batch.run()
    assert abs(values[1] - v0) < tol * weight and np.max(np.abs(grads[1] - g0)) < tol * weight * terms
