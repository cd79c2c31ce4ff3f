"""CX . D . CX with D diagonal on the target runs as one gate on the parity of two lanes: states, <H>
and gradients against the gate-by-gate path, where the pattern is whole, broken by other gates on
its lanes, or overlaps another one, on lanes inside and outside the tiles, alone and in a batch.

Tolerance: 8 N eps per norm, as for the other register ops."""
import math

import numpy as np
import pytest

from qgate_amd.adjoint import ParametricCircuit, PauliSum
from qgate_amd.model import gate_type as gtype
from qgate_amd.simulator.simulator import Simulator
from tests.helpers import tol
from tests.test_dense_fusion import _prepared, _read

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


# Queues that leave a pass nothing but parity gates, or parity gates and others on their target
# alone: (control, target) of each CX . D . CX, or the lane of a gate of its own.
QUEUES = {
    'one': [(0, 1)], 'reversed': [(9, 2)], 'far': [(12, 13)], 'near and far': [(13, 0)],
    'star': [(0, 5), (3, 5), (12, 5)], 'two': [(1, 6), (6, 1)], 'gate before': [7, (2, 7)],
    'gate after': [(2, 7), 7], 'gates around': [11, (13, 11), 11], 'chain': [(0, 1), (1, 2), (2, 3), (12, 13)],
}


def _queue(name, diagonal):
    """name's gates as (gate type, controls, target)."""
    out = []
    for k, at in enumerate(QUEUES[name]):
        if isinstance(at, int):
            out.append((gtype.U(0.7 + k, 0.3, 1.9), [], at))
        else:
            out += [(gtype.X(), [at[0]], at[1]), (diagonal(0.9 - k), [], at[1]), (gtype.X(), [at[0]], at[1])]
    return out


@pytest.mark.parametrize('dtype', DTYPES)
@pytest.mark.parametrize('diagonal', [gtype.RZ, gtype.U1])
@pytest.mark.parametrize('tile_bits', [0, 10, 13])
@pytest.mark.parametrize('name', sorted(QUEUES))
def test_queues_of_parity_gates(hip_module, port_module, name, tile_bits, diagonal, dtype):
    """Short queues on a random state of 14 lanes, applied by the next read, against the oracle, which
    applies every gate; tiles of the default size, a smaller and the widest one."""
    n, states = 14, []
    for module, real, read in ((hip_module, dtype, lambda qs: _read(hip_module, qs, n, dtype)),
                               (port_module, np.float64, lambda qs: qs.local_states())):
        qs = _prepared(module, n, real, 5)
        proc = qs.processor
        if module is hip_module:
            proc.set_fusion('tile', tile_bits)
        for gate, controls, target in _queue(name, diagonal):
            if controls:
                proc.apply_controlled_gate(gate, False, qs, controls, target)
            else:
                proc.apply_gate(gate, False, qs, target)
        states.append(read(qs))
        qs.delete()
    assert np.max(np.abs(states[0] - states[1])) < tol(dtype)


@pytest.mark.parametrize('dtype', DTYPES)
def test_trotter_steps_between_reads(hip_module, port_module, dtype):
    """Simulator.run of one step at a time, its state read after each."""
    from qgate_amd.script import ctrl, H as had, Rx, Rz, new_qregs
    n, out = 14, []
    for module, real in ((hip_module, dtype), (port_module, np.float64)):
        q = new_qregs(n)
        if module is hip_module:
            module.set_fusion('tile')
        try:
            sim = Simulator(module, circuit_prep='one_static', dtype=real)
            sim.qubits.set_ordering(list(q))
            sim.run([had(x) for x in q] + [Rx(0.1 * k)(x) for k, x in enumerate(q)])
            states = []
            for a, b in ((0, 1), (5, 13), (12, 11)):
                sim.run([ctrl(q[a]).X(q[b]), Rz(0.4 + a)(q[b]), ctrl(q[a]).X(q[b])])
                states.append(np.array(sim.qubits.states[:]))
            out.append(np.array(states))
            sim.terminate()
        finally:
            hip_module.set_fusion('off')
    assert np.max(np.abs(out[0] - out[1])) < tol(dtype)


@pytest.mark.parametrize('dtype', DTYPES)
@pytest.mark.parametrize('n', [14, 16])
def test_parity_gates_left_to_the_forward_pass(hip_module, dtype, n):
    """<H> and gradient, above the sizes of one workgroup, where the first pass is full and leaves the
    next one a rotation and the ZZ edges of its lane; tolerance as above."""
    last = 12 if dtype == np.float32 else 11     # lanes 0 .. last - 1 fill a tile
    h = PauliSum([(0.7, {last: 'X'}), (-0.4, {last: 'Y'}), (0.3, {0: 'X', last: 'Y'})])
    for controls in ([0], [0, 4, last - 1]):
        results = []
        for mode, real in (('off', np.float64), ('tile', dtype)):
            c, gates = ParametricCircuit(n, real), 2 * last
            for q in range(last + 1):
                c.rx(q, q)
            for q in range(last - 1):
                c.gate(np.diag([1, -1]), q + 1, controls=[q])
            for k, a in enumerate(controls):
                c.gate(X, last, controls=[a])
                c.rz(last, last + 1 + k)
                c.gate(X, last, controls=[a])
                gates += 3
            c.set_fusion(mode)
            params = np.linspace(0.5, 1.9, c.n_params)
            results.append((*c.gradient(params, h), c.expectation(params, h), c.state()))
        (v0, g0, e0, s0), (v1, g1, e1, s1) = results
        bound = 8 * gates * np.finfo(dtype).eps
        assert np.linalg.norm(s1 - s0) < bound
        assert max(abs(v1 - v0), abs(e1 - e0), np.max(np.abs(g1 - g0))) < bound * np.sum(np.abs(h.coefs))
