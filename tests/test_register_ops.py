"""Gates as the register passes apply them (diagonals as a global phase and a ratio, rotations
without their common factor, swaps, general matrices), on register, lane, wave and outer bits and
with controls there, against the gate-by-gate path.

Tolerance: the two paths round each of N gates differently by a few units in the last place of the
state's norm; 8 N eps times the norms that enter a result."""
import math

import numpy as np
import pytest

from qgate_amd.adjoint import ParametricCircuit, PauliSum

pytestmark = pytest.mark.gpu

DTYPES = [np.float64, np.float32]


def _e(x):
    return complex(math.cos(x), math.sin(x))


FIXED = {
    'phase': np.diag([1, _e(0.3)]), 'z': np.diag([1, -1]), 'both': np.diag([_e(0.7), _e(-1.9)]),
    'equal': np.diag([_e(0.4), _e(0.4)]), 'minus': np.diag([-1, -1]), 'scaled': np.diag([1.5, 0.75j]),
    'zero': np.diag([0, 1]), 'x': np.array([[0, 1], [1, 0]]), 'y': np.array([[0, -1j], [1j, 0]]),
    'h': np.array([[1, 1], [1, -1]]) / math.sqrt(2), 'real': np.array([[1, 2], [-2, 1]]) / math.sqrt(5),
    'general': np.array([[0.6, 0.8j], [0.3 - 0.2j, 1.1]]),
}
ANGLES = [0., math.pi, -math.pi, math.pi / 2, -math.pi / 2, 1e-9, math.pi - 1e-9, 2 * math.pi, 0.1, 2.5]


def _circuit(n, dtype, unitary):
    """Every fixed gate and every rotation kind on lanes and controls over the whole state."""
    rs = np.random.RandomState(n)
    c, k, gates = ParametricCircuit(n, dtype), 0, 0
    names = [m for m in sorted(FIXED) if not unitary or m not in ('scaled', 'zero', 'general')]
    for q in range(n):
        c.gate(FIXED['h'], q)
    for step in range(2 * n):
        q = step % n
        others = [int(v) for v in rs.permutation([v for v in range(n) if v != q])]
        for rot in (c.rz, c.rx, c.ry, c.rz):
            rot(q, k % len(ANGLES), controls=others[:max(0, step % 4 - 1)])
            k += 1
        for j in range(2):
            c.gate(FIXED[names[(2 * step + j) % len(names)]], others[j], controls=others[j + 1:j + 1 + step % 3])
        gates += 6
    return c, gates + n


@pytest.mark.parametrize('dtype', DTYPES)
@pytest.mark.parametrize('unitary', [True, False])
@pytest.mark.parametrize('n', [9, 12, 14, 15])
def test_ops_on_every_kind_of_bit(hip_module, dtype, n, unitary):
    h = PauliSum([(0.7, {0: 'Z', n - 1: 'Z'}), (-0.4, {1: 'X', n // 2: 'Y'}), (0.3, {n - 2: 'Y'}), (0.2, {3: 'X'})])
    params = np.array(ANGLES)
    out = {}
    for mode in ('off', 'tile'):
        circ, gates = _circuit(n, np.float64 if mode == 'off' else dtype, unitary)
        circ.set_fusion(mode)
        value = circ.expectation(params, h)
        state = circ.state()
        out[mode] = (value, state, circ.gradient(params, h)[1])
    (v0, s0, g0), (v1, s1, g1) = out['off'], out['tile']
    tol = 8 * gates * np.finfo(dtype).eps
    norm = float(np.linalg.norm(s0))
    assert np.linalg.norm(s1 - s0) < tol * norm
    assert abs(v1 - v0) < tol * norm * norm * np.sum(np.abs(h.coefs))
    if unitary:   # the sweep un-computes with U^dagger
        terms = 4 * 2 * n / len(ANGLES)
        assert np.max(np.abs(g1 - g0)) < tol * terms * np.sum(np.abs(h.coefs))


@pytest.mark.parametrize('diagonals', [False, True])
def test_a_run_on_one_lane_rounds_once(hip_module, diagonals):
    """4000 gates on one lane, in complex128, become one gate whose product is formed in extended
    precision: its amplitudes are off by the roundings of that gate's parts (a diagonal, a rotation, a
    diagonal, their product and its application, at most 2^-53 each and two components: 12 of them),
    not by those of 4000 products (13 and 14 2^-53 when each was rounded). Up to norm and phase, which the split drops from
    matrices that are rounded themselves."""
    from tests.test_dense_fusion import _read
    rs = np.random.RandomState(3)
    n, lane = 14, 9
    qs = hip_module.create_qubit_states(np.float64)
    proc = qs.processor
    proc.set_fusion('tile')
    proc.initialize_qubit_states(qs, n)
    proc.reset_qubit_states(qs)
    want = np.array([1, 0], np.clongdouble)
    for k in range(4000):
        t = rs.uniform(-3, 3)
        m = np.array([[math.cos(t), -math.sin(t)], [math.sin(t), math.cos(t)]], complex)
        if diagonals and k % 2:
            m = np.diag([_e(-t), _e(t)])
        proc.apply_matrix(m, qs, [], lane)
        want = m.astype(np.clongdouble) @ want
    out = _read(hip_module, qs, n, np.float64)
    qs.delete()
    got = out[[0, 1 << lane]].astype(np.clongdouble)
    got, want = (v / np.sqrt(np.sum(np.abs(v) ** 2)) for v in (got, want))
    phase = np.sum(np.conj(want) * got)
    error = float(np.sqrt(np.sum(np.abs(got - want * phase / np.abs(phase)) ** 2))) * 2. ** 53
    print('error', error)
    assert error < 12


FAR = {
    'ratio': np.diag([2e-30, 1e9]), 'small': np.diag([1e-25, 1e25j]), 'large': np.diag([1e20j, 1e-15]),
    'ry': 1e-25 * np.array([[0.8, -0.6], [0.6, 0.8]]), 'rx': 1e18 * np.array([[0.6, -0.8j], [-0.8j, 0.6]]),
}
FAR_DOUBLE = {   # squares and quotients beyond the range of FP64 itself
    'ratio64': np.diag([1e-25, 1e290]), 'ry64': 1e-200 * np.array([[0.8, -0.6], [0.6, 0.8]]),
    'rx64': 1e200 * np.array([[0.6, -0.8j], [-0.8j, 0.6]]),
}


@pytest.mark.parametrize('dtype,name', [(np.float32, m) for m in sorted(FAR)] +
                         [(np.float64, m) for m in sorted({**FAR, **FAR_DOUBLE})])
@pytest.mark.parametrize('controls', [0, 1])
def test_matrices_far_from_unitary(hip_module, dtype, name, controls):
    """Entries that the state's precision holds give the amplitudes that the gate-by-gate path gives,
    each within 32 eps, though their quotient or their squares leave its range."""
    from tests.test_dense_fusion import _prepared, _read
    n, m = 14, {**FAR, **FAR_DOUBLE}[name]
    h = FIXED['h']
    for target in (0, 5, 9, 13):
        out = []
        for mode in ('off', 'tile'):
            qs = _prepared(hip_module, n, dtype, 4)
            qs.processor.set_fusion(mode)
            for mat, ctrl, q in ((h, [], 3), (m, [7] * controls, target), (h, [], 4)):
                qs.processor.apply_matrix(mat, qs, ctrl, q)
            out.append(_read(hip_module, qs, n, dtype))
            qs.delete()
        off, tile = out
        assert np.all(np.isfinite(off.view(np.float64)))
        scale = np.max(np.abs(off).reshape(-1, 4, 8), 1)   # of the amplitudes that the H gates mix
        assert np.max(np.abs(tile - off).reshape(-1, 4, 8) / scale[:, None]) < 32 * np.finfo(dtype).eps
