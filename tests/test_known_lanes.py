"""Collapses and probabilities after earlier collapses visit only the amplitudes those left.

Random programs make the same processor calls on the HIP runtime and on the CPU oracle, which
visits every amplitude, in double precision (its float32 probabilities are float32 sums):
collapses (both outcomes, the same lane again, a lane collapsed onto the
value it does not have), probabilities of collapsed and free lanes, and every kind of write in
between that may end what is known. Lanes: inside a complex64 unit (0), inside a 128-byte line,
inside a wavefront's units and above; the smallest states, where no lane is fixed, too.
"""
import numpy as np
import pytest

from qgate_amd.model import gate_type as gtype
from tests.helpers import tol
from tests.test_dense_fusion import _prepared, _read

pytestmark = pytest.mark.gpu


def _program(proc, qs, n, seed, probs):
    rs = np.random.RandomState(seed)
    measured = {}
    for _ in range(40):
        kind = rs.choice(['measure', 'measure', 'measure', 'prob', 'again', 'gate', 'controlled', 'reset'])
        lane = int(rs.randint(n))
        if kind == 'measure':
            p = proc.calc_probability(qs, lane)
            probs.append(p)
            v = int(rs.randint(2))
            if min(p, 1. - p) < 0.3:       # keeps the norm of the collapse moderate
                v = 0 if p >= 0.5 else 1
            proc.decohere(v, p, qs, lane)
            measured[lane] = v
        elif kind == 'prob':
            probs.append(proc.calc_probability(qs, lane))
        elif kind == 'again' and measured:
            lane = sorted(measured)[int(rs.randint(len(measured)))]
            v = measured[lane]
            proc.decohere(v, 1. - v, qs, lane)
        elif kind == 'gate':
            proc.apply_gate(gtype.U(*rs.uniform(0, 6.3, 3)), False, qs, lane)
            measured.clear()
        elif kind == 'controlled' and n > 1:
            c = int((lane + 1 + rs.randint(n - 1)) % n)
            proc.apply_controlled_gate(gtype.H(), False, qs, [c], lane)
            measured.clear()
        elif kind == 'reset' and measured.get(lane) == 1:
            proc.apply_reset(qs, lane)
            measured.clear()
    probs.append(proc.calc_probability(qs, n - 1))


@pytest.mark.parametrize('dtype', [np.float64, np.float32])
@pytest.mark.parametrize('n,seed', [(1, 1), (2, 2), (4, 3), (7, 4), (10, 5), (13, 6), (13, 7), (14, 8)])
def test_random_programs_match_oracle(hip_module, port_module, n, seed, dtype):
    results = []
    for module, real, read in ((hip_module, dtype, lambda qs: _read(hip_module, qs, n, dtype)),
                               (port_module, np.float64, lambda qs: qs.local_states())):
        qs = _prepared(module, n, real, seed)
        probs = []
        _program(qs.processor, qs, n, seed, probs)
        results.append((np.array(probs), read(qs)))
        qs.delete()
    (gp, g), (wp, w) = results
    assert np.max(np.abs(gp - wp)) < tol(dtype), (gp, wp)
    assert np.max(np.abs(g - w)) < tol(dtype)


@pytest.mark.parametrize('dtype', [np.float64, np.float32])
@pytest.mark.parametrize('lane', [0, 2, 5, 9])
def test_collapse_onto_the_value_a_lane_does_not_have(hip_module, dtype, lane):
    """A finite norm leaves the zero vector; an infinite one makes every kept amplitude NaN,
    those that an earlier collapse had cleared included."""
    n = 11
    for prob, want in ((0.5, 'zero'), (0., 'nan')):
        qs = _prepared(hip_module, n, dtype, 3)
        proc = qs.processor
        p = proc.calc_probability(qs, lane)
        proc.decohere(1, p, qs, lane)
        p = proc.calc_probability(qs, 10)
        proc.decohere(0 if p > 0.5 else 1, p, qs, 10)
        proc.decohere(0, prob, qs, lane)
        out = _read(hip_module, qs, n, dtype)
        kept = (np.arange(1 << n) >> lane) & 1 == 0
        assert np.all(out[~kept] == 0.)
        assert np.all(out[kept] == 0.) if want == 'zero' else np.all(np.isnan(out[kept].real))
        qs.delete()


def _use_lane_again(proc, qs, n, lane, gate, probs):
    """Measures `lane`, applies `gate` to it, and reads every lane; then collapses `lane` again."""
    other = (lane + 2) % n
    for q, want in ((other, 0), (lane, 1), (lane, 0)):   # both outcomes, after an earlier collapse
        p = proc.calc_probability(qs, q)
        probs.append(p)
        proc.decohere(want, p, qs, q)
        if gate == 'controlled':
            proc.apply_controlled_gate(gtype.U(0.9, 0.4, 1.3), False, qs, [other], lane)
            proc.apply_controlled_gate(gtype.U(1.1, 0.2, 0.7), False, qs, [lane], other)
        proc.apply_gate(gtype.X() if gate == 'X' else gtype.U(1.2, 0.5, 2.1), False, qs, q)
        probs += [proc.calc_probability(qs, k) for k in range(n)]
    p = proc.calc_probability(qs, lane)
    if min(p, 1. - p) > 0.1:
        proc.decohere(1, p, qs, lane)
    probs += [proc.calc_probability(qs, k) for k in range(n)]


@pytest.mark.parametrize('dtype', [np.float64, np.float32])
@pytest.mark.parametrize('fusion', ['off', 'tile', 'dense'])
@pytest.mark.parametrize('gate', ['U', 'X', 'controlled'])
@pytest.mark.parametrize('lane', [2, 3, 4, 5, 8, 12])
def test_gate_on_the_lane_just_collapsed(hip_module, port_module, lane, gate, fusion, dtype):
    """A gate ends what a collapse that is launched together with it made known of its lane."""
    n, results = 13, []
    for module, real, read in ((hip_module, dtype, lambda qs: _read(hip_module, qs, n, dtype)),
                               (port_module, np.float64, lambda qs: qs.local_states())):
        qs = _prepared(module, n, real, 21)
        if module is hip_module:
            qs.processor.set_fusion(fusion)
        probs = []
        _use_lane_again(qs.processor, qs, n, lane, gate, probs)
        results.append((np.array(probs), read(qs)))
        qs.delete()
    (gp, g), (wp, w) = results
    assert np.max(np.abs(gp - wp)) < tol(dtype), (gp, wp)
    assert np.max(np.abs(g - w)) < tol(dtype)
