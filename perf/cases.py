"""Performance cases: what a user of the simulator has it do, through its public entry points.

Four kinds of call, from one training step of a 6-qubit circuit to a 30-qubit circuit:

  gradient   <H> and its gradient for one parameterised circuit (qgate_amd.adjoint.Expectation,
             forward and backward), the inner step of a variational optimisation
  batch      the same for many circuits of uneven sizes at once (qgate_amd.batch.AdjointBatch)
  circuit    Simulator.run of a whole circuit, then its output: all amplitudes, or the joint
             distribution of a register; with measurements in the circuit, also their outcomes
  pool       a sampling pool over every qubit of a state with draws from it, and the distribution
             of some of its qubits in another order

complex64 results are returned in 32 bits (float32 parameters, as a torch model holds them),
complex128 results in 64.
"""
import math
import random

import numpy as np
import torch

from qgate_amd import script
from qgate_amd.adjoint import Expectation, ParametricCircuit, PauliSum
from qgate_amd.batch import AdjointBatch
from qgate_amd.model import gate_type
from qgate_amd.simulator import hipruntime
from qgate_amd.simulator.simulator import Simulator

REAL = {'complex64': np.float32, 'complex128': np.float64}
TORCH_REAL = {'complex64': torch.float32, 'complex128': torch.float64}


def listed():
    return [
        # the smallest training step: a toy problem or a subcircuit in a hybrid model, called
        # thousands of times; launches and synchronisations are all of it
        {'name': 'gradient_6q_c128', 'kind': 'gradient', 'ansatz': 'hea', 'qubits': 6, 'layers': 3,
         'dtype': 'complex128'},
        # an ordinary variational step, on a circuit of ZZ and X rotations
        {'name': 'gradient_13q_c64', 'kind': 'gradient', 'ansatz': 'ising', 'qubits': 13, 'layers': 6,
         'dtype': 'complex64'},
        # a larger one in double precision, odd qubit count
        {'name': 'gradient_19q_c128', 'kind': 'gradient', 'ansatz': 'hea', 'qubits': 19, 'layers': 8,
         'dtype': 'complex128'},
        # the benchmark's ansatz: 24 qubits, 12 layers, 576 parameters
        {'name': 'gradient_24q_c64', 'kind': 'gradient', 'ansatz': 'hea', 'qubits': 24, 'layers': 12,
         'dtype': 'complex64'},
        # a minibatch of small circuits (one per data sample)
        {'name': 'batch_96x6_11q_c64', 'kind': 'batch', 'circuits': 96, 'low': 6, 'high': 11, 'layers': 4,
         'dtype': 'complex64'},
        # the benchmark's batch of circuits of 8..20 qubits, an eighth of its count
        {'name': 'batch_512x8_20q_c64', 'kind': 'batch', 'circuits': 512, 'low': 8, 'high': 20, 'layers': 10,
         'dtype': 'complex64'},
        # a small circuit with the simulator's defaults (float64, dynamic preparation, no
        # fusion) and its state vector: what a notebook does
        {'name': 'circuit_10q_c128', 'kind': 'circuit', 'circuit': 'brickwork', 'qubits': 10, 'gates': 120,
         'dtype': 'complex128', 'prep': 'dynamic', 'fusion': 'off', 'measured': 0, 'output': 'states'},
        # a deep circuit of middle size, fused, and its state vector
        {'name': 'circuit_20q_c64_tile', 'kind': 'circuit', 'circuit': 'brickwork', 'qubits': 20, 'gates': 600,
         'dtype': 'complex64', 'prep': 'one_static', 'fusion': 'tile', 'measured': 0, 'output': 'states'},
        # gate by gate in double precision: the largest that most users run without fusion
        {'name': 'circuit_27q_c128', 'kind': 'circuit', 'circuit': 'random', 'qubits': 27, 'gates': 100,
         'dtype': 'complex128', 'prep': 'one_static', 'fusion': 'off', 'measured': 0, 'output': 'register'},
        # the benchmark's 30-qubit random circuit, fused, a quarter of its gates
        {'name': 'circuit_30q_c64_tile', 'kind': 'circuit', 'circuit': 'random', 'qubits': 30, 'gates': 500,
         'dtype': 'complex64', 'prep': 'one_static', 'fusion': 'tile', 'measured': 0, 'output': 'register'},
        # a circuit that ends with a measurement of every qubit
        {'name': 'measure_25q_c64', 'kind': 'circuit', 'circuit': 'random', 'qubits': 25, 'gates': 75,
         'dtype': 'complex64', 'prep': 'one_static', 'fusion': 'tile', 'measured': 25, 'output': 'register'},
        # many shots of one state: pool and draws, and a marginal over some qubits
        {'name': 'pool_28q_c64', 'kind': 'pool', 'qubits': 28, 'dtype': 'complex64', 'shots': 200000, 'kept': 19},
    ]


def _log_int(rng, low, high):
    """An integer from low to high, spread over the logarithm."""
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    kind = rng.choice(['gradient', 'gradient', 'batch', 'circuit', 'circuit', 'circuit', 'pool'])
    dtype = rng.choice(['complex64', 'complex128'])
    if kind == 'gradient':
        n = rng.randint(4, 24 if dtype == 'complex64' else 23)
        return {'kind': kind, 'ansatz': rng.choice(['hea', 'hea', 'ising']), 'qubits': n,
                'layers': rng.randint(1, 12), 'dtype': dtype}
    if kind == 'batch':
        low = rng.randint(5, 12)
        high = rng.randint(low, min(low + 12, 19 if dtype == 'complex128' else 20))
        most = 512 if high < 17 else 2048 // (1 << (high - 15))
        return {'kind': kind, 'circuits': _log_int(rng, 16, most), 'low': low, 'high': high,
                'layers': rng.randint(2, 10), 'dtype': dtype}
    if kind == 'pool':
        n = rng.randint(12, 28 if dtype == 'complex64' else 27)
        return {'kind': kind, 'qubits': n, 'dtype': dtype, 'shots': _log_int(rng, 100, 1000000),
                'kept': rng.randint(1, min(n - 1, 22))}
    fusion = rng.choice(['off', 'off', 'tile', 'tile', 'tile', 'dense'])
    top = {'off': 27, 'tile': 29, 'dense': 27}[fusion] - (1 if dtype == 'complex128' else 0)
    n = rng.randint(4, top)
    gates = _log_int(rng, 20, {'off': 100, 'tile': 600, 'dense': 200}[fusion])
    return {'kind': 'circuit', 'circuit': rng.choice(['brickwork', 'random', 'random', 'qft']), 'qubits': n,
            'gates': gates, 'dtype': dtype,
            'prep': rng.choice(['one_static', 'one_static', 'dynamic']) if n <= 20 else 'one_static',
            'fusion': fusion, 'measured': rng.choice([0, 0, rng.randint(1, n)]),
            'output': rng.choice(['states', 'register']) if n <= 22 else 'register'}


# ---- circuits as plain lists: (name, controls, target, angles) ---------------------------

def _gates(kind, n, count, seed):
    r = random.Random(seed)
    angle = lambda: r.uniform(0., 2. * math.pi)  # noqa: E731
    out = []
    if kind == 'random':       # H on every qubit, then the benchmark's mix of kinds
        out += [('H', [], q, []) for q in range(n)]
        while len(out) < n + count:
            name = r.choice(['U3', 'H', 'Rz', 'CX', 'CCX'])
            lanes = r.sample(range(n), {'CX': 2, 'CCX': 3}.get(name, 1))
            out.append(('X' if name in ('CX', 'CCX') else name, lanes[:-1], lanes[-1],
                        [angle() for _ in range({'U3': 3, 'Rz': 1}.get(name, 0))]))
    elif kind == 'brickwork':  # U3 on every qubit, then CX on alternating neighbours
        layer = 0
        while len(out) < count:
            out += [('U3', [], q, [angle(), angle(), angle()]) for q in range(n)]
            out += [('X', [q], q + 1, []) for q in range(layer % 2, n - 1, 2)]
            layer += 1
    else:                      # a random product state, then the QFT
        out += [('U3', [], q, [angle(), angle(), angle()]) for q in range(n)]
        for i in reversed(range(n)):
            out.append(('H', [], i, []))
            out += [('U1', [j], i, [math.pi / (1 << (i - j))]) for j in reversed(range(i))]
    return out


def _ops(gates, q):
    out = []
    for name, controls, target, angles in gates:
        on = script.ctrl(*[q[c] for c in controls]) if controls else script
        gate = getattr(on, name)
        out.append((gate(*angles) if angles else gate)(q[target]))
    return out


def _measured_qubits(case):
    """The qubits that are measured at the end, and the register whose distribution is read."""
    n = case['qubits']
    step = 7 if n % 7 else 5     # not one after another
    order = [(k * step) % n for k in range(n)] if math.gcd(step, n) == 1 else list(range(n))
    return order[:case['measured']], list(range(n - 1, max(-1, n - 17), -1))


# ---- ansatz circuits: (name, controls, target, parameter index or None) -------------------

def _ansatz(kind, n, layers):
    out = []
    if kind == 'hea':          # RY and RZ on every qubit, then a ring of CZ
        k = 0
        for _ in range(layers):
            for name in ('RY', 'RZ'):
                for q in range(n):
                    out.append((name, [], q, k))
                    k += 1
            out += [('Z', [q], (q + 1) % n, None) for q in range(n)]
        return out, k
    out += [('H', [], q, None) for q in range(n)]
    for layer in range(layers):   # exp(-i a Z Z / 2) on neighbours, then RX on every qubit
        for q in range(n - 1):
            out += [('X', [q], q + 1, None), ('RZ', [], q + 1, 2 * layer), ('X', [q], q + 1, None)]
        out += [('RX', [], q, 2 * layer + 1) for q in range(n)]
    return out, 2 * layers


def _parametric(kind, n, layers, dtype):
    c = ParametricCircuit(n, REAL[dtype])
    fixed = {'H': gate_type.H(), 'X': gate_type.X(), 'Z': gate_type.Z()}
    rot = {'RX': c.rx, 'RY': c.ry, 'RZ': c.rz}
    for name, controls, target, k in _ansatz(kind, n, layers)[0]:
        if k is None:
            c.gate(fixed[name], target, controls=controls)
        else:
            rot[name](target, k, controls=controls)
    return c


def _step(n, n_params, seed):
    """Parameters and the coefficients of sum a_i Z_i Z_i+1 + sum b_i X_i."""
    r = np.random.RandomState(seed % (1 << 32))
    return r.uniform(-math.pi, math.pi, n_params), r.normal(size=n - 1), r.normal(size=n)


def _batch_sizes(case):
    span = case['high'] - case['low'] + 1
    return [case['low'] + i % span for i in range(case['circuits'])]


# ---- prepare and run ----------------------------------------------------------------------

def prepare(case, seed):
    kind, dtype = case['kind'], case['dtype']
    if kind == 'gradient':
        n, layers = case['qubits'], case['layers']
        p, a, b = _step(n, _ansatz(case['ansatz'], n, layers)[1], seed)
        params = torch.tensor(p, dtype=TORCH_REAL[dtype], device='cuda', requires_grad=True)
        return {'kind': kind, 'params': params, 'circuit': _parametric(case['ansatz'], n, layers, dtype),
                'observable': PauliSum.zz_x(a, b)}
    if kind == 'batch':
        batch = AdjointBatch(REAL[dtype])
        circuits, params = {}, []
        for i, n in enumerate(_batch_sizes(case)):
            if n not in circuits:
                circuits[n] = _parametric('hea', n, case['layers'], dtype)
            p, a, b = _step(n, circuits[n].n_params, 4099 * seed + i)
            p = p.astype(REAL[dtype])
            batch.add(circuits[n], p, PauliSum.zz_x(a, b))
            params.append(p)
        return {'kind': kind, 'batch': batch, 'params': params, 'dtype': TORCH_REAL[dtype]}
    n = case['qubits']
    q = script.new_qregs(n)
    if kind == 'circuit':
        hipruntime.set_fusion(case['fusion'])
        measured, register = _measured_qubits(case)
        refs = script.new_references(len(measured))
        ops = _ops(_gates(case['circuit'], n, case['gates'], seed), q)
        ops += [script.measure(ref, q[k]) for ref, k in zip(refs, measured)]
        sim = Simulator(hipruntime, circuit_prep=case['prep'], dtype=REAL[dtype])
        sim.qubits.set_ordering(q)
        return {'kind': kind, 'sim': sim, 'ops': ops, 'refs': refs, 'seed': seed % (1 << 32),
                'register': [q[k] for k in register] if case['output'] == 'register' else None}
    hipruntime.set_fusion('off')
    sim = Simulator(hipruntime, circuit_prep='one_static', dtype=REAL[dtype])
    sim.qubits.set_ordering(q)
    sim.run(_ops(_pool_gates(n, seed), q))
    kept = random.Random(seed).sample(range(n), case['kept'])
    return {'kind': kind, 'sim': sim, 'qregs': q, 'shots': case['shots'], 'kept': [q[k] for k in kept],
            'uniforms': np.random.RandomState(seed % (1 << 32)).random_sample(case['shots'])}


def _pool_gates(n, seed):
    return _gates('brickwork', n, n, seed)


def _distribution(prob, empty_lanes, ordering):
    return prob


def run(state):
    kind = state['kind']
    if kind == 'gradient':
        params = state['params']
        params.grad = None
        value = Expectation.apply(params, state['circuit'], state['observable'])
        value.backward()
        return {'value': value.detach(), 'grad': params.grad}
    if kind == 'batch':
        for i, p in enumerate(state['params']):
            state['batch'].set_params(i, p)
        values, grads = state['batch'].run()
        return {'values': torch.as_tensor(values, dtype=state['dtype']),
                'grads': torch.as_tensor(np.concatenate(grads), dtype=state['dtype'])}
    sim = state['sim']
    if kind == 'circuit':
        sim.reset()
        np.random.seed(state['seed'])
        sim.run(state['ops'])
        out = {}
        if state['refs']:
            out['outcomes'] = int(sim.obs(state['refs']).int)
        if state['register'] is None:
            out['states'] = sim.qubits.states[:]
        else:
            out['distribution'] = sim.qubits.create_sampling_pool(state['register'], _distribution)
        return out
    pool = sim.qubits.create_sampling_pool(state['qregs'])
    samples = pool.sample(state['shots'], state['uniforms']).intarray
    return {'samples': samples, 'distribution': sim.qubits.create_sampling_pool(state['kept'], _distribution)}


# ---- what a pass cannot do without --------------------------------------------------------

def _flops(gates, n):
    """Flops of a gate list: 14 an amplitude for a general 2x2, 6 for a real or a diagonal
    one, none for X and for diagonal signs; each control halves the amplitudes."""
    per = {'U3': 14, 'H': 6, 'Rz': 6, 'RY': 6, 'RX': 6, 'RZ': 6, 'U1': 3, 'X': 0, 'Z': 0}
    return sum(per[g[0]] * 2. ** (n - len(g[1])) for g in gates)


def work(case):
    kind, amp = case['kind'], 8 if case['dtype'] == 'complex64' else 16

    def gradient(ansatz, n, layers):
        # forward on one state, backward on two, 4 flops an amplitude per gradient term; both
        # states written once and read once
        gates, _ = _ansatz(ansatz, n, layers)
        terms = sum(1 for g in gates if g[3] is not None)
        return 4. * amp * 2. ** n, 3. * _flops(gates, n) + 4. * terms * 2. ** n

    if kind == 'gradient':
        nbytes, flops = gradient(case['ansatz'], case['qubits'], case['layers'])
        return {'bytes': nbytes, 'flops': flops}
    if kind == 'batch':
        parts = [gradient('hea', n, case['layers']) for n in _batch_sizes(case)]
        return {'bytes': sum(p[0] for p in parts), 'flops': sum(p[1] for p in parts)}
    n = case['qubits']
    if kind == 'circuit':
        gates = _gates(case['circuit'], n, case['gates'], 1)
        if case['fusion'] == 'off':   # gate by gate: the touched amplitudes read and written by each gate
            nbytes = sum(2. * amp * 2. ** (n - len(g[1]) - (g[0] == 'U1')) for g in gates)
        else:                         # the state written once and read once
            nbytes = 2. * amp * 2. ** n
        # half of the state for each probability, the output
        nbytes += case['measured'] * amp * 2. ** (n - 1) + amp * 2. ** n
        return {'bytes': nbytes, 'flops': _flops(gates, n)}
    # state read for the pool and for the marginal, probabilities written, draws in and out
    return {'bytes': 2. * amp * 2. ** n + 8. * 2. ** n + 16. * case['shots'], 'flops': 6. * 2. ** n}


# ---- results in 64 bits, in plain torch ---------------------------------------------------

def _matrix(name, angles):
    e = lambda x: complex(math.cos(x), math.sin(x))  # noqa: E731
    if name == 'U3':
        t, p, l = angles[0] / 2, angles[1] / 2, angles[2] / 2
        return [[e(-l - p) * math.cos(t), -e(l - p) * math.sin(t)], [e(-l + p) * math.sin(t), e(l + p) * math.cos(t)]]
    if name == 'H':
        r = math.sqrt(0.5)
        return [[r, r], [r, -r]]
    if name == 'U1':
        return [[1, 0], [0, e(angles[0])]]
    if name == 'X':
        return [[0, 1], [1, 0]]
    if name == 'Z':
        return [[1, 0], [0, -1]]
    t = angles[0] / 2
    if name in ('Rz', 'RZ'):
        return [[e(-t), 0], [0, e(t)]]
    if name == 'RY':
        return [[math.cos(t), -math.sin(t)], [math.sin(t), math.cos(t)]]
    return [[math.cos(t), -1j * math.sin(t)], [-1j * math.sin(t), math.cos(t)]]


def _halves(s, n, controls, target):
    """The amplitudes of s [items, 2^n] with every control 1 and the target 0, and 1."""
    v = s.view([s.shape[0]] + [2] * n)      # dimension n - q is qubit q
    at = [slice(None)] * (n + 1)
    for c in controls:
        at[n - c] = 1
    zero, one = list(at), list(at)
    zero[n - target], one[n - target] = 0, 1
    return v[tuple(zero)], v[tuple(one)]


def _apply(s, n, controls, target, m):
    """In place; an entry of m is a number, or one number per item."""
    a, b = _halves(s, n, controls, target)

    def entry(x):
        return x.reshape([-1] + [1] * (a.dim() - 1)) if isinstance(x, torch.Tensor) else x

    diagonal = all(not isinstance(x, torch.Tensor) and x == 0 for x in (m[0][1], m[1][0]))
    if diagonal:
        if isinstance(m[0][0], torch.Tensor) or m[0][0] != 1:
            a.mul_(entry(m[0][0]))
        b.mul_(entry(m[1][1]))
        return
    c = entry(m[0][0]) * a
    c += entry(m[0][1]) * b
    b.mul_(entry(m[1][1]))
    b += entry(m[1][0]) * a
    a.copy_(c)


def _zero_state(items, n):
    s = torch.zeros(items, 1 << n, dtype=torch.complex128, device='cuda')
    s[:, 0] = 1
    return s


def _run_exact(gates, n):
    s = _zero_state(1, n)
    for name, controls, target, angles in gates:
        _apply(s, n, controls, target, _matrix(name, angles))
    return s


def _marginal(s, n, lanes):
    """Joint distribution over `lanes` (bit i of the index is lanes[i]) of the state s [1, 2^n]."""
    p = s[0].real.square().add_(s[0].imag.square())
    left = list(range(n))
    q = n - 1
    while q >= 0:                # sum the runs of qubits that are not kept, from the top down
        run = 0
        while q >= 0 and q not in lanes:
            run, q = run + 1, q - 1
        if run:
            p = p.view(-1, 1 << run, 1 << (q + 1)).sum(1).reshape(-1)
            del left[q + 1:q + 1 + run]
        q -= 1
    index = torch.arange(1 << len(lanes), device='cuda')
    source = torch.zeros_like(index)
    for i, lane in enumerate(lanes):
        source |= ((index >> i) & 1) << left.index(lane)
    return p[source].cpu().numpy()


def _rotation_matrix(name, theta):
    """Entries per item for theta [items], and of its inverse."""
    c, s = torch.cos(theta / 2), torch.sin(theta / 2)
    c, s = c.to(torch.complex128), s.to(torch.complex128)
    if name == 'RY':
        return [[c, -s], [s, c]], [[c, s], [-s, c]]
    if name == 'RX':
        return [[c, -1j * s], [-1j * s, c]], [[c, 1j * s], [1j * s, c]]
    return [[c - 1j * s, 0], [0, c + 1j * s]], [[c + 1j * s, 0], [0, c - 1j * s]]


def _gradients(ansatz, n, layers, params, a, b):
    """Values [items] and gradients [items, parameters]; a, b: coefficients per item."""
    items = params.shape[0]
    gates, n_params = _ansatz(ansatz, n, layers)
    fixed = {name: _matrix(name, []) for name in ('H', 'X', 'Z')}
    matrices = {}

    def matrix(name, k, back):
        if k is None:
            return fixed[name]
        if (name, k) not in matrices:
            matrices[name, k] = _rotation_matrix(name, params[:, k])
        return matrices[name, k][back]

    psi = _zero_state(items, n)
    for name, controls, target, k in gates:
        _apply(psi, n, controls, target, matrix(name, k, 0))
    index = torch.arange(1 << n, device='cuda')
    diag = torch.zeros(items, 1 << n, dtype=torch.float64, device='cuda')
    for i in range(n - 1):
        sign = 1 - 2 * (((index >> i) ^ (index >> (i + 1))) & 1)
        diag += a[:, i:i + 1] * sign
    lam = diag * psi
    del diag
    for i in range(n):
        p0, p1 = _halves(psi, n, [], i)
        l0, l1 = _halves(lam, n, [], i)
        w = b[:, i].reshape([-1] + [1] * (p0.dim() - 1))
        l0 += w * p1
        l1 += w * p0
    inner = lambda x, y: (x.conj() * y).reshape(items, -1).sum(1)  # noqa: E731
    values = inner(psi, lam).real
    grads = torch.zeros(items, n_params, dtype=torch.float64, device='cuda')
    for name, controls, target, k in reversed(gates):
        if k is not None:
            p0, p1 = _halves(psi, n, controls, target)
            l0, l1 = _halves(lam, n, controls, target)
            if name == 'RX':
                t = inner(l0, p1) + inner(l1, p0)
            elif name == 'RY':
                t = -1j * inner(l0, p1) + 1j * inner(l1, p0)
            else:
                t = inner(l0, p0) - inner(l1, p1)
            grads[:, k] += t.imag
        m = matrix(name, k, 1)
        _apply(psi, n, controls, target, m)
        _apply(lam, n, controls, target, m)
    return values, grads


def exact(case, seed):
    kind = case['kind']
    cuda = lambda x: torch.as_tensor(np.asarray(x, np.float64), device='cuda')  # noqa: E731
    if kind == 'gradient':
        n, layers = case['qubits'], case['layers']
        p, a, b = _step(n, _ansatz(case['ansatz'], n, layers)[1], seed)
        p = p.astype(REAL[case['dtype']])
        values, grads = _gradients(case['ansatz'], n, layers, cuda(p)[None], cuda(a)[None], cuda(b)[None])
        return {'value': values[0], 'grad': grads[0]}
    if kind == 'batch':
        sizes = _batch_sizes(case)
        values, grads = [None] * len(sizes), [None] * len(sizes)
        for n in sorted(set(sizes)):
            at = [i for i, size in enumerate(sizes) if size == n]
            part = max(1, (1 << 26) >> n)    # items at a time
            for first in range(0, len(at), part):
                some = at[first:first + part]
                steps = [_step(n, 2 * n * case['layers'], 4099 * seed + i) for i in some]
                p = np.stack([x[0].astype(REAL[case['dtype']]) for x in steps])
                v, g = _gradients('hea', n, case['layers'], cuda(p), cuda([x[1] for x in steps]),
                                  cuda([x[2] for x in steps]))
                for i, x, y in zip(some, v, g):
                    values[i], grads[i] = x, y
        return {'values': torch.stack(values), 'grads': torch.cat(grads)}
    n = case['qubits']
    if kind == 'circuit':
        if case['measured']:
            return None          # the outcomes decide what is left; they are compared as whole numbers
        s = _run_exact(_gates(case['circuit'], n, case['gates'], seed), n)
        if case['output'] == 'states':
            return {'states': s[0].cpu().numpy()}
        return {'distribution': _marginal(s, n, _measured_qubits(case)[1])}
    s = _run_exact(_pool_gates(n, seed), n)
    kept = random.Random(seed).sample(range(n), case['kept'])
    return {'samples': None, 'distribution': _marginal(s, n, kept)}
