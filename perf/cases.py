"""Workloads that time the framework through its public entry points.

Each case is one call that a user's program makes again and again (an
optimiser's step, a shot-based gradient, an expectation value), over the sizes
that the tests, the benchmark and the serving trace of this repository use:
10 to 28 qubits, 2 to 40 layers, both state precisions, both entanglers,
history and checkpoint mode, single and batched circuits.

``exact`` restates the circuits in plain torch, one gate at a time in
complex128, without the framework's code.

A program that keeps its state in complex64 has single-precision results (the
framework's own bar there is 1e-6), so these cases keep them as float32.  The
value and its gradient travel as one array, as an optimiser takes them.
"""
import math

import numpy as np
import torch

from qradient_amd.batch import QaoaBatch
from qradient_amd.circuit_logic import McClean, Qaoa


def listed():
    return [
        # the smallest calls: a textbook VQE circuit, one optimiser step (launches and latency)
        {'name': 'mcclean_10q', 'kind': 'mcclean', 'mode': 'grad', 'n': 10, 'L': 10, 'dtype': 'complex128',
         'entangler': 'cnot', 'obs': 'z0z1', 'ckpt': 0},
        # the largest circuit that runs whole in one workgroup
        {'name': 'mcclean_13q', 'kind': 'mcclean', 'mode': 'grad', 'n': 13, 'L': 20, 'dtype': 'complex64',
         'entangler': 'cnot', 'obs': 'zmix', 'ckpt': 0},
        # the median request of the serving trace: a state that the caches hold, the CZ entangler
        {'name': 'mcclean_16q', 'kind': 'mcclean', 'mode': 'grad', 'n': 16, 'L': 20, 'dtype': 'complex64',
         'entangler': 'cz', 'obs': 'chain', 'ckpt': 0},
        # forward only: an expectation value with x, y, z and zz terms, odd qubit number
        {'name': 'expec_19q', 'kind': 'mcclean', 'mode': 'expec', 'n': 19, 'L': 12, 'dtype': 'complex128',
         'entangler': 'cnot', 'obs': 'xyz', 'ckpt': 0},
        # the plain complex128 method at an odd size whose state no cache holds
        {'name': 'mcclean_23q_c128', 'kind': 'mcclean', 'mode': 'grad', 'n': 23, 'L': 9, 'dtype': 'complex128',
         'entangler': 'cnot', 'obs': 'chain', 'ckpt': 0},
        # the headline benchmark
        {'name': 'mcclean_24q', 'kind': 'mcclean', 'mode': 'grad', 'n': 24, 'L': 40, 'dtype': 'complex64',
         'entangler': 'cnot', 'obs': 'chain', 'ckpt': 0},
        # a large state in checkpoint mode (psi uncomputed in the adjoint sweep)
        {'name': 'mcclean_27q_ckpt', 'kind': 'mcclean', 'mode': 'grad', 'n': 27, 'L': 10, 'dtype': 'complex64',
         'entangler': 'cnot', 'obs': 'chain', 'ckpt': 4},
        # one QAOA circuit of a weighted graph (real weights, odd qubit number)
        {'name': 'qaoa_17q', 'kind': 'qaoa', 'n': 17, 'p': 6, 'dtype': 'complex128', 'graph': 'weighted', 'batch': 1},
        # an optimiser over many small MaxCut graphs
        {'name': 'qaoa_batch_12q', 'kind': 'qaoa', 'n': 12, 'p': 4, 'dtype': 'complex64', 'graph': 'maxcut',
         'batch': 64},
        # the batched QAOA benchmark's shape, half its batch
        {'name': 'qaoa_batch_20q', 'kind': 'qaoa', 'n': 20, 'p': 8, 'dtype': 'complex64', 'graph': 'maxcut',
         'batch': 256},
        # a shot-based parameter-shift gradient
        {'name': 'sample_grad_14q', 'kind': 'sample', 'n': 14, 'L': 4, 'dtype': 'complex128', 'shots': 100},
        # a shot-based QAOA gradient measured in the computational basis (device-resident State)
        {'name': 'qaoa_dense_12q', 'kind': 'dense', 'n': 12, 'p': 2, 'dtype': 'complex128', 'shots': 64},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(['mcclean'] * 7 + ['qaoa'] * 3 + ['sample', 'dense'])
    dtype = rng.choice(['complex64', 'complex128'])
    if kind == 'mcclean':
        n = rng.randint(8, 27)
        most = 40 if n <= 22 else 30 if n <= 24 else 10
        L = _log_int(rng, 2, most)
        mode = 'expec' if rng.random() < 0.25 else 'grad'
        ckpt = 0
        if mode == 'grad' and n >= 14 and (n >= 26 or rng.random() < 0.2):
            ckpt = rng.randint(1, 6)
        if mode == 'expec' or (n >= 14 and rng.random() < 0.3):
            dtype = 'complex128'
        if mode == 'grad' and n >= 26:
            dtype = 'complex64'  # no dearer than the largest listed state
        obs = rng.choice(['z0z1', 'zmix', 'chain', 'chain', 'xyz'])
        return {'kind': kind, 'mode': mode, 'n': n, 'L': L, 'dtype': dtype,
                'entangler': rng.choice(['cnot', 'cnot', 'cnot', 'cz']), 'obs': obs, 'ckpt': ckpt}
    if kind == 'qaoa':
        n = rng.randint(8, 20)
        batch = 1 if rng.random() < 0.4 else _log_int(rng, 4, 256)
        amps = batch * 2 ** n
        return {'kind': kind, 'n': n, 'p': rng.randint(1, 8), 'dtype': dtype if amps < 2 ** 27 else 'complex64',
                'graph': rng.choice(['maxcut', 'weighted']) if amps < 2 ** 26 else 'maxcut', 'batch': batch}
    if kind == 'sample':
        return {'kind': kind, 'n': rng.randint(8, 16), 'L': rng.randint(1, 4), 'dtype': 'complex128',
                'shots': _log_int(rng, 10, 300)}
    return {'kind': kind, 'n': rng.randint(8, 12), 'p': rng.randint(1, 2), 'dtype': 'complex128',
            'shots': _log_int(rng, 10, 300)}


# ---------------------------------------------------------------------------
# inputs, from the seed alone
# ---------------------------------------------------------------------------
def _observable(n, kind, rs):
    """The framework's observable dict: weights of x, y, z and zz terms."""
    zz = np.full((n, n), None)
    if kind == 'z0z1':
        zz[0, 1] = 1.0
        return {'zz': zz}
    for i, w in enumerate(rs.standard_normal(n - 1)):
        zz[i, i + 1] = float(w)
    obs = {'zz': zz}
    if kind in ('zmix', 'xyz'):
        obs['z'] = np.array([float(rs.standard_normal()) if q % 2 == 0 else None for q in range(n)], dtype=object)
    if kind == 'xyz':
        obs['x'] = np.array([float(rs.standard_normal()) if q % 3 == 0 else None for q in range(n)], dtype=object)
        obs['y'] = np.array([float(rs.standard_normal()) if q % 4 == 1 else None for q in range(n)], dtype=object)
    return obs


def _graph(n, kind, rs):
    """A MaxCut graph as an observable: a ring with about n / 2 chords (degree
    3 on average), unit weights, or real ones."""
    zz = np.full((n, n), None)
    edges = {tuple(sorted((i, (i + 1) % n))) for i in range(n)}
    while len(edges) < n + n // 2:
        a, b = rs.randint(0, n, 2)
        if a != b:
            edges.add((int(min(a, b)), int(max(a, b))))
    for a, b in sorted(edges):
        zz[a, b] = 1.0 if kind == 'maxcut' else float(rs.uniform(0.2, 2.0))
    return {'zz': zz}


def _inputs(case, seed):
    rs = np.random.RandomState(seed % (2 ** 31))
    n = case['n']
    if case['kind'] in ('mcclean', 'sample'):
        L = case['L']
        axes = rs.randint(0, 3, (L, n))
        angles = 2 * np.pi * rs.rand(L, n)
        obs = _observable(n, case.get('obs', 'chain'), rs)
        return {'axes': axes, 'angles': angles, 'obs': obs, 'draws': int(rs.randint(2 ** 31 - 1))}
    B, p = case.get('batch', 1), case['p']
    return {'obs': [_graph(n, case.get('graph', 'maxcut'), rs) for _ in range(B)],
            'betas': rs.uniform(0.1, 1.2, (B, p)), 'gammas': rs.uniform(0.1, 1.2, (B, p)),
            'draws': int(rs.randint(2 ** 31 - 1))}


def prepare(case, seed):
    x = _inputs(case, seed)
    s = dict(case=case, x=x)
    n = case['n']
    if case['kind'] in ('mcclean', 'sample'):
        kw = {'ckpt_every': case['ckpt']} if case.get('ckpt') else {}
        s['circuit'] = McClean(n, x['obs'], case['L'], axes=x['axes'], angles=x['angles'], dtype=case['dtype'],
                               entangler=case.get('entangler', 'cnot'), **kw)
    elif case['kind'] == 'qaoa' and case['batch'] > 1:
        s['batch'] = QaoaBatch(n, case['p'], case['batch'], dtype=case['dtype'])
        s['graphs'] = s['batch'].pack(x['obs'])  # an optimiser over fixed graphs packs them once
    else:
        s['circuit'] = Qaoa(n, x['obs'][0], case['p'], dtype=case['dtype'])
    return s


def _value_and_gradient(case, E, grad):
    out = np.concatenate((np.ravel(E), np.ravel(grad)))
    return out.astype(np.float32) if case['dtype'] == 'complex64' else out


def run(state):
    case, x = state['case'], state['x']
    kind = case['kind']
    if kind == 'mcclean':
        if case['mode'] == 'expec':
            return state['circuit'].run_expec_val()
        return _value_and_gradient(case, *state['circuit'].grad_run())
    if kind == 'qaoa':
        if 'batch' in state:
            return _value_and_gradient(case, *state['batch'].grad_run(state['graphs'], x['betas'], x['gammas']))
        return _value_and_gradient(case, *state['circuit'].grad_run(x['betas'][0], x['gammas'][0]))
    np.random.seed(x['draws'])  # the estimates are functions of numpy's global stream
    if kind == 'sample':
        return _value_and_gradient(case, *state['circuit'].sample_grad(shot_num=case['shots']))
    return _value_and_gradient(case, *state['circuit'].sample_grad_dense(x['betas'][0], x['gammas'][0],
                                                                         shot_num=case['shots']))


# ---------------------------------------------------------------------------
# what one pass cannot do without
# ---------------------------------------------------------------------------
_GATE = 6     # flops per amplitude of a Pauli rotation (three FMAs)
_REDUCE = 4   # flops per amplitude of Im<lambda|P|psi>


def work(case):
    """Flops of the gates (every qubit once a layer; the adjoint sweep undoes
    them on lambda) and of the gradient reductions.  Bytes: the parameters and
    results, and for circuits past one workgroup (13 qubits) the state written
    once and read once per sweep."""
    n, N = case['n'], 2.0 ** case['n']
    S = N * (8 if case['dtype'] == 'complex64' else 16)
    if case['kind'] == 'mcclean':
        gates = n * case['L']
        io = 24.0 * gates
        if case['mode'] == 'expec':
            return {'bytes': io + (2 * S if n > 13 else 0), 'flops': _GATE * gates * N}
        return {'bytes': io + (4 * S if n > 13 else 0), 'flops': (2 * _GATE + _REDUCE) * gates * N}
    if case['kind'] == 'qaoa':
        gates, B = n * case['p'], case['batch']
        phase = 8 * case['p']  # one complex product a layer
        return {'bytes': B * (32.0 * case['p'] + (4 * S if n > 13 else 0)),
                'flops': B * N * ((2 * _GATE + _REDUCE) * gates + 2 * phase)}
    if case['kind'] == 'sample':
        layers = n * case['L'] * (case['L'] + 1)  # every shifted circuit from its layer on
        shifted = 2 * n * case['L']
        return {'bytes': (shifted * 2 * S if n > 13 else 0) + 8.0 * shifted * (n - 1) * case['shots'],
                'flops': N * (_GATE * n * layers + shifted * (3 + 2 * (n - 1)))}
    circuits = 2 * (n + n // 2 + n)  # a layer's shifted circuits: the edges' and the qubits'
    suffix = circuits * case['p'] * (case['p'] + 1) / 2
    return {'bytes': 8.0 * circuits * case['p'] * case['shots'],
            'flops': N * suffix * (_GATE * n + 8) + N * 3 * circuits * case['p']}


# ---------------------------------------------------------------------------
# the same values in 64 bits, one gate at a time
# ---------------------------------------------------------------------------
def _dev():
    return torch.device('cuda' if torch.cuda.is_available() else 'cpu')


def _rot(v, n, axis, angle, q):
    """v <- exp(-i angle/2 P_q) v in place; qubit 0 is the most significant bit."""
    w = v.view(2 ** q, 2, -1)
    x0, x1 = w[:, 0], w[:, 1]
    c, s = math.cos(0.5 * angle), math.sin(0.5 * angle)
    if axis == 2:
        x0.mul_(complex(c, -s))
        x1.mul_(complex(c, s))
        return
    old = x0.clone()
    f = (complex(0, -s), complex(0, -s)) if axis == 0 else (complex(-s), complex(s))
    x0.mul_(c).add_(x1, alpha=f[0])
    x1.mul_(c).add_(old, alpha=f[1])


def _pauli_im(lam, psi, axis, q):
    """Im<lam|P_q|psi>."""
    a, b = lam.view(2 ** q, 2, -1), psi.view(2 ** q, 2, -1)
    if axis == 2:
        return (a[:, 0].conj() * b[:, 0]).sum().imag - (a[:, 1].conj() * b[:, 1]).sum().imag
    up, down = (a[:, 0].conj() * b[:, 1]).sum(), (a[:, 1].conj() * b[:, 0]).sum()
    return (up + down).imag if axis == 0 else down.real - up.real


def _signs(n, q, dev):
    s = torch.ones(2 ** q, 2, 2 ** (n - 1 - q), dtype=torch.float64, device=dev)
    s[:, 1] = -1
    return s.view(-1)


def _diagonal(n, obs, dev):
    D = torch.zeros(2 ** n, dtype=torch.float64, device=dev)
    for i, w in enumerate(obs.get('z', ())):
        if w is not None:
            D.add_(_signs(n, i, dev), alpha=w)
    for i in range(n):
        for j in range(i + 1, n):
            if obs['zz'][i, j] is not None:
                D.add_(_signs(n, i, dev) * _signs(n, j, dev), alpha=obs['zz'][i, j])
    return D


def _apply_observable(psi, n, obs, dev):
    out = psi * _diagonal(n, obs, dev)
    for axis, key in ((0, 'x'), (1, 'y')):
        for q, w in enumerate(obs.get(key, ())):
            if w is not None:
                a, b = out.view(2 ** q, 2, -1), psi.view(2 ** q, 2, -1)
                f = (complex(w), complex(w)) if axis == 0 else (complex(0, -w), complex(0, w))
                a[:, 0].add_(b[:, 1], alpha=f[0])
                a[:, 1].add_(b[:, 0], alpha=f[1])
    return out


def _entangle(v, n, kind, undo):
    bonds = list(range(1, n - 1, 2)) + list(range(0, n - 1, 2))  # odd bonds act first
    for i in (reversed(bonds) if undo else bonds):
        w = v.view(2 ** i, 2, 2, -1)
        if kind == 'cz':
            w[:, 1, 1].neg_()
        else:
            old = w[:, 1, 0].clone()
            w[:, 1, 0] = w[:, 1, 1]
            w[:, 1, 1] = old


def _start(n, dev):
    v = torch.zeros(2 ** n, dtype=torch.complex128, device=dev)
    v[0] = 1
    for q in range(n):
        _rot(v, n, 1, math.pi / 4, q)
    return v


def _layer(v, n, axes, angles, entangler):
    _entangle(v, n, entangler, False)
    for q in range(n):
        _rot(v, n, axes[q], angles[q], q)


def _exact_mcclean(case, x):
    n, L, dev = case['n'], case['L'], _dev()
    ent = case['entangler']
    psi = _start(n, dev)
    for i in range(L):
        _layer(psi, n, x['axes'][i], x['angles'][i], ent)
    lam = _apply_observable(psi, n, x['obs'], dev)
    E = torch.vdot(psi, lam).real
    if case['mode'] == 'expec':
        return np.float64(E.item())
    g = [None] * (L * n)
    for i in reversed(range(L)):
        for q in range(n):
            g[i * n + q] = _pauli_im(lam, psi, x['axes'][i][q], q)
        for q in range(n):
            _rot(psi, n, x['axes'][i][q], -x['angles'][i][q], q)
            _rot(lam, n, x['axes'][i][q], -x['angles'][i][q], q)
        _entangle(psi, n, ent, True)
        _entangle(lam, n, ent, True)
    return torch.stack([E] + g).cpu().numpy()


def _plus(n, dev):
    return torch.full((2 ** n,), 2.0 ** (-0.5 * n), dtype=torch.complex128, device=dev)


def _phase(v, C, gamma):
    v.mul_(torch.polar(torch.ones_like(C), -gamma * C))


def _mixer(v, n, beta):
    for q in range(n):
        _rot(v, n, 0, beta, q)


def _exact_qaoa_circuit(n, obs, betas, gammas):
    dev = _dev()
    C = _diagonal(n, obs, dev)
    psi = _plus(n, dev)
    for b, g in zip(betas, gammas):
        _phase(psi, C, g)
        _mixer(psi, n, b)
    lam = psi * C
    E = torch.vdot(psi, lam).real
    out = []
    for b, g in zip(betas[::-1], gammas[::-1]):
        db = sum(_pauli_im(lam, psi, 0, q) for q in range(n))
        _mixer(psi, n, -b)
        _mixer(lam, n, -b)
        out += [2 * torch.vdot(lam, psi * C).imag, db]
        _phase(psi, C, -g)
        _phase(lam, C, -g)
    return torch.stack([E] + out[::-1]).cpu().numpy()


def _exact_sample(case, x):
    """Parameter shifts by +-pi/2; per term, shots of the +1 projector's
    probability from numpy's global stream, circuit by circuit."""
    n, L, shots, dev = case['n'], case['L'], case['shots'], _dev()
    terms = [(i, i + 1, x['obs']['zz'][i, i + 1]) for i in range(n - 1)]
    Z = torch.stack([_signs(n, i, dev) * _signs(n, j, dev) for i, j, _ in terms])
    w = np.array([t[2] for t in terms])
    ends = [_start(n, dev)]
    for i in range(L):
        v = ends[-1].clone()
        _layer(v, n, x['axes'][i], x['angles'][i], 'cnot')
        ends.append(v)
    psi = ends.pop()
    E = float(torch.vdot(psi, _apply_observable(psi, n, x['obs'], dev)).real)
    probs = []
    for i in range(L):
        for q in range(n):
            for d in (np.pi / 2, -np.pi / 2):
                ang = x['angles'].copy()
                ang[i, q] += d
                v = ends[i].clone()
                for k in range(i, L):
                    _layer(v, n, x['axes'][k], ang[k], 'cnot')
                m = v.abs().square()
                probs.append(0.5 * (m.sum() + Z @ m))
    probs = np.clip(torch.stack(probs).cpu().numpy(), 0.0, 1.0)
    np.random.seed(x['draws'])
    u = np.random.uniform(size=(2 * n * L, len(terms), shots))
    o = np.where(u <= probs[..., None], w[None, :, None], -w[None, :, None]).mean(axis=2).sum(axis=1)
    return np.concatenate(([E], 0.5 * (o[0::2] - o[1::2])))


def _exact_dense(case, x):
    """QAOA circuits with one component phase or one mixer angle shifted,
    measured in the computational basis at numpy's global uniforms."""
    n, p, shots, dev = case['n'], case['p'], case['shots'], _dev()
    betas, gammas, obs = x['betas'][0], x['gammas'][0], x['obs'][0]
    C = _diagonal(n, obs, dev)
    Ch = C.cpu().numpy()
    parts = []
    for i in range(n):
        for j in range(i + 1, n):
            if obs['zz'][i, j] is not None:
                parts.append(obs['zz'][i, j] * _signs(n, i, dev) * _signs(n, j, dev))
    before, between = [], []  # the state after each layer's phase, and after its mixer
    v = _plus(n, dev)
    for i in range(p):
        _phase(v, C, gammas[i])
        before.append(v.clone())
        _mixer(v, n, betas[i])
        between.append(v.clone())
    E = float(torch.vdot(v, v * C).real)
    np.random.seed(x['draws'])

    def estimate(v, i):
        for k in range(i + 1, p):
            _phase(v, C, gammas[k])
            _mixer(v, n, betas[k])
        cum = np.cumsum(v.abs().square().cpu().numpy())
        u = np.random.uniform(size=shots)
        at = np.searchsorted(cum, u, side='left')
        return Ch[np.where(at < len(cum), at, 0)].mean()

    grad = np.empty((p, 2))
    for i in range(p):
        dg = db = 0.0
        for part in parts:
            o = []
            for a in (np.pi / 4, -np.pi / 4):
                v = before[i].clone()
                _phase(v, part, a)
                _mixer(v, n, betas[i])
                o.append(estimate(v, i))
            dg += o[0] - o[1]
        for q in range(n):
            o = []
            for a in (np.pi / 2, -np.pi / 2):
                v = between[i].clone()
                _rot(v, n, 0, a, q)
                o.append(estimate(v, i))
            db += o[0] - o[1]
        grad[i] = 0.5 * db, dg
    return np.concatenate(([E], grad.ravel()))


def exact(case, seed):
    x = _inputs(case, seed)
    with torch.no_grad():
        if case['kind'] == 'mcclean':
            return _exact_mcclean(case, x)
        if case['kind'] == 'sample':
            return _exact_sample(case, x)
        if case['kind'] == 'dense':
            return _exact_dense(case, x)
        rows = [_exact_qaoa_circuit(case['n'], x['obs'][b], x['betas'][b], x['gammas'][b])
                for b in range(case['batch'])]
        return np.concatenate([r[:1] for r in rows] + [r[1:] for r in rows])
