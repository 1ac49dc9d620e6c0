"""The engine's everyday work as measurable cases.

Every case goes through the entry points that a program calls (`apply`,
`Circuit.run_on`, `Circuit.run_batch`, `Circuit.run_dm`, `expect`,
`correlation`, `sample`, `Server`).  Circuits are the brickwork of the
benchmark configurations (three rotations per qubit, a line of entangling
gates, optionally depolarizing noise, amplitude damping and mid-circuit
measurements), plus circuits with distant and controlled gates.  States stay
on the device, and a state that a case returns is a torch view of its buffer.

`exact` is a separate dense simulator in complex128 torch operations.  It
follows the trajectory rules (one uniform per channel, `u <= cumulative sum`;
one per Z measurement, `u < p0`) on the counter-based uniform stream.
"""
import cmath
import math
import random

import numpy as np
import torch

import __graft_entry__ as _entry

bt = _entry.load_package()

P1, P2, GAMMA = 1e-3, 1e-2, 5e-3  # depolarizing on 1 and 2 qubits, amplitude damping
GIB = 1 << 30


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # the reference's own call pattern on a small register: op by op, noise and
        # measurements decided between calls.  Latency of each call.
        dict(name="ops_n12", kind="ops", state="sv", N=12, prec="c128", layers=1, noisy=True, mz=0.1),
        # gates one at a time on a large register (the per-gate kernels at HBM size)
        dict(name="gates_n27", kind="ops", state="sv", N=27, prec="c64", layers=1, noisy=False, mz=0.0),
        # a small noiseless circuit to its final probabilities
        dict(name="circuit_n12", kind="circuit", N=12, prec="c128", layers=20, shape="brick", probs=True),
        # a large noiseless circuit
        dict(name="circuit_n30", kind="circuit", N=30, prec="c64", layers=2, shape="brick", probs=False),
        # one noisy trajectory with mid-circuit measurements (to_state)
        dict(name="traj_n22", kind="traj", N=22, prec="c64", layers=12, mz=0.1),
        # many noisy trajectories at once (run): the headline workload, fewer shots
        dict(name="batch_n22", kind="batch", N=22, prec="c64", layers=32, ntraj=256, mz=0.1, states=False),
        # many small trajectories in double precision, with their final states
        dict(name="batch_n13", kind="batch", N=13, prec="c128", layers=4, ntraj=48, mz=0.1, states=True),
        # exact noisy evolution of a small and a large density matrix (to_rho)
        dict(name="rho_n8", kind="rho", N=8, prec="c64", layers=16),
        dict(name="rho_n12", kind="rho", N=12, prec="c64", layers=4),
        # magnetisations and neighbour correlations of a state
        dict(name="expect_n25", kind="expect", N=25, prec="c64"),
        # shots from a state
        dict(name="sample_n24", kind="sample", N=24, prec="c64", shots=8192),
        # a burst of mixed requests through the server
        dict(name="serve_16", kind="serve", requests=16, top=18, prec="c64"),
    ]


def draw(rng):
    """One more case of the same ranges; sizes are spread over their logarithm."""
    kind = rng.choice(("ops", "ops", "circuit", "circuit", "traj", "batch", "rho", "rho", "expect", "sample", "serve"))
    prec = rng.choice(("c64", "c64", "c128"))
    wide = 1 if prec == "c128" else 0  # one qubit fewer at twice the bytes per amplitude
    if kind == "ops":
        if rng.random() < 0.25:
            return dict(kind="ops", state="dm", N=rng.randint(5, 10), prec=prec, layers=1, noisy=True, mz=0.0)
        noisy = rng.random() < 0.6
        n = rng.randint(9, 22) if noisy else rng.randint(10, 27 - wide)
        return dict(kind="ops", state="sv", N=n, prec=prec, layers=rng.randint(1, 2), noisy=noisy,
                    mz=rng.choice((0.0, 0.1, 0.2)) if noisy else 0.0)
    if kind == "circuit":
        n = rng.randint(9, 29 - wide)
        most = 24 if n <= 20 else 8 if n <= 26 else 2
        return dict(kind="circuit", N=n, prec=prec, layers=rng.randint(2, most) if most > 2 else 2,
                    shape=rng.choice(("brick", "mixed")), probs=prec == "c128" and n <= 16)
    if kind == "traj":
        return dict(kind="traj", N=rng.randint(10, 23 - wide), prec=prec, layers=rng.randint(3, 12),
                    mz=rng.choice((0.0, 0.05, 0.1, 0.2)))
    if kind == "batch":
        if rng.random() < 0.5:
            return dict(kind="batch", N=rng.randint(9, 14), prec="c128", layers=rng.randint(2, 5),
                        ntraj=int(round(2 ** rng.uniform(3, 6))), mz=rng.choice((0.0, 0.1)), states=True)
        return dict(kind="batch", N=rng.randint(14, 22), prec="c64", layers=rng.randint(4, 24),
                    ntraj=int(round(2 ** rng.uniform(3, 8))), mz=rng.choice((0.1, 0.2)), states=False)
    if kind == "rho":
        n = rng.randint(5, 12 - wide)
        return dict(kind="rho", N=n, prec=prec, layers=rng.randint(2, 16 if n <= 9 else 5))
    if kind == "expect":
        return dict(kind="expect", N=rng.randint(10, 27 - wide), prec=prec)
    if kind == "sample":
        return dict(kind="sample", N=rng.randint(10, 26 - wide), prec=prec, shots=int(round(2 ** rng.uniform(6, 14))))
    return dict(kind="serve", requests=rng.randint(4, 24), top=rng.randint(12, 18), prec=prec)


# ---------------------------------------------------------------------------
# circuits
# ---------------------------------------------------------------------------
def _spec(rng, N, layers, mz=0.0, damp=False, shape="brick"):
    """Plain description of a circuit: ("r", axis, angle, q), ("cx", a, b),
    ("cr", angle, q, control), ("cz", a, b), ("damp", q), ("mz", q).  The angles
    come from `rng`; which qubits meet and are measured is part of the case."""
    spec, plan = [], random.Random(1000 * N + layers)
    for layer in range(layers):
        for q in range(1, N + 1):
            for axis in "XYZ":
                spec.append(("r", axis, rng.uniform(0, 2 * math.pi), q))
        if shape == "brick":
            for i in range(1 + layer % 2, N, 2):
                spec.append(("cx", i, i + 1))
        else:  # distant pairs and controlled rotations
            qs = list(range(1, N + 1))
            plan.shuffle(qs)
            for i in range(0, N - 1, 2):
                a, b = qs[i], qs[i + 1]
                pick = plan.randrange(3)
                spec.append(("cx", a, b) if pick == 0 else ("cz", a, b) if pick == 1 else
                            ("cr", rng.uniform(0, 2 * math.pi), a, b))
        if damp:
            for q in range(1, N + 1):
                spec.append(("damp", q))
        for q in range(1, N + 1):
            if mz and plan.random() < mz:
                spec.append(("mz", q))
    return spec


def _ops(spec):
    out = []
    for s in spec:
        if s[0] == "r":
            out.append(bt.Op("R%s(%r)" % (s[1], s[2]), s[3]))
        elif s[0] == "cx":
            out.append(bt.Op("CNOT", s[1], s[2]))
        elif s[0] == "cz":
            out.append(bt.Op("CZ", s[1], s[2]))
        elif s[0] == "cr":
            out.append(bt.Op("RY(%r)" % s[1], s[2], control=s[3]))
        elif s[0] == "damp":
            out.append(bt.OpQC("amplitude_damping", GAMMA, s[1]))
        else:
            out.append(bt.Op("MZ", s[1]))
    return out


def _noise():
    return bt.NoiseModel("depolarizing", P1, "depolarizing", P2)


def _case_spec(case, rng):
    k = case["kind"]
    if k == "ops":
        return _spec(rng, case["N"], case["layers"], case["mz"], case["noisy"])
    if k == "circuit":
        return _spec(rng, case["N"], case["layers"], shape=case["shape"])
    if k == "rho":
        return _spec(rng, case["N"], case["layers"], damp=True)
    return _spec(rng, case["N"], case["layers"], case["mz"], True)


def _requests(case, rng):
    """(kind, N, spec, trajectory) of a burst: three state vectors to one density matrix."""
    reqs, plan = [], random.Random(case["requests"])
    for i in range(case["requests"]):
        dm = i % 4 == 3
        n = plan.randint(6, 8) if dm else plan.randint(10, case["top"])
        reqs.append(("dm" if dm else "sv", n, _spec(rng, n, plan.randint(4, 10), 0.0 if dm else 0.1, True), i))
    return reqs


# ---------------------------------------------------------------------------
# states as torch tensors
# ---------------------------------------------------------------------------
class _Buffer:
    """A device state's memory for torch (zero copy)."""

    def __init__(self, state):
        import ctypes
        p, q = ctypes.c_void_p(), ctypes.c_void_p()
        L = bt.core.L
        L.check(L.lib().bt_state_device_ptr(state.handle, ctypes.byref(p), ctypes.byref(q)))
        self.state = state
        self.__cuda_array_interface__ = dict(shape=(state.length,), typestr="<c8" if state.precision == "c64" else "<c16",
                                             data=(p.value, False), version=2)


def _view(state):
    return torch.as_tensor(_Buffer(state), device="cuda")


def _random_values(n, seed, dtype, device):
    g = torch.Generator(device=device)
    g.manual_seed(seed)
    x = torch.view_as_complex(torch.randn(n, 2, generator=g, dtype=torch.float32, device=device))
    return (x / torch.linalg.vector_norm(x)).to(dtype)


def _random_state(N, prec, seed):
    state = bt.zero_state(N, prec).sync()
    v = _view(state)
    v.copy_(_random_values(v.numel(), seed, v.dtype, "cuda"))
    torch.cuda.synchronize()
    return state, v


# ---------------------------------------------------------------------------
# prepare and run
# ---------------------------------------------------------------------------
def prepare(case, seed):
    rng = random.Random(seed)
    k = case["kind"]
    s = dict(case, seed=rng.randrange(1 << 40))
    if k == "serve":
        s["server"] = bt.Server(hbm_budget_bytes=8 * GIB)
        s["work"] = []
        for kind, n, spec, traj in _requests(case, rng):
            s["work"].append((bt.Circuit(_ops(spec), n, _noise()), kind, traj))
        return s
    if k in ("expect", "sample"):
        s["state"], _ = _random_state(case["N"], case["prec"], s["seed"])
        return s
    spec = _case_spec(case, rng)
    if k == "ops":
        s["ops"] = _ops(spec)
        s["noise"] = _noise() if case["noisy"] else False
        if case["state"] == "dm":
            s["state"] = bt.zero_rho(case["N"], case["prec"])
            s["view"] = _view(s["state"])
        else:
            s["state"], s["view"] = _random_state(case["N"], case["prec"], s["seed"])
        return s
    noisy = k != "circuit"
    s["circuit"] = bt.Circuit(_ops(spec), case["N"], _noise() if noisy else False)
    if k in ("circuit", "traj"):
        s["state"] = bt.zero_state(case["N"], case["prec"])
        s["view"] = _view(s["state"])
    elif k == "rho":
        s["state"] = bt.zero_rho(case["N"], case["prec"])
        s["view"] = _view(s["state"])
    return s


def _bits(outcomes):
    """Outcome lists of equal length as one array."""
    return np.array(outcomes, dtype=np.int64).reshape(len(outcomes), -1)


def run(s):
    k = s["kind"]
    if k == "ops":
        rng = bt.UniformStream(s["seed"], 0)
        if s["mz"]:
            _, outs = bt.apply(s["state"], s["ops"], noise=s["noise"], track_measurements=True, rng=rng)
            return s["view"], np.array(outs, dtype=np.int64)
        bt.apply(s["state"], s["ops"], noise=s["noise"], rng=rng)
        return s["view"]
    if k == "circuit":
        s["circuit"].run_on(s["state"].set_basis(0))
        return (s["view"], s["state"].probabilities()) if s["probs"] else s["view"]
    if k == "traj":
        outs, _ = s["circuit"].run_on(s["state"].set_basis(0), seed=s["seed"], traj=3)
        return s["view"], np.array(outs, dtype=np.int64)
    if k == "batch":
        outs, states, _ = s["circuit"].run_batch(s["ntraj"], seed=s["seed"], prec=s["prec"], keep_states=s["states"])
        return (states, _bits(outs)) if s["states"] else _bits(outs)
    if k == "rho":
        s["circuit"].run_dm(s["state"].set_basis(0))
        trace, purity = s["state"].trace_purity()
        return s["view"], trace, purity
    if k == "expect":
        st, n = s["state"], s["N"]
        zz = [bt.correlation(st, "Z,Z", [q, q + 1]) for q in range(1, n)]
        xy = [bt.correlation(st, "X,Y", [q, q + 2]) for q in range(1, n - 1, 4)]
        return bt.expect(st, "Z"), bt.expect(st, "X"), np.array(zz), np.array(xy)
    if k == "sample":
        return bt.sample(s["state"], s["shots"], rng=bt.UniformStream(s["seed"], 0))
    srv = s["server"]
    ids = [srv.submit(c, kind, s["prec"], seed=s["seed"], traj=t) for c, kind, t in s["work"]]
    left = set(ids)
    while left:
        for r in srv.poll(wait=True):
            if r["status"]:
                raise RuntimeError("request %d failed with %d" % (r["id"], r["status"]))
            left.discard(r["id"])
    got = [srv.fetch(i) for i in ids]
    # a complex64 state's probabilities carry single precision
    probs = [p.astype(np.float32) if s["prec"] == "c64" else p for _, p in got]
    return probs, np.array([b for o, _ in got for b in o], dtype=np.int64)


# ---------------------------------------------------------------------------
# work: each input read once, each output written once; the products of the
# entangling blocks (4 x 4 complex per pair, 8 flops per multiply-add)
# ---------------------------------------------------------------------------
def work(case):
    k = case["kind"]
    amp = 8 if case["prec"] == "c64" else 16
    if k == "serve":
        return dict(bytes=float(case["requests"]) * 2 ** (case["top"] - 2) * (amp + 8),
                    flops=float(case["requests"]) * 7 * case["top"] / 2 * 32 * 2 ** (case["top"] - 2))
    N = case["N"]
    if k == "expect":
        count = 2 * N + (N - 1) + len(range(1, N - 1, 4))
        return dict(bytes=float(amp * 2 ** N), flops=float(count * 4 * 2 ** N))
    if k == "sample":
        return dict(bytes=float(amp * 2 ** N + 16 * case["shots"]), flops=float(4 * 2 ** N))
    dm = k == "rho" or case.get("state") == "dm"
    D = 4 ** N if dm else 2 ** N
    flops = case["layers"] * (N / 2) * 32 * D * (4 if dm else 1)
    if k == "ops":  # every call reads and writes the state
        calls = case["layers"] * (3 * N + N // 2)
        return dict(bytes=float(calls * 2 * amp * D), flops=float(flops))
    if k == "batch":
        per = 2 * case["layers"] if case["mz"] else 1  # a decision needs the whole state
        return dict(bytes=float(case["ntraj"]) * D * (amp * per + (16 if case["states"] else 0)),
                    flops=float(case["ntraj"] * flops))
    if k == "traj" and case["mz"]:
        return dict(bytes=float(2 * case["layers"] * amp * D), flops=float(flops))
    return dict(bytes=float(amp * D + (8 * D if case.get("probs") else 0)), flops=float(flops))


# ---------------------------------------------------------------------------
# exact: dense complex128 simulation, without the engine
# ---------------------------------------------------------------------------
_M64 = (1 << 64) - 1


def _mix(x):
    x = (x + 0x9E3779B97F4A7C15) & _M64
    x = ((x ^ (x >> 30)) * 0xBF58476D1CE4E5B9) & _M64
    x = ((x ^ (x >> 27)) * 0x94D049BB133111EB) & _M64
    return x ^ (x >> 31)


class _Draws:
    """The counter-based uniform stream u(seed, trajectory, draw)."""

    def __init__(self, seed, traj):
        self.seed, self.traj, self.i = seed, traj, 0

    def __call__(self):
        u = (_mix(self.seed ^ _mix(self.traj ^ _mix(self.i))) >> 11) * 2.0 ** -53
        self.i += 1
        return u


_PAULI = {"I": ((1, 0), (0, 1)), "X": ((0, 1), (1, 0)), "Y": ((0, -1j), (1j, 0)), "Z": ((1, 0), (0, -1))}


def _rot(axis, t):
    c, s = math.cos(t / 2), math.sin(t / 2)
    if axis == "X":
        return ((c, -1j * s), (-1j * s, c))
    if axis == "Y":
        return ((c, -s), (s, c))
    return ((cmath.exp(-0.5j * t), 0), (0, cmath.exp(0.5j * t)))


class _Sim:
    """A vector of `nbits` index bits; qubit q of N is bit N - q."""

    def __init__(self, nbits, v=None):
        self.n = nbits
        self.dev = "cuda" if nbits >= 15 and torch.cuda.is_available() else "cpu"
        if v is None:
            v = torch.zeros(1 << nbits, dtype=torch.complex128, device=self.dev)
            v[0] = 1
        self.v = v

    def _part(self, where):
        """The entries whose bits have the given values."""
        x, lo = self.v, self.n
        shape, pick = [], []
        for b in sorted(where, reverse=True):
            shape += [1 << (lo - b - 1), 2]
            pick += [slice(None), where[b]]
            lo = b
        return x.view(shape + [1 << lo])[tuple(pick)]

    def apply(self, m, bit, ctrl=None):
        rest = {} if ctrl is None else {ctrl: 1}
        a, b = self._part({bit: 0, **rest}), self._part({bit: 1, **rest})
        (p, q), (r, s) = m
        if q == 0 and r == 0:
            if p != 1:
                a.mul_(p)
            if s != 1:
                b.mul_(s)
            return
        old = a.clone()
        a.mul_(p)
        if q != 0:
            a.add_(b, alpha=q)
        b.mul_(s)
        if r != 0:
            b.add_(old, alpha=r)

    def weight(self, bit, value):
        x = torch.view_as_real(self._part({bit: value}))
        return float((x * x).sum())


def _gate_of(s, N):
    """(matrix, bit, control bit) of a unitary entry."""
    if s[0] == "r":
        return _rot(s[1], s[2]), N - s[3], None
    if s[0] == "cx":
        return _PAULI["X"], N - s[2], N - s[1]
    if s[0] == "cz":
        return _PAULI["Z"], N - s[2], N - s[1]
    return _rot("Y", s[1]), N - s[2], N - s[3]


def _noise_qubits(s):
    return {"r": lambda: (s[3],), "cx": lambda: (s[1], s[2]), "cz": lambda: (s[1], s[2]),
            "cr": lambda: (s[3], s[2])}[s[0]]()


def _branch(weights, u):
    c = 0.0
    for i, w in enumerate(weights):
        c += w
        if u <= c:
            return i
    return len(weights) - 1


def _trajectory(sim, spec, N, noisy, u):
    """Runs `spec` on a normalised state vector; the recorded outcomes."""
    outs = []
    for s in spec:
        if s[0] == "mz":
            bit = N - s[1]
            p0 = sim.weight(bit, 0)
            got = 0 if u() < p0 else 1
            outs.append(got)
            keep = 1 / math.sqrt(p0 if got == 0 else sim.weight(bit, 1))
            sim.apply(((keep, 0), (0, 0)) if got == 0 else ((0, 0), (0, keep)), bit)
        elif s[0] == "damp":
            bit, x = N - s[1], u()
            one = sim.weight(bit, 1)
            stay = (1 - one) + (1 - GAMMA) * one
            if x <= stay:
                k = 1 / math.sqrt(stay)
                sim.apply(((k, 0), (0, k * math.sqrt(1 - GAMMA))), bit)
            else:
                sim.apply(((0, 1 / math.sqrt(one)), (0, 0)), bit)
        else:
            m, bit, ctrl = _gate_of(s, N)
            sim.apply(m, bit, ctrl)
            if noisy:
                qs = _noise_qubits(s)
                p = P1 if len(qs) == 1 else P2
                one = [1 - p, p / 3, p / 3, p / 3]
                names = [(i,) for i in "IXYZ"] if len(qs) == 1 else [(i, j) for i in "IXYZ" for j in "IXYZ"]
                w = one if len(qs) == 1 else [x * y for x in one for y in one]
                for q, name in zip(qs, names[_branch(w, u())]):
                    if name != "I":
                        sim.apply(_PAULI[name], N - q)
    return outs


def _density(spec, N):
    """vec(rho) after `spec` with the noise on: row bits low, column bits high."""
    sim = _Sim(2 * N)

    def both(m, bit, ctrl):
        sim.apply(m, bit, ctrl)
        conj = tuple(tuple(complex(x).conjugate() for x in row) for row in m)
        sim.apply(conj, bit + N, None if ctrl is None else ctrl + N)

    def depolarize(bit, p):
        # (1 - p) rho + p / 3 (X rho X + Y rho Y + Z rho Z)
        a, b = sim._part({bit: 0, bit + N: 0}), sim._part({bit: 1, bit + N: 1})
        m = (a + b) * (p * 2 / 3)
        a.mul_(1 - 4 * p / 3).add_(m)
        b.mul_(1 - 4 * p / 3).add_(m)
        sim._part({bit: 0, bit + N: 1}).mul_(1 - 4 * p / 3)
        sim._part({bit: 1, bit + N: 0}).mul_(1 - 4 * p / 3)

    for s in spec:
        if s[0] == "damp":
            bit = N - s[1]
            one = sim._part({bit: 1, bit + N: 1})
            sim._part({bit: 0, bit + N: 0}).add_(one, alpha=GAMMA)
            one.mul_(1 - GAMMA)
            sim._part({bit: 0, bit + N: 1}).mul_(math.sqrt(1 - GAMMA))
            sim._part({bit: 1, bit + N: 0}).mul_(math.sqrt(1 - GAMMA))
        else:
            both(*_gate_of(s, N))
            qs = _noise_qubits(s)
            for q in qs:
                depolarize(N - q, P1 if len(qs) == 1 else P2)
    return sim.v


def _expectation(v, n, xmask, zmask):
    """sum conj(v_i) (-1)^parity(i & zmask) v_{i ^ xmask}, in 64 bits."""
    w = v.view([2] * n)
    flip = [n - 1 - b for b in range(n) if xmask >> b & 1]
    y = (torch.flip(w, flip) if flip else w).reshape(-1)
    i = torch.arange(v.numel(), device=v.device) & zmask
    for sh in (32, 16, 8, 4, 2, 1):
        i = i ^ (i >> sh)
    y = torch.where((i & 1).bool(), -y, y)
    return complex((v.conj() * y).sum())


def exact(case, seed):
    rng = random.Random(seed)
    k = case["kind"]
    stream = rng.randrange(1 << 40)
    if k == "serve":
        probs = []
        for kind, n, spec, traj in _requests(case, rng):
            if kind == "dm":
                v = _density(spec, n)
                probs.append(v.view(1 << n, 1 << n).diagonal().real.contiguous().cpu().numpy())
            else:
                sim = _Sim(n)
                _trajectory(sim, spec, n, True, _Draws(stream, traj))
                probs.append(torch.view_as_real(sim.v).square().sum(1).cpu().numpy())
        return probs, None
    if k == "sample":
        return None
    N = case["N"]
    if k == "expect":
        if N > 26:  # 2 GiB per vector, a few hundred passes: too long
            return None
        v = _random_values(1 << N, stream, torch.complex64, "cuda").to(torch.complex128)
        z = [_expectation(v, N, 0, 1 << (N - q)).real for q in range(1, N + 1)]
        x = [_expectation(v, N, 1 << (N - q), 0).real for q in range(1, N + 1)]
        zz = [_expectation(v, N, 0, 3 << (N - q - 1)).real for q in range(1, N)]
        xy = [(-1j * _expectation(v, N, 5 << (N - q - 2), 1 << (N - q - 2))).real for q in range(1, N - 1, 4)]
        return np.array(z), np.array(x), np.array(zz), np.array(xy)
    spec = _case_spec(case, rng)
    if k == "rho" or case.get("state") == "dm":
        v = _density(spec, N)
        if k == "ops":
            return v
        return v, float(v.view(1 << N, 1 << N).diagonal().real.sum()), float(torch.view_as_real(v).square().sum())
    if k == "batch":
        if not case["states"]:
            return None
        states = []
        for t in range(case["ntraj"]):
            sim = _Sim(N)
            _trajectory(sim, spec, N, True, _Draws(stream, t))
            states.append(sim.v.cpu().numpy())
        return np.stack(states), None
    sim = _Sim(N)
    if k == "ops":
        v = _random_values(1 << N, stream, torch.complex64, "cuda").to(torch.complex128)
        sim = _Sim(N, v.to(sim.dev))
        if case["noisy"]:
            # the trajectory rules hold for the state as it is, and renormalise it
            sim.v /= torch.linalg.vector_norm(sim.v)
    noisy = k == "traj" or (k == "ops" and case["noisy"])
    outs = _trajectory(sim, spec, N, noisy, _Draws(stream, 3 if k == "traj" else 0))
    if k == "circuit":
        return (sim.v, torch.view_as_real(sim.v).square().sum(1)) if case["probs"] else sim.v
    if k == "traj":
        return sim.v, None
    return (sim.v, None) if case["mz"] else sim.v
