"""The calls that this framework's performance is measured on.

Each case is one call, or one training step, through the public entry points
(``quantum_amd.layers``, the simulation ops, ``tfq.math``, ``tfq.noise``).
Together the cases cover the ops over circuit widths from 3 to 28 qubits: small
batches where latency counts, batches of thousands of uneven circuits, and
single states that fill the GPU.  A circuit is described by ``_moments`` as
plain tuples, from which ``prepare`` builds the framework's circuits and
``exact`` an independent complex128 simulation.

The circuits of a case are fixed by its ``circuits`` number (a program keeps its
model); the seed gives the symbol values, the upstream gradients and, in the
layer case, the data encoded into each row's circuit.
"""

import functools
import math
import random

import numpy as np
import torch

from quantum_amd import circuits as C
from quantum_amd import layers, math_ops, noise, serialize
from quantum_amd import tfq_adj_grad_op, tfq_simulate_ops


def listed():
    return [
        # A classifier's minibatch: data encoded by rotations, a few trainable
        # layers, the Expectation layer and its backward pass.  The smallest call.
        dict(name="layer_5q_32", op="layer", kind="encoded", n=5, depth=2, batch=32, circuits=1),
        # One VQE iteration: energy and gradient of one 12-qubit ansatz.
        dict(name="vqe_12q", op="value_and_gradient", kind="hea", n=12, depth=6, batch=1,
             circuits=1),
        # Gradients of a deep 10-qubit circuit with 600 symbols over a minibatch.
        dict(name="gradient_10q_64", op="gradient", kind="rotations", n=10, depth=20, batch=64,
             circuits=1),
        # The framework's headline workload: thousands of circuits of 4-16 qubits
        # and 10-60 moments, expectations and gradients in one call.
        dict(name="uneven_2048", op="value_and_gradient", kind="uneven", n=16, depth=60,
             batch=2048, circuits=1),
        # Many parameter sets of one circuit whose state fills a compute unit's memory.
        dict(name="expectation_13q_512", op="expectation", kind="hea", n=13, depth=6, batch=512,
             circuits=1),
        # Energies of a circuit wider than the batched kernel takes.
        dict(name="expectation_22q_2", op="expectation", kind="hea", n=22, depth=6, batch=2,
             circuits=1),
        # Energy and gradient of one 24-qubit ansatz.
        dict(name="gradient_24q", op="value_and_gradient", kind="hea", n=24, depth=4, batch=1,
             circuits=1),
        # The whole final state of a 25-qubit random grid circuit.
        dict(name="state_25q", op="state", kind="grid", n=25, depth=14, batch=1, circuits=1),
        # Bitstrings of a 28-qubit random grid circuit: the largest state.
        dict(name="samples_28q", op="samples", kind="grid", n=28, depth=14, batch=1, circuits=1,
             shots=100000),
        # Shot-based expectations, as on hardware, of a 12-qubit ansatz.
        dict(name="sampled_12q_64", op="sampled", kind="hea", n=12, depth=4, batch=64, circuits=1,
             shots=1000),
        # Monte-Carlo trajectories of noisy variational circuits.
        dict(name="noisy_8q_32", op="noisy", kind="noisy", n=8, depth=8, batch=32, circuits=1,
             shots=1000),
        # Overlaps of a batch of 11-qubit states with two reference states each.
        dict(name="overlap_11q_64", op="overlap", kind="rotations", n=11, depth=8, batch=64,
             circuits=1),
    ]


def draw(rng):
    def log(a, b):
        return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))

    circuits = rng.randrange(2, 1 << 20)
    op = rng.choice(["layer", "vqe", "gradient", "uneven", "expectation", "wide_expectation",
                     "wide_gradient", "state", "samples", "sampled", "noisy", "overlap"])
    if op == "layer":
        return dict(op="layer", kind="encoded", n=rng.randint(3, 9), depth=rng.randint(1, 4),
                    batch=log(4, 64), circuits=circuits)
    if op == "vqe":
        return dict(op="value_and_gradient", kind="hea", n=rng.randint(6, 14),
                    depth=rng.randint(2, 8), batch=log(1, 8), circuits=circuits)
    if op == "gradient":
        return dict(op="gradient", kind="rotations", n=rng.randint(4, 13), depth=rng.randint(4, 20),
                    batch=log(8, 128), circuits=circuits)
    if op == "uneven":
        return dict(op="value_and_gradient", kind="uneven", n=rng.randint(10, 16),
                    depth=rng.randint(20, 60), batch=log(100, 1500), circuits=circuits)
    if op == "expectation":
        return dict(op="expectation", kind="hea", n=rng.randint(8, 17), depth=rng.randint(2, 8),
                    batch=log(16, 256), circuits=circuits)
    if op == "wide_expectation":
        return dict(op="expectation", kind="hea", n=rng.randint(19, 24), depth=rng.randint(2, 6),
                    batch=log(1, 4), circuits=circuits)
    if op == "wide_gradient":
        return dict(op="value_and_gradient", kind="hea", n=rng.randint(19, 23),
                    depth=rng.randint(2, 5), batch=log(1, 3), circuits=circuits)
    if op == "state":
        return dict(op="state", kind="grid", n=rng.randint(12, 25), depth=rng.randint(6, 14),
                    batch=1, circuits=circuits)
    if op == "samples":
        return dict(op="samples", kind="grid", n=rng.randint(12, 26), depth=rng.randint(6, 14),
                    batch=1, circuits=circuits, shots=log(1000, 100000))
    if op == "sampled":
        return dict(op="sampled", kind="hea", n=rng.randint(6, 14), depth=rng.randint(2, 6),
                    batch=log(8, 64), circuits=circuits, shots=log(200, 5000))
    if op == "noisy":
        return dict(op="noisy", kind="noisy", n=rng.randint(3, 12), depth=rng.randint(2, 8),
                    batch=log(4, 32), circuits=circuits, shots=log(50, 500))
    return dict(op="overlap", kind="rotations", n=rng.randint(4, 13), depth=rng.randint(2, 12),
                batch=log(8, 64), circuits=circuits)


# ----------------------------------------------------------------------------- circuits
# A gate is (name, qubits, params); a param is a number or a symbol's name.
# Rotations rx, ry, rz take an angle; xp, yp, zp, czp, iswp an exponent.

def _ladder(n):
    return [[("cz", (i, i + 1), ()) for i in range(0, n - 1, 2)],
            [("cz", (i, i + 1), ()) for i in range(1, n - 1, 2)]]


def _rotations(n, depth):
    out = []
    for l in range(depth):
        for k in "xyz":
            out.append([("r" + k, (i,), (f"{k}{l}_{i}",)) for i in range(n)])
        out += _ladder(n)
    return out


def _hea(n, depth):
    out = []
    for l in range(depth):
        out.append([("ry", (i,), (f"y{l}_{i}",)) for i in range(n)])
        out.append([("rz", (i,), (f"z{l}_{i}",)) for i in range(n)])
        out.append([("cz", (i, i + 1), ()) for i in range(0, n - 1, 2)])
        out.append([("cz", (i, (i + 1) % n), ()) for i in range(1, n if n % 2 == 0 else n - 1, 2)])
    return out


def _grid_shape(n):
    """The most square grid of n places: (rows, columns)."""
    r = max(d for d in range(1, int(math.isqrt(n)) + 1) if n % d == 0)
    return r, n // r


def _grid(n, depth, rng):
    rows, cols = _grid_shape(n)
    at = lambda r, c: r * cols + c  # noqa: E731
    pairs = [[(at(r, c), at(r, c + 1)) for r in range(rows) for c in range(p, cols - 1, 2)]
             for p in (0, 1)]
    pairs += [[(at(r, c), at(r + 1, c)) for r in range(p, rows - 1, 2) for c in range(cols)]
              for p in (0, 1)]
    last = [None] * n
    out = [[("ry", (q,), (f"a{q}",)) for q in range(n)]]  # the product state it starts from
    for cycle in range(depth):
        ops = []
        for q in range(n):
            last[q] = rng.choice([g for g in ("x", "y", "w") if g != last[q]])
            ops.append(("w", (q,), (0.25, 0.5)) if last[q] == "w" else (last[q] + "p", (q,), (0.5,)))
        out.append(ops)
        out.append([("fsim", p, (math.pi / 2, math.pi / 6)) for p in pairs[cycle % 4]])
    return out


def _uneven(n_max, depth_max, rng):
    n, depth = rng.randint(4, n_max), rng.randint(10, depth_max)

    def param():
        return f"p{rng.randrange(256)}" if rng.random() < 0.3 else rng.uniform(-1, 1)

    out = []
    for _ in range(depth):
        free, ops = rng.sample(range(n), n), []
        while free:
            if len(free) >= 2 and rng.random() < 0.5:
                q = (free.pop(), free.pop())
                g = rng.choice(["cnot", "czp", "iswp", "fsim"])
                ops.append((g, q, {"cnot": 0, "czp": 1, "iswp": 1, "fsim": 2}[g]))
            else:
                g = rng.choice(["h", "xp", "yp", "zp"])
                ops.append((g, (free.pop(),), 0 if g == "h" else 1))
        out.append([(g, q, tuple(param() for _ in range(k))) for g, q, k in ops])
    return n, out


def _noisy(n, depth):
    out = []
    for l in range(depth):
        out.append([("ry", (i,), (f"y{l}_{i}",)) for i in range(n)])
        out += _ladder(n)
        out.append([("depolarize", (i,), (0.01,)) for i in range(n)])
        out.append([("damp", (i,), (0.02,)) for i in range(n)])
    return out


def _symbols(moments):
    seen = {}
    for m in moments:
        for _, _, params in m:
            for p in params:
                if isinstance(p, str):
                    seen.setdefault(p, len(seen))
    return list(seen)


def _build(moments, qubits):
    """The framework's circuit of ``moments``."""
    def p(x):
        return C.Symbol(x) if isinstance(x, str) else x

    def gate(g, a):
        if g == "cz":
            return C.CZ
        if g == "cnot":
            return C.CNOT
        if g == "h":
            return C.H
        if g in ("rx", "ry", "rz"):
            return getattr(C, g)(p(a[0]))
        if g == "w":
            return C.PhasedXPowGate(phase_exponent=a[0], exponent=a[1])
        if g == "fsim":
            return C.FSimGate(p(a[0]), p(a[1]))
        if g == "depolarize":
            return C.depolarize(a[0])
        if g == "damp":
            return C.amplitude_damp(a[0])
        return {"xp": C.XPowGate, "yp": C.YPowGate, "zp": C.ZPowGate, "czp": C.CZPowGate,
                "iswp": C.ISwapPowGate}[g](exponent=p(a[0]))

    return C.Circuit.from_moments([[gate(g, a).on(*[qubits[i] for i in q]) for g, q, a in m]
                                   for m in moments])


def _qubits(case, n):
    if case["kind"] == "grid":
        rows, cols = _grid_shape(n)
        return [C.GridQubit(r, c) for r in range(rows) for c in range(cols)]
    return C.LineQubit.range(n)


def _pauli_sum(terms, qubits):
    return C.PauliSum([C.PauliString({qubits[i]: c for i, c in p.items()}, w) for w, p in terms])


# Observables as lists of Pauli sums; a sum is a list of (weight, {qubit: "X" | "Y" | "Z"}).
def _observables(case, n, rng):
    zz = [(1.0, {i: "Z", i + 1: "Z"}) for i in range(n - 1)]
    if case["kind"] == "uneven":
        sums = []
        for _ in range(rng.randint(1, 8)):
            where = rng.sample(range(n), rng.randint(1, min(4, n)))
            sums.append([(round(rng.uniform(0.1, 1), 4), {i: rng.choice("XYZ") for i in where})])
        return sums + [[] for _ in range(8 - len(sums))]
    if case["op"] in ("expectation", "value_and_gradient"):  # transverse-field Ising energy
        return [zz + [(0.7, {i: "X"}) for i in range(n)]]
    if case["op"] == "sampled":
        return [zz, [(1.0, {0: "X"}), (0.5, {n - 1: "Y"})]]
    return [zz, [(1.0, {0: "X"})]]


def _distinct(case):
    """How many different circuits an uneven batch holds; each is there with
    several parameter sets."""
    return min(256, max(16, case["batch"] // 4))


@functools.lru_cache(maxsize=4)
def _model_of(key):
    case = dict(key)
    rng = random.Random(case["circuits"])
    n, depth, kind = case["n"], case["depth"], case["kind"]
    if kind == "uneven":
        shapes = [_uneven(n, depth, rng) for _ in range(_distinct(case))]
        names = [f"p{i}" for i in range(256)]
    else:
        shapes = [(n, {"rotations": _rotations, "hea": _hea, "encoded": _rotations,
                       "noisy": _noisy}[kind](n, depth) if kind != "grid" else
                   _grid(n, depth, rng))]
        names = _symbols(shapes[0][1])
    models = []
    for m, moments in shapes:
        q = _qubits(case, m)
        sums = _observables(case, m, rng)
        models.append((m, moments, serialize.convert_to_tensor([_build(moments, q)])[0], sums,
                       serialize.convert_to_tensor([[_pauli_sum(s, q) for s in sums]])[0]))
    others = None
    if case["op"] == "overlap":  # two fixed reference states
        rows = []
        for _ in range(2):
            fixed = [[(g if g == "cz" else g[1] + "p", q, tuple(rng.uniform(-1, 1) for _ in a))
                      for g, q, a in mo] for mo in _rotations(n, 2)]
            rows.append((fixed, serialize.convert_to_tensor([_build(fixed, C.LineQubit.range(n))])[0]))
        others = rows
    return models, names, others


def _model(case):
    return _model_of(tuple(sorted((k, v) for k, v in case.items() if k != "name")))


def _row_model(case, models, row):
    return models[row % len(models)]


def _data(case, seed):
    """Symbol values, upstream gradients and encoded data of one seed."""
    models, names, _ = _model(case)
    rng = np.random.default_rng(seed)
    batch, slots = case["batch"], len(models[0][3])
    values = rng.uniform(-math.pi, math.pi, (batch, len(names))).astype(np.float32)
    grads = rng.uniform(0.5, 1.5, (batch, slots)).astype(np.float32)
    grads *= np.where(rng.random((batch, slots)) < 0.5, -1, 1).astype(np.float32)
    data = rng.uniform(-1, 1, (batch, case["n"])).astype(np.float32)
    return values, grads, data


def _encoding(row):
    return [[("xp", (i,), (float(x),)) for i, x in enumerate(row)]]


def prepare(case, seed):
    models, names, others = _model(case)
    values, grads, data = _data(case, seed)
    batch = case["batch"]
    state = dict(case=case, names=names, values=values, grads=grads)
    if case["kind"] == "encoded":
        q = C.LineQubit.range(case["n"])
        state["programs"] = serialize.convert_to_tensor(
            [_build(_encoding(data[i]) + models[0][1], q) for i in range(batch)])
    else:
        programs = np.empty(batch, dtype=object)
        programs[:] = [_row_model(case, models, i)[2] for i in range(batch)]
        state["programs"] = programs
    sums = np.empty((batch, len(models[0][3])), dtype=object)
    for i in range(batch):
        sums[i, :] = _row_model(case, models, i)[4]
    state["sums"] = sums
    if case["op"] == "layer":
        state["layer"] = layers.Expectation()
        state["values"] = torch.from_numpy(values).cuda().requires_grad_(True)
        state["grads"] = torch.from_numpy(grads).cuda()
    if others is not None:
        state["others"] = np.empty((batch, len(others)), dtype=object)
        for k, (_, program) in enumerate(others):
            state["others"][:, k] = program
    if "shots" in case:
        state["shots"] = np.full(sums.shape, case["shots"], np.int32)
        state["seed"] = int(seed) & 0xFFFFFFFF
    return state


def run(state):
    case, op = state["case"], state["case"]["op"]
    args = (state["programs"], state["names"], state["values"])
    if op == "layer":
        out = state["layer"](state["programs"], symbol_names=state["names"],
                             symbol_values=state["values"], operators=state["sums"])
        grad, = torch.autograd.grad(out, state["values"], state["grads"])
        return out, grad
    if op == "value_and_gradient":
        return tfq_adj_grad_op.expectation_and_gradient(*args, state["sums"], state["grads"])
    if op == "gradient":
        return tfq_adj_grad_op.tfq_adj_grad(*args, state["sums"], state["grads"])
    if op == "expectation":
        return tfq_simulate_ops.tfq_simulate_expectation(*args, state["sums"])
    if op == "state":
        return tfq_simulate_ops.tfq_simulate_state(*args)
    if op == "samples":
        return tfq_simulate_ops.tfq_simulate_samples(*args, [case["shots"]], seed=state["seed"])
    if op == "sampled":
        return tfq_simulate_ops.tfq_simulate_sampled_expectation(
            *args, state["sums"], state["shots"], seed=state["seed"])
    if op == "noisy":
        return noise.expectation(*args, state["sums"], state["shots"], seed=state["seed"])
    return math_ops.inner_product(*args, state["others"])


# ----------------------------------------------------------------------------- work
_DIAGONAL = ("cz", "czp", "zp", "rz")
_CHANNELS = ("depolarize", "damp")


def _gate_flops(g, q):
    """Real operations per amplitude of one gate applied by itself."""
    return 6 if g in _DIAGONAL else 8 * 2 ** len(q) - 2


def _row_flops(case, n, moments, sums):
    amps = 2.0 ** n
    gates = [(g, q, a) for m in moments for g, q, a in m if g not in _CHANNELS]
    forward = sum(_gate_flops(g, q) for g, q, _ in gates)
    terms = 8 * sum(len(s) for s in sums)
    op = case["op"]
    if op == "noisy":
        # Per channel: the reduced density matrix of its qubit (damping only).
        forward += sum(8 for m in moments for g, _, _ in m if g == "damp")
        return amps * (forward + terms) * case["shots"]
    flops = forward
    if op in ("gradient", "value_and_gradient", "layer"):
        flops += 2 * forward + terms  # both states run back, lambda is summed
        flops += sum(sum(isinstance(p, str) for p in a) * (_gate_flops(g, q) + 8)
                     for g, q, a in gates)
    if op in ("expectation", "value_and_gradient", "layer"):
        flops += terms
    if op in ("samples", "sampled"):
        flops += 4
    return amps * flops


def work(case):
    models, names, others = _model(case)
    batch, op, slots = case["batch"], case["op"], len(models[0][3])
    flops = bytes_ = 0.0
    for i in range(batch):
        n, moments, _, sums, _ = _row_model(case, models, i)
        flops += _row_flops(case, n, moments, sums)
        if n > 20:  # a state that does not stay in a cache is written and read once
            bytes_ += 16 * 2.0 ** n
    if others is not None:
        flops += batch * sum(_row_flops(case, case["n"], m, []) + 8 * 2.0 ** case["n"]
                             for m, _ in others)
    bytes_ += 4.0 * batch * len(names)
    if op == "state":
        bytes_ += 8 * 2.0 ** case["n"] * batch
    elif op == "samples":
        bytes_ += float(case["shots"]) * case["n"] * batch
    elif op == "overlap":
        bytes_ += 8.0 * batch * len(others)
    if op in ("expectation", "value_and_gradient", "layer", "sampled", "noisy"):
        bytes_ += 4.0 * batch * slots
    if op in ("gradient", "value_and_gradient", "layer"):
        bytes_ += 4.0 * batch * (len(names) + slots)
    return {"bytes": bytes_, "flops": flops}


def tolerance(case):
    # About four times what other fusions of the gates and the path without the
    # register engine differ by (float32 amplitudes, float64 sums): 1.7e-6 at most.
    # Shots and Kraus choices are drawn by comparing a prefix sum of the state
    # with a uniform, so a rounding can move one to its neighbour.
    if case["op"] == "samples":
        return {"rel": 0.0, "differ": 0.008}
    if case["op"] == "sampled":
        return {"rel": 4e-3, "max": 0.03}
    if case["op"] == "noisy":  # one trajectory in a row's hundreds may choose otherwise
        return {"rel": 4e-3, "max": 0.1}
    if case["op"] in ("gradient", "value_and_gradient", "layer"):
        return {"rel": 8e-6, "max": 2e-4}
    return {"rel": 4e-6, "max": 3e-5}


# ----------------------------------------------------------------------------- exact
# complex128 simulation of the tuples above.  A state is [batch, 2^n], qubit 0
# the most significant bit.  Arguments are float32 and rotations scale them by
# 1/pi in float32, and the wire format rounds every number to six decimals (the
# 1/pi too): that is how the op's inputs are defined.
_F32 = torch.float32
_X = [[0, 1], [1, 0]]
_Y = [[0, -1j], [1j, 0]]
_Z = [[1, 0], [0, -1]]


def _mat(rows, device):
    return torch.tensor(rows, dtype=torch.complex128, device=device)


def _projectors(name, device):
    """[(eigenvalue, projector)] with U(t) = sum exp(i pi t (eigenvalue + shift)) P."""
    eye = torch.eye(2, dtype=torch.complex128, device=device)
    if name in ("x", "y", "z", "h"):
        h = [[math.sqrt(0.5), math.sqrt(0.5)], [math.sqrt(0.5), -math.sqrt(0.5)]]
        p = _mat({"x": _X, "y": _Y, "z": _Z, "h": h}[name], device)
        return [(0.0, (eye + p) / 2), (1.0, (eye - p) / 2)]
    four = torch.eye(4, dtype=torch.complex128, device=device)
    if name in ("cz", "cnot"):
        sub = _projectors("z" if name == "cz" else "x", device)[1][1]
        low = torch.zeros(4, 4, dtype=torch.complex128, device=device)
        low[2:, 2:] = sub
        return [(0.0, four - low), (1.0, low)]
    plus = torch.zeros(4, 4, dtype=torch.complex128, device=device)
    minus = plus.clone()
    plus[1:3, 1:3] = 0.5
    minus[1:3, 1:3] = _mat([[0.5, -0.5], [-0.5, 0.5]], device)
    return [(0.0, four - plus - minus), (0.5, plus), (-0.5, minus)]


_PROJECTORS = {}


def _eigen(name, t, shift):
    """U(t) for t [batch] in float64: [batch, d, d]."""
    key = (name, str(t.device))
    if key not in _PROJECTORS:
        _PROJECTORS[key] = _projectors(name, t.device)
    out = 0
    for lam, p in _PROJECTORS[key]:
        out = out + torch.polar(torch.ones_like(t), math.pi * t * (lam + shift))[:, None, None] * p
    return out


def _unitary(g, args):
    """args: float32 tensors [batch], one per parameter; [batch, d, d]."""
    if g in ("rx", "ry", "rz"):
        scale = torch.tensor(round(1.0 / math.pi, 6), dtype=_F32, device=args[0].device)
        return _eigen(g[1], (args[0] * scale).double(), -0.5)
    if g in ("xp", "yp", "zp"):
        return _eigen(g[0], args[0].double(), 0.0)
    if g == "czp":
        return _eigen("cz", args[0].double(), 0.0)
    if g == "iswp":
        return _eigen("iswap", args[0].double(), 0.0)
    if g == "w":
        u = _eigen("x", args[1].double(), 0.0)
        ph = torch.polar(torch.ones_like(args[0].double()), math.pi * args[0].double())
        z = torch.zeros(ph.shape[0], 2, 2, dtype=torch.complex128, device=ph.device)
        z[:, 0, 0], z[:, 1, 1] = 1, ph
        return z @ u @ z.conj()
    theta, phi = args[0].double(), args[1].double()
    u = torch.zeros(theta.shape[0], 4, 4, dtype=torch.complex128, device=theta.device)
    u[:, 0, 0] = 1
    u[:, 1, 1] = u[:, 2, 2] = torch.cos(theta).to(torch.complex128)
    u[:, 1, 2] = u[:, 2, 1] = -1j * torch.sin(theta)
    u[:, 3, 3] = torch.polar(torch.ones_like(phi), -phi)
    return u


_FIXED = {"cz": ("cz", 1.0), "cnot": ("cnot", 1.0), "h": ("h", 1.0)}


class _Gates:
    """Matrices of a circuit's gates for values [batch, symbols] (float32)."""

    def __init__(self, names, values):
        self.column = {s: i for i, s in enumerate(names)}
        self.values = values

    def args(self, a):
        return [self.values[:, self.column[p]] if isinstance(p, str) else
                torch.full((1,), round(p, 6), dtype=_F32, device=self.values.device) for p in a]

    def broadcast(self, args):
        b = max((x.shape[0] for x in args), default=1)
        return [x.expand(b) for x in args]

    def unitary(self, g, a):
        if g in _FIXED:
            name, t = _FIXED[g]
            return _eigen(name, torch.full((1,), t, dtype=torch.float64, device=self.values.device),
                          0.0)
        return _unitary(g, self.broadcast(self.args(a)))

    def derivative(self, g, a, k):
        """The gradient gate of parameter k: the float32 central difference with
        eps = 5e-3 that the ops define their default gradient by."""
        eps = np.float32(5e-3)
        up, down = self.args(a), self.args(a)
        up[k], down[k] = up[k] + float(eps), down[k] - float(eps)
        u, d = _unitary(g, self.broadcast(up)), _unitary(g, self.broadcast(down))
        scale = float(np.float32(0.5 / float(eps)))
        diff = [(x.to(_F32) - y.to(_F32)) * scale for x, y in ((u.real, d.real), (u.imag, d.imag))]
        return torch.complex(diff[0].double(), diff[1].double())


def _apply(s, u, q, n):
    """u [1 or batch, d, d] on qubits q of s [batch, 2^n]."""
    b = s.shape[0]
    if len(q) == 1:
        v = s.view(b, 2 ** q[0], 2, -1)
        m = u[:, None, :, :, None]
        return (m[:, :, :, 0] * v[:, :, :1] + m[:, :, :, 1] * v[:, :, 1:]).reshape(b, -1)
    i, j = q
    if i > j:  # swap the gate's qubits
        u = u.view(-1, 2, 2, 2, 2).permute(0, 2, 1, 4, 3).reshape(-1, 4, 4)
        i, j = j, i
    v = s.view(b, 2 ** i, 2, 2 ** (j - i - 1), 2, -1).permute(0, 2, 4, 1, 3, 5).reshape(b, 4, -1)
    v = torch.matmul(u.expand(b, 4, 4).contiguous(), v.contiguous())
    v = v.view(b, 2, 2, 2 ** i, 2 ** (j - i - 1), -1).permute(0, 3, 1, 4, 2, 5)
    return v.reshape(b, -1)


def _zero(batch, n, device):
    s = torch.zeros(batch, 2 ** n, dtype=torch.complex128, device=device)
    s[:, 0] = 1
    return s


def _simulate(n, moments, names, values):
    gates = _Gates(names, values)
    s = _zero(values.shape[0], n, values.device)
    for m in moments:
        for g, q, a in m:
            s = _apply(s, gates.unitary(g, a), q, n)
    return s


def _pauli(s, term, n):
    for q, p in term.items():
        s = _apply(s, _mat({"X": _X, "Y": _Y, "Z": _Z}[p], s.device)[None], (q,), n)
    return s


def _inner(a, b):
    return (a.conj() * b).sum(-1)


def _expectations(s, sums, n):
    out = torch.zeros(s.shape[0], len(sums), dtype=torch.float64, device=s.device)
    for j, terms in enumerate(sums):
        for w, p in terms:
            out[:, j] += float(np.float32(w)) * _inner(s, _pauli(s, p, n)).real
    return out


def _gradients(s, n, moments, names, values, sums, grads):
    """d(sum_j grads[:, j] <O_j>) / d values by running s and lambda back."""
    gates = _Gates(names, values)
    lam = torch.zeros_like(s)
    for j, terms in enumerate(sums):
        for w, p in terms:
            c = grads[:, j] * float(np.float32(w))
            lam += c.double()[:, None] * _pauli(s, p, n)
    out = torch.zeros(values.shape, dtype=torch.float64, device=s.device)
    for m in reversed(moments):
        for g, q, a in reversed(m):
            back = gates.unitary(g, a).conj().transpose(1, 2)
            s = _apply(s, back, q, n)
            for k, p in enumerate(a):
                if isinstance(p, str):
                    d = _apply(s, gates.derivative(g, a, k), q, n)
                    out[:, gates.column[p]] += 2 * _inner(d, lam).real
            lam = _apply(lam, back, q, n)
    return out


def exact(case, seed):
    op = case["op"]
    if op in ("samples", "sampled", "noisy"):
        return None  # drawn at random
    models, names, others = _model(case)
    values, grads, data = _data(case, seed)
    device = "cuda" if torch.cuda.is_available() else "cpu"
    batch, slots = case["batch"], len(models[0][3])
    values = torch.from_numpy(values).to(device)
    grads = torch.from_numpy(grads).to(device)
    if op == "state":
        return _simulate(case["n"], models[0][1], names, values)
    if op == "overlap":
        s = _simulate(case["n"], models[0][1], names, values)
        return torch.stack([_inner(s, _simulate(case["n"], m, [], values[:1, :0]))
                            for m, _ in others], 1)
    value = torch.zeros(batch, slots, dtype=torch.float64, device=device)
    gradient = torch.zeros(batch, len(names), dtype=torch.float64, device=device)
    if case["kind"] == "encoded":
        rows = [([i], case["n"], _encoding(data[i]) + models[0][1], models[0][3])
                for i in range(batch)]
    else:
        # Rows of one circuit together, within 8 GiB per state.
        rows = []
        for k, (n, moments, _, sums, _) in enumerate(models):
            mine = list(range(k, batch, len(models)))
            step = max(1, 2 ** 29 // 2 ** n)
            rows += [(mine[i:i + step], n, moments, sums) for i in range(0, len(mine), step)]
    for at, n, moments, sums in rows:
        if not at:
            continue
        s = _simulate(n, moments, names, values[at])
        if op != "gradient":
            value[at] = _expectations(s, sums, n)
        if op != "expectation":
            gradient[at] = _gradients(s, n, moments, names, values[at], sums, grads[at])
    if op == "expectation":
        return value
    return gradient if op == "gradient" else (value, gradient)
