"""Circuits of 14-16 qubits on the HBM-streaming path (the streaming threshold
lowered to 14): expectation, adjoint gradient with expectation, and state
against the complex128 oracle at 1e-5, one circuit per plan and a mixed batch.
The default planner runs these widths inside the batched kernel; the lowered
threshold is what a lone wide circuit uses on its own."""

import sys

import numpy as np
import pytest

from oracle import tfq_oracle as O
from quantum_amd import _lib
from quantum_amd import circuits as C
from quantum_amd import serialize as S
from quantum_amd import workloads as W

pytestmark = pytest.mark.gpu

TOL = 1e-5


def _say(msg):
    print(f"[gpu-case] {msg}", file=sys.stderr, flush=True)


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    _lib.set_streaming_min_qubits(14)
    yield
    _lib.set_streaming_min_qubits(-1)


def _batch(seed, widths):
    rng = np.random.default_rng(seed)
    names = [f"s{i}" for i in range(4)]
    circuits, sums = [], []
    for n in widths:
        q = C.LineQubit.range(n)
        circuits.append(W.random_circuit(rng, q, 2 * n, symbols=names, p_symbol=0.5,
                                         p_control=0.1) + C.Circuit([C.I(x) for x in q]))
        sums.append([W.random_pauli_sum(rng, q, 3, max_weight=4) for _ in range(2)])
    B = len(widths)
    return (S.convert_to_tensor(circuits), names, rng.uniform(-3, 3, size=(B, 4)).astype(np.float32),
            S.convert_to_tensor(sums), rng.uniform(-1, 1, size=(B, 2)).astype(np.float32))


@pytest.mark.parametrize("widths", [[14], [15], [16], [16, 14, 15]])
def test_streaming_expectation_and_adjoint(widths):
    from quantum_amd import tfq_adj_grad_op as A
    from quantum_amd import tfq_simulate_ops as sim
    progs, names, vals, ps, g = _batch(sum(widths), widths)
    plan, _ = A.plan_adj_grad(progs, names, vals, ps, g, with_expectation=True)
    assert plan.stats()["streaming"], "threshold 14 must select the streaming path"
    del plan
    _say(f"streaming expectation+adjoint widths={widths}")
    e = sim.tfq_simulate_expectation(progs, names, vals, ps).cpu().numpy()
    ee, gg = A.expectation_and_gradient(progs, names, vals, ps, g, derivative="analytic")
    eo = O.simulate_expectation(list(progs), names, vals, ps)
    go = O.adjoint_gradient(list(progs), names, vals, ps, g, mode="analytic")
    np.testing.assert_allclose(e, eo, atol=TOL * max(1, np.abs(eo).max()))
    np.testing.assert_allclose(ee.cpu().numpy(), eo, atol=TOL * max(1, np.abs(eo).max()))
    np.testing.assert_allclose(gg.cpu().numpy(), go, atol=TOL * max(1, np.abs(go).max()))


def test_streaming_state():
    from quantum_amd import tfq_simulate_ops as sim
    progs, names, vals, _, _ = _batch(3, [15, 14])
    _say("streaming state widths=[15, 14]")
    st = sim.tfq_simulate_state(progs, names, vals).cpu().numpy()
    so = O.simulate_state(list(progs), names, vals)
    np.testing.assert_allclose(st, so, atol=TOL)


def _strings(kind, n, rng):
    """Pauli strings (as {qubit: axis}) that the term sweeps take apart."""
    high = lambda b: n - 1 - b  # qubit of bit b  # noqa: E731
    if kind == "z":
        return [{high(i): "Z", high((i + 5) % n): "Z"} for i in range(n)]
    if kind == "every bit":  # one flipped qubit each, with Y and Z beside it
        return [{high(i): "XY"[i % 2], high((i + 1) % n): "Z"} for i in range(n)]
    if kind == "wide":  # flips more high qubits than a tile holds
        return [{high(b): "XY"[b % 2] for b in range(6, 14)}, {high(0): "Z"},
                {high(b): "X" for b in range(n)}]
    if kind == "only high":  # nothing for the contiguous tile
        return [{high(n - 1): "X", high(n - 2): "Y"}, {high(n - 1): "Y", high(2): "X"}]
    # More different sets of high qubits than there are sweeps.
    return [{high(b): "XYZ"[rng.integers(3)] for b in rng.choice(n, 5, replace=False)}
            for _ in range(60)]


@pytest.mark.parametrize("n,kind", [(14, "z"), (14, "every bit"), (16, "every bit"), (14, "wide"),
                                    (15, "only high"), (16, "many")])
def test_streaming_terms(n, kind):
    from quantum_amd import tfq_adj_grad_op as A
    rng = np.random.default_rng(n)
    q = C.LineQubit.range(n)
    circuit = W.random_circuit(rng, q, n, symbols=["a", "b"], p_symbol=0.5) + \
        C.Circuit([C.H(x) for x in q])
    strings = _strings(kind, n, rng)
    terms = [C.PauliString({q[i]: c for i, c in s.items()}, float(rng.uniform(-1, 1)))
             for s in strings]
    sums = [C.PauliSum(terms), C.PauliSum(terms[:1] + [C.PauliString({}, 0.5)]), C.PauliSum([])]
    progs, ps = S.convert_to_tensor([circuit]), S.convert_to_tensor([sums])
    v = rng.uniform(-2, 2, (1, 2)).astype(np.float32)
    g = np.array([[0.7, -0.4, 1.0]], np.float32)
    _say(f"streaming terms n={n} {kind}")
    e, grad = A.expectation_and_gradient(progs, ["a", "b"], v, ps, g, derivative="analytic")
    eo = O.simulate_expectation(list(progs), ["a", "b"], v, ps)
    go = O.adjoint_gradient(list(progs), ["a", "b"], v, ps, g, mode="analytic")
    np.testing.assert_allclose(e.cpu().numpy(), eo, atol=TOL * max(1, np.abs(eo).max()))
    np.testing.assert_allclose(grad.cpu().numpy(), go, atol=TOL * max(1, np.abs(go).max()))
