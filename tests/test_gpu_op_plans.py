"""Ops that reuse their plans across calls (state, samples, sampled expectation,
inner product): a call with new values, and a new seed, equals the same call with the
cache off, bit for bit, since either evaluates the matrices on the device."""

import numpy as np
import pytest

from quantum_amd import circuits as C
from quantum_amd import plan_cache
from quantum_amd import serialize as S
from quantum_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _need_gpu():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    plan_cache.clear()
    yield
    plan_cache.set_capacity(8)


def _ops(progs, names, sums, other):
    from quantum_amd import math_ops, tfq_simulate_ops as sim
    B = len(progs)
    counts = np.arange(1, 2 * B + 1, dtype=np.int32).reshape(B, 2) * 50
    return {
        "state": lambda v, seed: sim.tfq_simulate_state(progs, names, v),
        "samples": lambda v, seed: sim.tfq_simulate_samples(progs, names, v, [300], seed=seed),
        "sampled": lambda v, seed: sim.tfq_simulate_sampled_expectation(
            progs, names, v, sums, counts, seed=seed),
        "inner": lambda v, seed: math_ops.inner_product(progs, names, v, other),
    }


@pytest.mark.parametrize("op", ["state", "samples", "sampled", "inner"])
@pytest.mark.parametrize("widths", [(4, 4, 4), (3, 9, 12), (13, 5, 2)])
def test_reused_plan_equals_a_fresh_one(op, widths):
    rng = np.random.default_rng(sum(widths))
    names = ["a", "b"]
    circuits, sums, other = [], [], []
    for n in widths:
        q = C.LineQubit.range(n)
        make = lambda sym: W.random_circuit(  # noqa: E731
            rng, q, 3 * n, symbols=sym, p_symbol=0.6) + C.Circuit([C.I(x) for x in q])
        circuits.append(make(names))
        sums.append([W.random_pauli_sum(rng, q, 3) for _ in range(2)])
        other.append([make(()), make(())])
    progs, psums, others = map(S.convert_to_tensor, (circuits, sums, other))
    fn = _ops(progs, names, psums, others)[op]
    print(f"[gpu-case] reused plan, {op}, widths {widths}", flush=True)
    values = [rng.uniform(-2, 2, (3, 2)).astype(np.float32) for _ in range(3)]
    got = [fn(v, seed).cpu().numpy() for seed, v in enumerate(values)]
    assert len(plan_cache._CACHE) == 1
    plan_cache.set_capacity(0)
    for seed, (v, g) in enumerate(zip(values, got)):
        np.testing.assert_array_equal(g, fn(v, seed).cpu().numpy())


def test_other_counts_and_shapes_are_other_plans():
    from quantum_amd import tfq_simulate_ops as sim
    q = C.LineQubit.range(3)
    progs = S.convert_to_tensor([C.Circuit(C.H(q[0]), C.CNOT(q[0], q[1]), C.I(q[2]))])
    a = sim.tfq_simulate_samples(progs, [], np.zeros((1, 0), np.float32), [10], seed=1)
    b = sim.tfq_simulate_samples(progs, [], np.zeros((1, 0), np.float32), [20], seed=1)
    assert a.shape == (1, 10, 3) and b.shape == (1, 20, 3)
    np.testing.assert_array_equal(a.cpu().numpy(), b.cpu().numpy()[:, :10])
    assert len(plan_cache._CACHE) == 2


@pytest.mark.parametrize("op", ["state", "samples", "sampled", "inner"])
def test_equal_calls_give_equal_results(op):
    """The same arguments as the first call, with other values in between, after the
    plan has left the cache, and without a cache: the same bits.  A gate and its inverse
    leave matrix entries in which the last bit of a sine or cosine shows."""
    B = 64
    q = C.LineQubit.range(2)
    a = C.Symbol("a")
    circuit = C.Circuit([C.XPowGate(exponent=e).on(x) for e in (a, a * -1.0) for x in q])
    progs = S.convert_to_tensor([circuit] * B)
    sums = S.convert_to_tensor([[C.PauliSum([C.PauliString({q[0]: "X"}, 0.7)])] * 2] * B)
    other = S.convert_to_tensor([[C.Circuit([C.I(x) for x in q])] * 2] * B)
    fn = _ops(progs, ["a"], sums, other)[op]
    v = np.random.default_rng(8).uniform(-3, 3, (B, 1)).astype(np.float32)
    print(f"[gpu-case] equal calls, {op}", flush=True)
    first = fn(v, 3).cpu().numpy()
    fn(np.zeros_like(v), 4)
    np.testing.assert_array_equal(fn(v, 3).cpu().numpy(), first)
    plan_cache.clear()
    np.testing.assert_array_equal(fn(v, 3).cpu().numpy(), first)
    plan_cache.set_capacity(0)
    np.testing.assert_array_equal(fn(v, 3).cpu().numpy(), first)
