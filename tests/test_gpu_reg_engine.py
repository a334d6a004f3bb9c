"""The register engine's variants: a two-qubit op permutes the register slots, so
every op runs on the slot pair that the ops before it left its targets in, in
either order, and its controls are register slots, thread bits or both.  Long
random op lists on the sizes of each register count (12 qubits: 3, 13: 4, one
wavefront per circuit: 4; streaming tiles of 14 qubits: 5) reach all pairs.

float32 gates and states against the complex128 oracle: the suite's 1e-5 of the
largest value, for lists of a few hundred ops."""

import numpy as np
import pytest

from oracle import tfq_oracle as O
from quantum_amd import _lib
from quantum_amd import circuits as C
from quantum_amd import serialize as S
from quantum_amd import workloads as W

pytestmark = pytest.mark.gpu

TOL = 1e-5


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    yield
    _lib.set_fusion_width(0)


def _circuit(rng, q, ops, names, p_control):
    """Random gates with a diagonal two-qubit gate (plain or controlled) between them."""
    out = C.Circuit([C.I(x) for x in q])
    for _ in range(ops // 4):
        out = out + W.random_circuit(rng, q, 3, symbols=names, p_symbol=0.4, p_control=p_control)
        a, b, c = (q[int(i)] for i in rng.choice(len(q), 3, replace=False))
        gate = (C.CZ**float(rng.uniform(-1, 1)))(a, b)
        out = out + C.Circuit([gate.controlled_by(c) if rng.random() < p_control else gate])
    return out


@pytest.mark.parametrize("n,ops,width,p_control,batch", [
    (12, 240, 2, 0.0, 2), (12, 160, 1, 0.4, 2), (13, 240, 2, 0.1, 2), (13, 160, 1, 0.4, 2),
    (8, 120, 2, 0.2, 1100), (10, 80, 1, 0.3, 1100)])
def test_every_slot_pair(n, ops, width, p_control, batch):
    from quantum_amd import tfq_adj_grad_op as A
    from quantum_amd import tfq_simulate_ops as sim
    _lib.set_fusion_width(width)
    rng = np.random.default_rng(n * 1000 + ops)
    q = C.LineQubit.range(n)
    names = [f"s{i}" for i in range(6)]
    two = S.convert_to_tensor([_circuit(rng, q, ops, names, p_control) for _ in range(2)])
    sums2 = S.convert_to_tensor([[W.random_pauli_sum(rng, q, 4)]] * 2)
    reps = batch // 2
    progs, sums = np.tile(two, reps), np.tile(sums2, (reps, 1))
    v = rng.uniform(-2, 2, size=(2, 6)).astype(np.float32)
    g = rng.uniform(-1, 1, size=(2, 1)).astype(np.float32)
    vs, gs = np.tile(v, (reps, 1)), np.tile(g, (reps, 1))
    print(f"[gpu-case] register engine n={n} ops={ops} width={width} batch={batch}", flush=True)
    e, grad = A.expectation_and_gradient(progs, names, vs, sums, gs, derivative="analytic")
    e, grad = e.cpu().numpy(), grad.cpu().numpy()
    ref_e = O.simulate_expectation(list(two), names, v, sums2)
    ref_g = O.adjoint_gradient(list(two), names, v, sums2, g, mode="analytic")
    scale = max(1.0, np.abs(ref_g).max())
    np.testing.assert_allclose(e, np.tile(ref_e, (reps, 1)), atol=TOL * max(1.0, np.abs(ref_e).max()))
    np.testing.assert_allclose(grad, np.tile(ref_g, (reps, 1)), atol=TOL * scale)
    state = sim.tfq_simulate_state(progs, names, vs).cpu().numpy()
    np.testing.assert_allclose(state, np.tile(O.simulate_state(list(two), names, v), (reps, 1)),
                               atol=TOL)


@pytest.mark.parametrize("tile,width,p_control", [(12, 2, 0.2), (13, 1, 0.4), (14, 2, 0.2)])
def test_streaming_tiles(tile, width, p_control):
    from quantum_amd import tfq_adj_grad_op as A
    n, ops = 15, 160
    _lib.set_fusion_width(width)
    rng = np.random.default_rng(tile)
    q = C.LineQubit.range(n)
    names = [f"s{i}" for i in range(6)]
    progs = S.convert_to_tensor([_circuit(rng, q, ops, names, p_control)])
    sums = S.convert_to_tensor([[W.random_pauli_sum(rng, q, 4)]])
    v = rng.uniform(-2, 2, size=(1, 6)).astype(np.float32)
    g = rng.uniform(-1, 1, size=(1, 1)).astype(np.float32)
    print(f"[gpu-case] register engine streaming tile={tile} width={width}", flush=True)
    _lib.set_streaming_min_qubits(14)
    try:
        _lib.set_tuning(tile_single=tile, tile_two=min(tile, 13))
        e, grad = A.expectation_and_gradient(progs, names, v, sums, g, derivative="analytic")
        e, grad = e.cpu().numpy(), grad.cpu().numpy()
    finally:
        _lib.set_tuning()
        _lib.set_streaming_min_qubits(-1)
    ref_e = O.simulate_expectation(list(progs), names, v, sums)
    ref_g = O.adjoint_gradient(list(progs), names, v, sums, g, mode="analytic")
    np.testing.assert_allclose(e, ref_e, atol=TOL * max(1.0, np.abs(ref_e).max()))
    np.testing.assert_allclose(grad, ref_g, atol=TOL * max(1.0, np.abs(ref_g).max()))
