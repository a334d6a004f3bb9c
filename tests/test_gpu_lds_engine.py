"""The LDS gate engine (circuits of 2-11 qubits run by workgroups) where it
changes what it does: one wavefront up to 8 qubits and several above, groups that
do not fill a wavefront, op lists longer than the descriptor window (144 ops),
more derivatives than the partial ring holds (8), one-qubit ops whose other group
qubit is a control, and more Pauli terms than the term window (240).

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


def _close(out, ref):
    np.testing.assert_allclose(out, ref, atol=TOL * max(1.0, np.abs(ref).max()))


@pytest.mark.parametrize("n,ops,width", [(2, 200, 1), (3, 40, 1), (7, 60, 2), (8, 330, 1),
                                         (9, 60, 2), (10, 330, 1), (11, 60, 2)])
def test_adjoint_and_state(n, ops, width):
    from quantum_amd import tfq_adj_grad_op as A
    from quantum_amd import tfq_simulate_ops as sim
    _lib.set_fusion_width(width)
    rng = np.random.default_rng(n * 100 + ops)
    q = C.LineQubit.range(n)
    names = [f"s{i}" for i in range(6)]
    circuits = [W.random_circuit(rng, q, ops, symbols=names, p_symbol=0.5, p_control=0.3) +
                C.Circuit([C.I(x) for x in q]) for _ in range(2)]
    progs = S.convert_to_tensor(circuits)
    sums = S.convert_to_tensor([[W.random_pauli_sum(rng, q, 4) for _ in range(2)]] * 2)
    v = rng.uniform(-2, 2, size=(2, 6)).astype(np.float32)
    g = rng.uniform(-1, 1, size=(2, 2)).astype(np.float32)
    print(f"[gpu-case] lds engine n={n} ops={ops} width={width}", flush=True)
    e, grad = A.expectation_and_gradient(progs, names, v, sums, g, derivative="analytic")
    _close(e.cpu().numpy(), O.simulate_expectation(list(progs), names, v, sums))
    _close(grad.cpu().numpy(), O.adjoint_gradient(list(progs), names, v, sums, g, mode="analytic"))
    state = sim.tfq_simulate_state(progs, names, v).cpu().numpy()
    np.testing.assert_allclose(state, O.simulate_state(list(progs), names, v), atol=TOL)


@pytest.mark.parametrize("n,ops", [(4, 40), (9, 60)])
def test_inner_product_grad(n, ops):
    from quantum_amd import math_ops
    rng = np.random.default_rng(n)
    q = C.LineQubit.range(n)
    names = [f"s{i}" for i in range(5)]
    make = lambda sym: W.random_circuit(rng, q, ops, symbols=sym, p_symbol=0.6,  # noqa: E731
                                        p_control=0.2) + C.Circuit([C.I(x) for x in q])
    progs = S.convert_to_tensor([make(names) for _ in range(2)])
    other = S.convert_to_tensor([[make(()) for _ in range(2)] for _ in range(2)])
    v = rng.uniform(-2, 2, size=(2, 5)).astype(np.float32)
    g = rng.uniform(-1, 1, size=(2, 2)).astype(np.float32)
    print(f"[gpu-case] lds engine inner-product gradient n={n}", flush=True)
    out = math_ops.inner_product_grad(progs, names, v, other, g, derivative="analytic")
    # The op returns the conjugate of the oracle's <d psi | phi> sums.
    ref = O.inner_product_gradient(list(progs), names, v, other, g, mode="analytic")
    _close(out.cpu().numpy(), np.conj(ref))


def test_more_terms_than_the_window():
    from quantum_amd import tfq_adj_grad_op as A
    rng = np.random.default_rng(5)
    n = 6
    q = C.LineQubit.range(n)
    progs = S.convert_to_tensor([W.random_circuit(rng, q, 30, symbols=["a"], p_symbol=0.5) +
                                 C.Circuit([C.I(x) for x in q])])
    sums = S.convert_to_tensor([[W.random_pauli_sum(rng, q, 239), W.random_pauli_sum(rng, q, 2),
                                 W.random_pauli_sum(rng, q, 260)]])
    v = np.array([[0.37]], np.float32)
    g = np.array([[0.5, -1.0, 0.25]], np.float32)
    print("[gpu-case] lds engine, 501 Pauli terms", flush=True)
    e, grad = A.expectation_and_gradient(progs, ["a"], v, sums, g, derivative="analytic")
    _close(e.cpu().numpy(), O.simulate_expectation(list(progs), ["a"], v, sums))
    _close(grad.cpu().numpy(), O.adjoint_gradient(list(progs), ["a"], v, sums, g, mode="analytic"))
