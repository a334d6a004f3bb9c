"""The LDS gate engine (circuits of 2-11 qubits run by workgroups) multiplies in
the order of the general gate path (``apply_dense`` and ``apply_diag`` in
``lds_ops.h``), so that seeded draws do not depend on which of them ran.

The state is compared bit for bit with a float32 replica of that order.  A value that is not finite stays with the amplitudes that the general path leaves
it in: a one-qubit op mixes pairs only.  Gradient partials of different pairs of a
one-qubit op are added in float64, as there."""

import numpy as np
import pytest

from oracle import gate_order
from oracle import tfq_oracle as O
from quantum_amd import _lib
from quantum_amd import circuits as C
from quantum_amd import serialize as S
from quantum_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    yield
    _lib.set_fusion_width(0)


@pytest.mark.parametrize("width", [1, 2])
@pytest.mark.parametrize("n", [2, 3, 6, 8, 9, 10, 11])
def test_bits_of_the_general_path(n, width):
    from quantum_amd import tfq_simulate_ops as sim
    _lib.set_fusion_width(width)
    rng = np.random.default_rng(100 * n + width)
    q = C.LineQubit.range(n)
    names = [f"s{i}" for i in range(6)]
    circuits = [C.Circuit([C.H(x) for x in q]) +
                W.random_circuit(rng, q, 40, symbols=names, p_symbol=0.5, p_control=0.3)
                for _ in range(3)]
    progs = S.convert_to_tensor(circuits)
    values = rng.uniform(-2, 2, size=(3, 6)).astype(np.float32)
    print(f"[gpu-case] lds engine bits, n={n} width={width}", flush=True)
    got = sim.tfq_simulate_state(progs, names, values).cpu().numpy()
    want = np.stack([gate_order.state(p, names, v, width) for p, v in zip(progs, values)])
    np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize("n,control", [(3, 0), (3, 2), (8, 7), (10, 9), (10, 8), (11, 0)])
@pytest.mark.parametrize("value", [np.nan, np.inf])
def test_non_finite_amplitudes_stay_where_they_are(n, control, value):
    """A symbol that is not finite in a controlled gate spoils the control's half of the
    state; one-qubit gates on the other qubits keep the other half as it is."""
    from quantum_amd import tfq_simulate_ops as sim
    _lib.set_fusion_width(1)
    q = C.LineQubit.range(n)
    rest = [x for i, x in enumerate(q) if i != control]
    gate = C.XPowGate(exponent=C.Symbol("a")).on(rest[0]).controlled_by(q[control])
    progs = S.convert_to_tensor([C.Circuit([C.H(x) for x in q]) + C.Circuit([gate]) +
                                 C.Circuit([C.YPowGate(exponent=0.3).on(x) for x in rest])])
    print(f"[gpu-case] lds engine, {value} in half of {n} qubits", flush=True)
    got = sim.tfq_simulate_state(progs, ["a"], np.array([[value]], np.float32)).cpu().numpy()[0]
    fine = sim.tfq_simulate_state(progs, ["a"], np.array([[0.5]], np.float32)).cpu().numpy()[0]
    spoilt = ((np.arange(2 ** n) >> (n - 1 - control)) & 1) == 1
    assert not np.isfinite(got[spoilt]).any()
    np.testing.assert_array_equal(got[~spoilt], fine[~spoilt])


@pytest.mark.parametrize("n,ring", [(4, True), (9, True), (10, True), (11, True), (12, False)])
def test_pairs_of_one_qubit_derivatives_meet_in_float64(n, ring):
    """d<Z_p Z_t>/da after an entangler that leaves <Z_p> = d^2, d^2 about 1e-5: the pairs
    with o = 0 contribute +x and -x, equal bits of opposite p, and the pair with o = 1
    the d^2 x that is left.  Its float32 value is good to a few 2^-24 of itself; added
    in float32 to the +x pair it would keep an error of 2^-24 / d^2, up to 6e-3.
    12 qubits without the register engine: more rounds than the ring takes."""
    from quantum_amd import tfq_adj_grad_op as A
    _lib.set_fusion_width(1)
    if not ring:
        _lib.set_tuning(register_engine=0)
    q = C.LineQubit.range(n)
    o, t, p = q[n - 1], q[n - 2], q[n - 3]
    circuit = C.Circuit([C.I(x) for x in q]) + C.Circuit(
        [C.YPowGate(exponent=0.002).on(o), C.H(p)]) + C.Circuit(
        [C.H(p).controlled_by(o), C.YPowGate(exponent=C.Symbol("a")).on(t)])
    batch = 8
    progs = S.convert_to_tensor([circuit] * batch)
    sums = S.convert_to_tensor([[C.PauliSum([C.PauliString({p: "Z", t: "Z"}, 1.0)])]] * batch)
    values = np.linspace(0.2, 0.8, batch).astype(np.float32)[:, None]
    grads = np.ones((batch, 1), np.float32)
    print(f"[gpu-case] lds engine, cancelling pairs, n={n}", flush=True)
    try:
        got = A.tfq_adj_grad(progs, ["a"], values, sums, grads, derivative="analytic").cpu().numpy()
    finally:
        _lib.set_tuning()
    want = O.adjoint_gradient(list(progs), ["a"], values, sums, grads, mode="analytic")
    assert np.abs(want).max() < 1e-4
    # Squares of amplitudes after four gates: 16 roundings of 2^-24 at most.
    np.testing.assert_allclose(got, want, rtol=16 * 2.0 ** -24)
