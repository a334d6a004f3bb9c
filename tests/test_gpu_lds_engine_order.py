"""The LDS gate engine (circuits of 2-11 qubits run by workgroups) multiplies in
the order of the general gate path (``apply_dense`` and ``apply_diag`` in
``lds_ops.h``), so that seeded draws do not depend on which of them ran.

The state is compared bit for bit with a float32 replica of that order: the
matrices are rounded to float32, a product of two complex numbers is one rounded
product (the one with the amplitude's imaginary part) and one fused multiply-add per
part, and every further column adds its real products by fused multiply-adds.  A fused multiply-add is evaluated in
float64 (the product is exact there) and rounded to float32; rounding twice
changes one result in 2^29.

A value that is not finite stays with the amplitudes that the general path leaves
it in: a one-qubit op mixes pairs only.  Gradient partials of different pairs of a
one-qubit op are added in float64, as there."""

import numpy as np
import pytest

from oracle import fuser
from oracle import tfq_oracle as O
from quantum_amd import _lib
from quantum_amd import circuits as C
from quantum_amd import serialize as S
from quantum_amd import workloads as W

pytestmark = pytest.mark.gpu

F32, F64 = np.float32, np.float64
DIAGONAL = {"I", "ZP", "I2", "CZP", "ZZP"}


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    yield
    _lib.set_fusion_width(0)


def _fma(a, b, c):
    return (a.astype(F64) * b.astype(F64) + c.astype(F64)).astype(F32)


def _cmul(m, v):
    """m * v: (re, im) float32, the products with v's imaginary part rounded first."""
    return _fma(m[0], v[0], -(m[1] * v[1])), _fma(m[1], v[0], m[0] * v[1])


def _cmac(acc, m, v):
    re = _fma(-m[1], v[1], _fma(m[0], v[0], acc[0]))
    return re, _fma(m[1], v[0], _fma(m[0], v[1], acc[1]))


def _block(gates, bits):
    """The block's matrix; index bit j is ``bits[j]``, controls of a gate inside."""
    k = len(bits)
    at = {b: j for j, b in enumerate(bits)}
    cols = []
    for c in range(2 ** k):
        v = np.zeros(2 ** k, np.complex128)
        v[c] = 1
        for g in gates:
            inside = [b for b in g.cbits if b in at]
            cv = [x for b, x in zip(g.cbits, g.cvals) if b in at]
            v = O.apply_matrix(v, g.unitary(), [at[b] for b in g.bits], k, [at[b] for b in inside], cv)
        cols.append(v)
    return np.stack(cols, 1)


def _replica(program, names, values, width):
    prog = O.Program(program, {n: F32(v) for n, v in zip(names, values)})
    n = prog.n
    masks = [(sum(1 << b for b in g.bits), sum(1 << b for b in g.cbits)) for g in prog.gates]
    x = np.arange(2 ** n)
    re, im = np.zeros(2 ** n, F32), np.zeros(2 ** n, F32)
    re[0] = 1
    for bits, outside, idx in fuser.fuse(masks, width):
        gates = [prog.gates[i] for i in idx]
        ok = np.ones(2 ** n, bool)
        if outside:
            for b, v in zip(gates[0].cbits, gates[0].cvals):
                ok &= ((x >> b) & 1) == v
        U = _block(gates, bits)
        at = sum(((x >> b) & 1) << j for j, b in enumerate(bits))  # this amplitude's row
        if all(g.gid in DIAGONAL for g in gates):
            d = np.diag(U).astype(np.complex64)[at]
            new = _cmul((d.real, d.imag), (re, im))
        else:
            M = U.astype(np.complex64)
            rest = x & ~sum(1 << b for b in bits)
            new = None
            for c in range(2 ** len(bits)):
                src = rest | sum(((c >> j) & 1) << b for j, b in enumerate(bits))
                m, v = (M[at, c].real, M[at, c].imag), (re[src], im[src])
                new = _cmul(m, v) if c == 0 else _cmac(new, m, v)
        re, im = np.where(ok, new[0], re), np.where(ok, new[1], im)
    return re + 1j * im


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
    values = rng.uniform(-2, 2, size=(3, 6)).astype(F32)
    print(f"[gpu-case] lds engine bits, n={n} width={width}", flush=True)
    got = sim.tfq_simulate_state(progs, names, values).cpu().numpy()
    want = np.stack([_replica(p, names, v, width) for p, v in zip(progs, values)])
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
    got = sim.tfq_simulate_state(progs, ["a"], np.array([[value]], F32)).cpu().numpy()[0]
    fine = sim.tfq_simulate_state(progs, ["a"], np.array([[0.5]], F32)).cpu().numpy()[0]
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
    values = np.linspace(0.2, 0.8, batch).astype(F32)[:, None]
    grads = np.ones((batch, 1), F32)
    print(f"[gpu-case] lds engine, cancelling pairs, n={n}", flush=True)
    try:
        got = A.tfq_adj_grad(progs, ["a"], values, sums, grads, derivative="analytic").cpu().numpy()
    finally:
        _lib.set_tuning()
    want = O.adjoint_gradient(list(progs), ["a"], values, sums, grads, mode="analytic")
    assert np.abs(want).max() < 1e-4
    # Squares of amplitudes after four gates: 16 roundings of 2^-24 at most.
    np.testing.assert_allclose(got, want, rtol=16 * 2.0 ** -24)
