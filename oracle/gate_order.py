"""Float32 replica of the order in which the gate kernels add a gate's products (test
infrastructure only): a state from it has the bits of theirs.

Matrices are rounded to float32.  A product of two complex numbers m v is one rounded
product and one fused multiply-add per part (rounded first: m.im v.im of the real part,
m.re v.im of the imaginary part), and every further column adds its real products by
fused multiply-adds.  With ``engine`` the order is the register engine's: of the
imaginary part m.im v.re is rounded first, and two-qubit gates (not diagonal ones) add
the products with the real parts of all four amplitudes and then those with the
imaginary parts.

A fused multiply-add is evaluated in float64 (the product is exact there) and rounded to
float32; rounding twice changes one result in 2^29.
"""

import numpy as np

from . import fuser
from . import tfq_oracle as O

F32, F64 = np.float32, np.float64
DIAGONAL = {"I", "ZP", "I2", "CZP", "ZZP"}


def _fma(a, b, c):
    return (a.astype(F64) * b.astype(F64) + c.astype(F64)).astype(F32)


def _cmul(m, v, engine):
    re = _fma(m[0], v[0], -(m[1] * v[1]))
    if engine:
        return re, _fma(m[0], v[1], m[1] * v[0])
    return re, _fma(m[1], v[0], m[0] * v[1])


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


def _parts(cols):
    """Sum of m * v over [(m, v)]: the products with v's real parts first."""
    re, im = np.zeros_like(cols[0][1][0]), np.zeros_like(cols[0][1][0])
    for m, v in cols:
        re, im = _fma(m[0], v[0], re), _fma(m[1], v[0], im)
    for m, v in cols:
        re, im = _fma(-m[1], v[1], re), _fma(m[0], v[1], im)
    return re, im


def state(program, names, values, width, engine=False):
    """The final state (complex64 bits) of one program for one row of symbol values,
    fused to ``width`` qubits."""
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
            new = _cmul((d.real, d.imag), (re, im), engine)
        else:
            M = U.astype(np.complex64)
            rest = x & ~sum(1 << b for b in bits)
            cols = []
            for c in range(2 ** len(bits)):
                src = rest | sum(((c >> j) & 1) << b for j, b in enumerate(bits))
                cols.append(((M[at, c].real, M[at, c].imag), (re[src], im[src])))
            if engine and len(bits) == 2:
                new = _parts(cols)
            else:
                new = _cmul(*cols[0], engine)
                for m, v in cols[1:]:
                    new = _cmac(new, m, v)
        re, im = np.where(ok, new[0], re), np.where(ok, new[1], im)
    return re + 1j * im
