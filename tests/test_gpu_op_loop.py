"""The compiled op loop (no generated kernels): every op family on every register bit, controlled and not, and
phase ops with their integer form (equal multiples of one angle) and without, against the oracle."""

import numpy as np
import pytest

from aleph_amd.circuit import Circuit, DiagonalPhase, Gate, PhaseTerm
from tests.helpers import max_abs

pytestmark = pytest.mark.gpu


def _mixed(n, seed):
    rng = np.random.default_rng(seed)
    c = Circuit(n)
    for q in range(n):
        c.u3(*rng.uniform(0, 6, 3), q)
    for _ in range(6):
        a, b, d = (int(x) for x in rng.permutation(n)[:3])
        c.gate(Gate.Iswap(), [a, b])
        c.gate(Gate.Iswap(), [b, d], [a])
        c.gate(Gate.Ry(float(rng.uniform(0, 3))), [d], [b])
        c.ccx(a, b, d)
        c.gate(Gate.diag(np.exp(1j * rng.uniform(0, 6, 4)) * 1.0), [a, d], [b])
        c.cz(a, d)
        c.cp(float(rng.uniform(0, 3)), b, d)
        c.add(DiagonalPhase(n, [PhaseTerm((1 << a, 1 << b, 1 << d), 0.4), PhaseTerm((1 << a | 1 << d,), -0.9)]))
        c.u3(*rng.uniform(0, 6, 3), a)
    return c


def _cut_layers(n, seed, weighted):
    """MaxCut layers on a random graph: whole multiples of one angle, or not (edge k weighted 1 + weighted * k)."""
    rng = np.random.default_rng(seed)
    c = Circuit(n)
    for q in range(n):
        c.h(q)
    edges = sorted({tuple(sorted(int(x) for x in rng.permutation(n)[:2])) for _ in range(2 * n)})
    for g in (0.83, -1.9, 2.9):
        for k, (u, v) in enumerate(edges):
            w = 1.0 + weighted * k
            c.cx(u, v).rz(g * w, v).cx(u, v)
        for q in range(n):
            c.rx(0.3 + g, q)
    return c


# One register stage, one chunk, and several chunks; FP32 rounds each op to 6e-8.
@pytest.mark.parametrize("precision,tol", [(64, 1e-13), (32, 3e-6)])
@pytest.mark.parametrize("n", [4, 7, 11, 12, 13, 15])
def test_op_loop_matches_oracle(hip, oracle_lib, n, precision, tol):
    for c in (_mixed(n, n), _cut_layers(n, n, 0.0), _cut_layers(n, n, 0.1)):
        for kw in ({}, {"fuse_2q": False}, {"reg_bits": 5} if n >= 5 else {}):
            st = hip.allocate(n, precision)
            hip.run_program(st, c, **kw)
            assert max_abs(st.amplitudes(), oracle_lib.OracleSv().run(c).amplitudes()) < tol, kw
            st.free()


def test_cut_form_is_taken_and_left():
    from aleph_amd.plan_tools import HostPlan
    phases = [o for o in HostPlan(_cut_layers(14, 3, 0.0)).ops if o.type == 5]
    assert phases and all(o.cut for o in phases)
    # Weights up to some 20 units in the last place apart are different angles too.
    for weighted in (0.1, 2e-16):
        phases = [o for o in HostPlan(_cut_layers(14, 3, weighted)).ops if o.type == 5]
        assert phases and not any(o.cut for o in phases)


def test_fp32_phase_op_rounds_an_amplitude_once(hip):
    # 36 phases on three register bits (the high qubits) and one or two thread bits, in one phase op.
    from aleph_amd.plan_tools import HostPlan
    n, rng = 12, np.random.default_rng(7)
    c, i = Circuit(n), np.arange(1 << n)
    phi = np.zeros(1 << n)
    for a in range(8):
        for b in range(a, 8):
            theta = float(rng.uniform(-3, 3))
            c.gate(Gate.Phase(theta), [10], sorted({8, 9, a, b}))
            mask = 1 << 10 | 1 << 9 | 1 << 8 | 1 << a | 1 << b
            phi[(i & mask) == mask] += theta
    ops = HostPlan(c, precision=32).ops
    assert [o.type for o in ops] == [5] and ops[0].b == 36
    psi = rng.standard_normal(1 << n) + 1j * rng.standard_normal(1 << n)
    st = hip.allocate(n, 32)
    st.load(psi / np.linalg.norm(psi))
    psi = st.amplitudes()
    hip.run_program(st, c)
    on = (i >> 8) & 7 == 7
    err, want = (st.amplitudes() - psi * np.exp(1j * phi))[on], psi[on]
    # Rounding of the factor, of a product and of the sum, each by at most 2^-24 relative: sqrt(3) 2^-24 RMS.
    assert np.linalg.norm(err) < 1.04e-7 * np.linalg.norm(want)
