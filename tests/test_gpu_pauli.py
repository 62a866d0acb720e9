"""Pauli sums (aleph_hip_expectation_sum): strings whose X masks share a read of the state, strings that fit no
shared read, and the norm check that rides on the first read, against plain numpy sums."""

import numpy as np
import pytest

from aleph_amd.backend import InvalidState
from aleph_amd.circuit import PauliString

pytestmark = pytest.mark.gpu


def _expect(psi, terms):
    x = zy = ny = 0
    for q, p in terms:
        x |= (p in "XY") << q
        zy |= (p in "YZ") << q
        ny += p == "Y"
    i = np.arange(psi.size)
    par = np.zeros(psi.size, dtype=np.int64)
    for q in range(psi.size.bit_length() - 1):
        if (zy >> q) & 1:
            par ^= (i >> q) & 1
    return float(np.real((1j ** ny) * np.sum(np.conj(psi[i ^ x]) * (1 - 2 * par) * psi)))


# Below and at the four register qubits, partial wavefronts, one chunk (12) and the first sizes of several chunks
# and sweeps; at 17 qubits the wide strings' X masks fit no chunk.
@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("n", [2, 4, 5, 9, 11, 12, 13, 17])
def test_pauli_sum_matches_numpy(hip, n, precision):
    rng = np.random.default_rng(n)
    psi = rng.standard_normal(1 << n) + 1j * rng.standard_normal(1 << n)
    st = hip.allocate(n, precision)
    st.load(psi / np.linalg.norm(psi))
    psi = st.amplitudes()
    terms = [PauliString.new(-1.0, [(q, "Z"), (q + 1, "Z")]) for q in range(n - 1)]
    terms += [PauliString.new(-0.7, [(q, "X")]) for q in range(n)]
    terms += [PauliString.new(0.3, [(q, "Y"), (n - 1 - q, "Y")]) for q in range(n // 2)]
    terms += [PauliString.new(0.2, [(q, "Y")]) for q in range(n)]
    for width in (2, 3, n):
        for _ in range(6):
            qs = rng.permutation(n)[:width]
            terms.append(PauliString.new(float(rng.normal()), [(int(q), str(rng.choice(list("XYZ")))) for q in qs]))
    terms += [PauliString.new(0.5, [(q, "X") for q in range(n)]), PauliString.identity(1.5), PauliString.new(0.0, [(0, "Z")])]
    want = [_expect(psi, t.terms) for t in terms]
    # FP64 sums of 2^n products on the state's own amplitudes: rounding of 1e-16 per unit weight.
    tol = 1e-13 * sum(abs(t.coefficient) for t in terms)
    assert abs(hip.expectation_pauli_sum(st, terms) - sum(t.coefficient * w for t, w in zip(terms, want))) < tol
    for t, w in zip(terms[::5], want[::5]):
        assert abs(hip.expectation_value(st, t) - t.coefficient * w) < 1e-13 * max(1.0, abs(t.coefficient))
    # The validity check reads the same sweep: a norm off 1 and a non-finite amplitude are still refused.
    st.load(psi * 1.1)
    with pytest.raises(InvalidState):
        hip.expectation_pauli_sum(st, terms)
    psi[-1] = np.nan
    st.load(psi)
    with pytest.raises(InvalidState, match="non-finite|invalid"):
        hip.expectation_pauli_sum(st, terms)


# Random strings whose X masks spread over many sweeps (about 20 at 14 qubits, 100 at 16): their sums meet in the
# same rows of partial sums.
@pytest.mark.parametrize("n,count,precision", [(14, 300, 64), (16, 300, 32)])
def test_strings_of_many_sweeps_add_up(hip, n, count, precision):
    rng = np.random.default_rng(n)
    psi = rng.standard_normal(1 << n) + 1j * rng.standard_normal(1 << n)
    st = hip.allocate(n, precision)
    st.load(psi / np.linalg.norm(psi))
    psi = st.amplitudes()
    terms = []
    for _ in range(count):
        qs = np.sort(rng.permutation(n)[:rng.integers(2, 9)])
        terms.append(PauliString.new(float(rng.normal()), [(int(q), str(rng.choice(list("XYZ")))) for q in qs]))
    want = sum(t.coefficient * _expect(psi, t.terms) for t in terms)
    # As above: rounding of 1e-16 per unit weight and product.
    assert abs(hip.expectation_pauli_sum(st, terms) - want) < 1e-13 * sum(abs(t.coefficient) for t in terms)


# Coefficients near the largest double: their sum is in range where each string's value is small enough.
@pytest.mark.parametrize("n", [6, 13])
def test_large_coefficients_do_not_overflow(hip, n):
    st = hip.allocate(n, 64)
    st.load(np.full(1 << n, 2.0 ** (-0.5 * n)))             # <X> = 1, <Z> = 0 on every qubit
    assert hip.expectation_pauli_sum(st, [PauliString.new(1.5e308, [(1, "X")])]) == pytest.approx(1.5e308, rel=1e-12)
    terms = [PauliString.new(1e308, [(0, "X"), (2, "X")]), PauliString.new(1.2e308, [(0, "X"), (2, "X"), (3, "Z")]),
             PauliString.new(-1.7e308, [(n - 1, "Z")]), PauliString.new(2.0, [])]
    assert hip.expectation_pauli_sum(st, terms) == pytest.approx(1e308, rel=1e-12)
