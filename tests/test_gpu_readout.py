"""Readout in one read of the state: marginals by split index bits and shots by sub-blocks, with the validity check
on the same read, against plain numpy."""

import numpy as np
import pytest

from aleph_amd.backend import InvalidState
from aleph_amd.backend import HipSvBackend
from aleph_amd.circuit import PauliString

pytestmark = pytest.mark.gpu


def _state(hip, n, precision, seed):
    rng = np.random.default_rng(seed)
    psi = rng.standard_normal(1 << n) + 1j * rng.standard_normal(1 << n)
    psi[rng.random(1 << n) < 0.3] = 0.0
    psi[0] = 1.0
    st = hip.allocate(n, precision)
    st.load(psi / np.linalg.norm(psi))
    return st, np.abs(st.amplitudes()) ** 2


# Fewer amplitudes than threads, one workgroup, both sides of the thread bits (8), every qubit asked for, and more
# than 12 qubits above the thread bits (the wide kernel).
@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("n,qubits", [(1, [0]), (5, [4, 0]), (8, [7, 2, 3]), (9, [8]), (12, list(range(11, -1, -1))),
                                      (20, [0, 19, 8, 7, 13]), (20, [9, 10, 11]), (21, list(range(8, 21))),
                                      (21, list(range(21)))])
def test_marginal_matches_numpy(hip, n, qubits, precision):
    st, p = _state(hip, n, precision, n)
    i = np.arange(1 << n)
    bins = sum(((i >> q) & 1) << j for j, q in enumerate(qubits))
    want = np.bincount(bins, weights=p, minlength=1 << len(qubits))
    # FP64 sums of the state's own probabilities: a few hundred roundings at most.
    assert np.max(np.abs(hip.probabilities(st, qubits) - want)) < 1e-14


# One block, a partial block, many blocks; 64 shots on a boundary grid and random ones.
@pytest.mark.parametrize("n", [1, 6, 11, 12, 13, 18, 21])
def test_shots_match_the_cumulative_distribution(hip, n):
    st, p = _state(hip, n, 64, n)
    u = np.concatenate([np.random.default_rng(n).random(500), [0.0, 1.0 - 2.0**-53]])
    got = hip.sample(st, u.size, u).astype(np.int64)
    cum = np.cumsum(p)
    assert np.all(p[got] > 0.0)
    # The drawn index is where the running sum passes u (to the rounding of 2^n additions).
    slack = 1e-15 * (n + 10)
    t = u * cum[-1]
    assert np.all(cum[got] > t - slack) and np.all(cum[got] - p[got] <= t + slack)


def test_invalid_state_leaves_the_generator_alone(hip):
    a, b = HipSvBackend(seed=9), HipSvBackend(seed=9)
    sa, sb = a.allocate(6), b.allocate(6)
    sa.load(np.full(64, 0.2))
    with pytest.raises(InvalidState):
        a.sample(sa, 5)
    with pytest.raises(InvalidState):
        a.probabilities(sa, [0])
    for st in (sa, sb):
        st.load(np.full(64, 0.125))
    assert np.array_equal(a.sample(sa, 20), b.sample(sb, 20))


def test_shots_of_a_state_at_the_norm_budget(hip):
    # Norms within a few roundings of the budget's edge, where the sampler's own sum and the validity check's
    # compensated one fall on different sides (all but the first eighth of the state adds 0.55 units in the last
    # place of the norm an eighth, which a plain sum rounds up): what is accepted gives shots of the state and
    # moves the generator on, what is refused leaves it alone.
    n = 21
    part = 1 << (n - 3)
    psi = np.full(1 << n, np.sqrt(0.55 * 2.0**-52 / part))
    psi[:part] = 1.0 + 0.1 * np.random.default_rng(2).standard_normal(part)
    psi[:part] *= np.sqrt(0.75) / np.linalg.norm(psi[:part])
    psi[5] = 0.0
    psi[5] = np.sqrt(1.0 + 1e-10 * 2.0 ** (0.5 * n) - float(np.sum(psi.astype(np.longdouble) ** 2)))
    unit = psi / np.linalg.norm(psi)

    def fresh(v):
        b = HipSvBackend(seed=77)
        st = b.allocate(n, 64)
        st.load(v)
        return b, st

    b, st = fresh(unit)
    want = [b.sample(st, 8), b.sample(st, 8)]
    refused = accepted = 0
    for step in range(-14, 15):
        v = psi.copy()
        v[5] += step * np.spacing(psi[5])     # half a unit in the last place of the norm
        b, st = fresh(v)
        try:
            got = [b.sample(st, 8), b.sample(st, 8)]
            accepted += 1
            assert np.array_equal(got, want)
        except InvalidState:
            refused += 1
            st.load(unit)
            assert np.array_equal(b.sample(st, 8), want[0])
    assert refused and accepted


def test_readouts_accept_what_the_compensated_norm_accepts(hip):
    # Norms around the budget's edge, in states whose plain sums round up (one amplitude in 16 holds the mass, the
    # others 0.55 units in the last place of its probability each): marginals, energies and shots are given exactly
    # when the compensated norm is within the budget.
    n, budget = 22, 1e-10 * 2.0**11
    psi = np.full(1 << n, np.sqrt(0.55 * 2.0**-70))
    psi[((np.arange(1 << n) >> 8) & 15) == 0] = 2.0**-9
    psi[0] = 0.0
    psi[0] = np.sqrt(1.0 + budget - float(np.sum(psi.astype(np.longdouble) ** 2)))
    st = hip.allocate(n, 64)
    z, x = PauliString.new(1.0, [(0, "Z")]), PauliString.new(1.0, [(12, "X")])
    calls = [lambda: hip.probabilities(st, [0]), lambda: hip.probabilities(st, [20, 21]),
             lambda: hip.expectation_pauli_sum(st, [z]), lambda: hip.expectation_pauli_sum(st, [z, x]),
             lambda: hip.sample(st, 4, [0.1, 0.4, 0.7, 0.9])]
    seen = set()
    scale = psi[0]
    for step in range(-20, 21):
        psi[0] = scale + step * 2.0**-53 / (2.0 * scale)
        st.load(psi)
        accept = abs(hip.norm_sqr(st) - 1.0) <= budget
        for call in calls:
            try:
                call()
                assert accept
            except InvalidState:
                assert not accept
        seen.add(accept)
    assert seen == {True, False}


# One workgroup (up to 11 qubits), the first size of several, and every position of the measured bit relative to
# the pairs' order; forced outcomes use no draw, a refused state is left as it was.
@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("n,qubit", [(1, 0), (4, 3), (11, 0), (11, 10), (12, 0), (12, 11), (17, 8), (18, 17)])
def test_measure_collapses_like_numpy(hip, n, qubit, precision):
    st, p = _state(hip, n, precision, n)
    psi = st.amplitudes()
    one = ((np.arange(1 << n) >> qubit) & 1).astype(bool)
    p1 = float(np.sum(p[one]))
    # FP64: two roundings of the product; FP32: the scaled amplitude is rounded once more.
    tol = 4e-16 if precision == 64 else 1.2e-7
    for u, bit in ((p1 * 0.5, True), (p1 + 0.5 * (1 - p1), False)):
        st.load(psi)
        assert hip.measure_with_uniform(st, qubit, u) == (bit, True)
        want = np.where(one == bit, psi, 0) / np.sqrt(p1 if bit else 1.0 - p1)
        got = st.amplitudes()
        assert np.max(np.abs(got - want)) <= tol * max(1.0, np.max(np.abs(want))) + 1e-14 * np.max(np.abs(want))
        assert hip.measure_with_uniform(st, qubit, 0.3) == (bit, False)
    bad = psi.copy()
    bad[-1] = np.inf
    st.load(bad)
    with pytest.raises(InvalidState):
        hip.measure_with_uniform(st, qubit, 0.5)
    assert np.array_equal(st.amplitudes()[:-1], psi[:-1])


# The first size whose collapse is a launch of its own.
@pytest.mark.parametrize("precision", [64, 32])
def test_measure_collapses_a_large_state(hip, precision):
    n = 25
    v = np.random.default_rng(3).standard_normal(1 << n)
    st = hip.allocate(n, precision)
    st.load(v / np.linalg.norm(v))
    psi = st.amplitudes()
    tol = 4e-16 if precision == 64 else 1.2e-7
    for qubit, bit in ((0, True), (9, False), (n - 1, True)):
        half = np.abs(psi.reshape(-1, 2, 1 << qubit)) ** 2
        p1 = float(np.sum(half[:, 1]))
        st.load(psi)
        assert hip.measure_with_uniform(st, qubit, 0.5 * p1 if bit else 0.5 * (1 + p1)) == (bit, True)
        got = st.amplitudes().reshape(-1, 2, 1 << qubit)
        want = psi.reshape(-1, 2, 1 << qubit)[:, int(bit)] / np.sqrt(p1 if bit else 1.0 - p1)
        assert not np.any(got[:, 1 - int(bit)])
        # As above: two roundings of the product, and the sum behind p1.
        assert np.max(np.abs(got[:, int(bit)] - want)) <= (tol + 1e-14) * np.max(np.abs(want))
    psi[-1] = np.inf
    st.load(psi)
    with pytest.raises(InvalidState):
        hip.measure_with_uniform(st, 3, 0.5)
    assert np.array_equal(st.amplitudes()[:-1], psi[:-1])


def test_unused_and_refused_draws_stay_in_the_generator(hip):
    a, b = HipSvBackend(seed=31), HipSvBackend(seed=31)
    sa, sb = a.allocate(5), b.allocate(5)
    assert a.measure(sa, 2) is False                   # forced: |0...0>
    sa.load(np.full(32, 1.0))
    with pytest.raises(InvalidState):
        a.measure(sa, 2)
    for st in (sa, sb):
        st.load(np.full(32, 32.0**-0.5))
    assert [a.measure(sa, q) for q in range(5)] == [b.measure(sb, q) for q in range(5)]
