"""The single-particle density matrix at its limits: amplitudes that overflow or are infinite reach the entries whose sums they
are in and no other; a budget with room for one vector beside the sector."""
import numpy as np
import pytest

import bhx
import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n", [(6, 5), (17, 3), (5, 16)])
@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, 1e200])
def test_spdm_infinite_amplitude(m, n, value):
    """all bosons on site 0 with an infinite amplitude: no pair of other sites has a term with it"""
    print(f"spdm m={m} n={n} amplitude {value}", flush=True)
    st, _, _ = O.basis(m, n)
    phi = np.random.default_rng(n).uniform(0.1, 1.0, len(st))
    phi[np.flatnonzero(st[:, 0] == n)[0]] = value
    with np.errstate(all="ignore"):
        want = O.spdm(st, phi)
    with bhx.Context(0) as c:
        b = c.basis(m, n)
        assert np.array_equal(b.states(), st)
        got = b.spdm(phi)
        b.close()
    fin = np.isfinite(want)
    assert np.count_nonzero(fin) >= (m - 1) * (m - 2)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(got[np.isinf(want)], want[np.isinf(want)])
    small = fin & (np.abs(want) < 1e100)  # sums without the large amplitude
    assert np.abs(got[small] - want[small]).max() <= len(st) * 2.3e-16 * np.abs(want[small]).max()


def test_spdm_with_room_for_one_vector():
    """D = 352,716 in the default order: 3.6 MB for the vector and the partial sums fit, a second vector does not"""
    m, n = 11, 11
    off, sites = O.chain_neighbours(m, True)
    st, _, _ = O.basis(m, n)
    phi = np.random.default_rng(2).uniform(0.0, 1.0, len(st))
    phi /= np.linalg.norm(phi)
    with bhx.Context(0) as c:
        b = c.basis(m, n)
        h = b.hamiltonian(off, sites)
        used = c.memory()[0]
        want = b.spdm(phi)
        h.close()
        b.close()
    ref = O.spdm(st, phi)
    assert np.abs(want - ref).max() <= len(st) * 2.3e-16 * n
    with bhx.Context(0, hbm_budget=used + 4_900_000) as c:
        b = c.basis(m, n)
        h = b.hamiltonian(off, sites)
        assert np.array_equal(b.spdm(phi), want)
        h.close()
        b.close()
