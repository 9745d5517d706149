"""The single-particle density matrix at its limits: amplitudes that overflow or are infinite reach the entries whose sums they
are in and no other."""
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
