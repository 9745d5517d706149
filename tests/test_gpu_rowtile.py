"""Products of one thread per row (V = B: the row-tile engine, whose waves stage the words of 64 rows in LDS) at
the edges of its tiles: fewer rows than a wave, a last tile of one row, rows longer than the staged part (several rounds),
sectors without entries; in both precisions, in the plain product and inside a solve.  The oracle's product is the
reference, FP64 within 1e-13 and FP32-stored vectors within 2e-6 of the largest entry, as in the operator tests."""
import math

import numpy as np
import pytest

import bhx
import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = bhx.Context(0)
    yield c
    c.close()


def complete(m):
    """every site a neighbour of every other one: m (m - 1) directed bonds"""
    lists = [[j for j in range(m) if j != i] for i in range(m)]
    return np.arange(m + 1, dtype=np.int32) * (m - 1), np.array([j for x in lists for j in x], np.int32)


CASES = [("chain", 2, 5),      # D = 6: less than a wave
         ("chain", 3, 10),     # D = 66: a second tile of two rows
         ("chain", 3, 21),     # D = 253
         ("chain", 1, 4),      # D = 1, no entries
         ("chain", 10, 6),     # D = 5,005: several workgroups
         ("complete", 11, 5),  # D = 3,003, up to 50 entries a row: 64 rows do not fit 2,048 words
         ("square", 16, 4)]    # D = 3,876 on the 4 x 4 torus


@pytest.mark.parametrize("geom,m,n", CASES)
def test_rowtile_matches_oracle(ctx, geom, m, n):
    print(f"row tiles {geom} m={m} n={n}", flush=True)
    off, sites = {"chain": lambda: O.chain_neighbours(m, m > 2), "complete": lambda: complete(m),
                  "square": lambda: O.square_neighbours(4, 4, True)}[geom]()
    ho = O.hamiltonian(m, n, off, sites)
    b = ctx.basis(m, n)
    h = b.hamiltonian(off, sites)
    assert h.D == ho.D == math.comb(m + n - 1, n)
    for B in (1, 2, 4):
        rng = np.random.default_rng(B)
        X = rng.standard_normal((h.D, B))
        J, U = rng.uniform(0.1, 1.0, B), rng.uniform(0.5, 2.0, B)
        for prec, tol in ((bhx.PREC_FP64, 1e-13), (bhx.PREC_MIXED, 2e-6)):
            if prec == bhx.PREC_FP64 and B == 4:
                continue
            x = X if prec == bhx.PREC_FP64 else X.astype(np.float32).astype(np.float64)
            want = np.stack([O.spmv(ho, J[i], U[i], x[:, i].copy()) for i in range(B)], axis=1)
            h.set_tuned(1, prec, B, B)
            got = h.spmv(J, U, X, prec=prec)
            assert np.abs(got - want).max() <= tol * max(np.abs(want).max(), 1e-300), (B, prec)
            if B > 1:  # the row-lane engine's sums, bit for bit
                h.set_tuned(1, prec, B, 1)
                assert np.array_equal(h.spmv(J, U, X, prec=prec), got)
    h.close()
    b.close()


@pytest.mark.parametrize("prec,B,variant", [(bhx.PREC_FP64, 1, 1), (bhx.PREC_FP64, 2, 2), (bhx.PREC_FP64, 1, 17),
                                            (bhx.PREC_MIXED, 4, 4)])
def test_rowtile_in_a_solve(ctx, prec, B, variant):
    m, n = 11, 5
    off, sites = complete(m)
    ho = O.hamiltonian(m, n, off, sites)
    b = ctx.basis(m, n)
    h = b.hamiltonian(off, sites)
    h.set_tuned(0, prec, B, variant)
    J = 0.1 + 0.05 * np.arange(B)
    r = h.lanczos(J, 1.0, k=2, prec=prec, fullre_d=-1)
    for i in range(B):
        want = np.linalg.eigvalsh(ho.dense(J[i], 1.0))[:2]
        assert abs(r.evals[i, 0] - want[0]) <= 1e-9 * abs(want[0])
    h.close()
    b.close()
