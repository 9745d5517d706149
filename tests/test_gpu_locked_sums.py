"""Solves whose steps carry many locked vectors (k = 6 above the size of full reorthogonalisation: eight, then sixteen in the later
passes), with few lanes, where the update adds up the operator pass's partial sums, and with eight, where launches of
their own do; and the row-tile operator in whole solves, every level and status.  Open chains and a complete graph, against the
oracle and the dense spectrum."""
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


def agree(got, want, prec):
    """the solver's bars: FP64 1e-9 of a value's magnitude (or of the lowest's) on every level; mixed 1e-9 on the
    lowest and 1e-5 on the others"""
    err = np.abs(got - want)
    if prec == bhx.PREC_FP64:
        assert np.all(err <= 1e-9 * np.maximum(np.abs(want), abs(want[0]))), (got, want)
    else:
        assert err[0] <= 1e-9 * abs(want[0]) and np.all(err <= 1e-5 * np.maximum(np.abs(want), 1.0)), (got, want)


@pytest.mark.parametrize("prec", [bhx.PREC_FP64, bhx.PREC_MIXED])
@pytest.mark.parametrize("m,n", [(8, 10), (9, 9)])  # D = 19,448 and 24,310
def test_many_locked_vectors(ctx, m, n, prec):
    off, sites = O.chain_neighbours(m, False)
    ho = O.hamiltonian(m, n, off, sites)
    b = ctx.basis(m, n)
    h = b.hamiltonian(off, sites)
    J = 0.2 * 1.1 ** np.arange(5)
    want = {}
    for i in (0, 1):
        rc, want[i], _, _ = O.lanczos_mult(ho, J[i], 1.0, 6)
        assert rc == 0
    for B in (1, 2, 3, 5):
        print(f"locked sums m={m} n={n} prec={prec} B={B}", flush=True)
        r = h.lanczos(J[:B], 1.0, k=6, prec=prec)
        assert np.all(r.status == 0)
        for i in range(min(B, 2)):
            agree(r.evals[i], want[i], prec)
    h.close()
    b.close()


@pytest.mark.parametrize("prec,B,variant", [(bhx.PREC_FP64, 1, 1), (bhx.PREC_FP64, 2, 2), (bhx.PREC_FP64, 1, 17), (bhx.PREC_MIXED, 1, 1),
                                            (bhx.PREC_MIXED, 2, 2), (bhx.PREC_MIXED, 4, 4)])
def test_rowtile_solve_levels(ctx, prec, B, variant):
    """eleven sites, each bonded to every other (rows of up to 50 entries, D = 3,003), selective orthogonalisation"""
    print(f"rowtile solve prec={prec} B={B} variant={variant}", flush=True)
    m, n = 11, 5
    lists = [[j for j in range(m) if j != i] for i in range(m)]
    off = np.arange(0, m * (m - 1) + 1, m - 1).astype(np.int32)
    sites = np.array(sum(lists, []), np.int32)
    ho = O.hamiltonian(m, n, off, sites)
    b = ctx.basis(m, n)
    h = b.hamiltonian(off, sites)
    h.set_tuned(0, prec, B, variant)
    J = 0.1 + 0.05 * np.arange(B)
    r = h.lanczos(J, 1.0, k=2, prec=prec, fullre_d=-1)
    assert np.all(r.status == 0)
    for i in range(B):
        agree(r.evals[i], np.linalg.eigvalsh(ho.dense(J[i], 1.0))[:2], prec)
    h.close()
    b.close()
