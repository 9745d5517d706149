"""Basis and Hamiltonian builders at the edges of their branches, bit for bit against the oracle: sectors ordered by
counting (up to 16,384 states) and by the radix sort of the truncated keys (several tiles, a last tile of few
states, 128-bit keys, many states with one truncation), rows that cross a count tile, rows copied out through LDS and
straight, long hops, every order; and scratch that the context keeps between calls of different sizes."""
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
    lists = [[j for j in range(m) if j != i] for i in range(m)]
    return np.arange(m + 1, dtype=np.int32) * (m - 1), np.array([j for x in lists for j in x], np.int32)


def relabelled(m, seed):
    """a ring whose sites are numbered at random: hops between any two sites"""
    p = np.random.default_rng(seed).permutation(m)
    lists = [None] * m
    for i in range(m):
        lists[p[i]] = sorted({int(p[(i - 1) % m]), int(p[(i + 1) % m])} - {int(p[i])})
    return np.concatenate([[0], np.cumsum([len(x) for x in lists])]).astype(np.int32), np.array([j for x in lists for j in x], np.int32)


@pytest.mark.parametrize("order", [bhx.ORDER_REFERENCE, bhx.ORDER_ASCENDING])
@pytest.mark.parametrize("m,n", [(2, 80), (3, 54), (4, 44), (4, 45), (5, 24), (6, 13), (7, 12), (22, 4), (24, 4)])
def test_order(ctx, m, n, order):
    D = math.comb(m + n - 1, n)
    print(f"order m={m} n={n} D={D} order={order}", flush=True)
    b = ctx.basis(m, n, order)
    st, _, lex = O.basis(m, n, order)
    lop, pol = b.perm()
    assert np.array_equal(lop.astype(np.int64), lex) and np.array_equal(pol[lop], np.arange(D))
    assert np.array_equal(b.states(), st)
    b.close()


@pytest.mark.parametrize("order", [bhx.ORDER_REFERENCE, bhx.ORDER_LEX])
@pytest.mark.parametrize("name,m,n", [("ring", 1, 3), ("ring", 2, 9), ("ring", 9, 5), ("ring", 7, 7), ("ring", 12, 4), ("ring", 18, 3),
                                      ("ring", 5, 18), ("complete", 11, 5), ("complete", 11, 7), ("complete", 4, 0)])
def test_hamiltonian(ctx, name, m, n, order):
    print(f"hamiltonian {name} m={m} n={n} order={order}", flush=True)
    off, sites = complete(m) if name == "complete" else (np.zeros(m + 1, np.int32), np.zeros(0, np.int32)) if m == 1 else relabelled(m, m + n)
    b = ctx.basis(m, n, order)
    h = b.hamiltonian(off, sites)
    st, _, _ = O.basis(m, n)
    ho = O.hamiltonian(m, n, off, sites if sites.size else np.zeros(1, np.int32), states=st)
    rp, col, val, diag = h.csr()
    if order == bhx.ORDER_REFERENCE:
        assert np.array_equal(rp, ho.row_ptr) and np.array_equal(col, ho.col) and np.array_equal(val, ho.val)
        assert np.array_equal(diag, ho.diag)
    else:  # the oracle's matrix with its rows and columns in lexicographic order
        _, _, lex = O.basis(m, n)
        for p in range(0, h.D, max(1, h.D // 700)):
            q = int(np.flatnonzero(lex == p)[0])
            want = sorted(zip(lex[ho.col[ho.row_ptr[q]:ho.row_ptr[q + 1]]], ho.val[ho.row_ptr[q]:ho.row_ptr[q + 1]]))
            got = list(zip(col[rp[p]:rp[p + 1]], val[rp[p]:rp[p + 1]]))
            assert [tuple(map(float, x)) for x in want] == [tuple(map(float, x)) for x in got]
            assert diag[p] == ho.diag[q]
    h.close()
    b.close()


def test_scratch_is_kept_and_given_back():
    """builds of growing and shrinking sectors in one context; a budget with no room beside the kept scratch"""
    with bhx.Context(0) as c:
        base = c.memory()[0]
        for m, n in ((6, 6), (10, 9), (5, 5), (10, 9)):
            b = c.basis(m, n)
            h = b.hamiltonian(*O.chain_neighbours(m, True))
            assert h.nnz == O.hamiltonian(m, n, *O.chain_neighbours(m, True)).nnz
            h.close()
            b.close()
        assert c.memory()[0] == base  # kept scratch is not counted as used
    off, sites = O.chain_neighbours(10, True)
    with bhx.Context(0) as c:
        b = c.basis(10, 9)
        h = b.hamiltonian(off, sites)
        all_of_it = c.memory()[0]
        h.close()
        b.close()
    with bhx.Context(0, hbm_budget=all_of_it + (1 << 17)) as c:  # no room for the matrix beside the basis' scratch
        for _ in range(2):
            b = c.basis(10, 9)
            h = b.hamiltonian(off, sites)
            assert h.D == math.comb(18, 9)
            h.close()
            b.close()


def test_spare_block_budget():
    """sectors whose matrix (34 and 44 MB) is kept as the spare block when freed: reused by the next, given up when the budget
    has no room for another beside it"""
    off, sites = O.chain_neighbours(12, True)
    with bhx.Context(0) as c:
        b = c.basis(12, 10, bhx.ORDER_LEX)
        base = c.memory()[0]
        h = b.hamiltonian(off, sites)
        one = c.memory()[0] - base
        want = h.packed()[0]
        h.close()
        assert c.memory()[0] == base
        for _ in range(2):
            h = b.hamiltonian(off, sites)
            assert np.array_equal(h.packed()[0], want)
            h.close()
        b.close()
    with bhx.Context(0, hbm_budget=base + one + (2 << 20)) as c:
        b = c.basis(12, 10, bhx.ORDER_LEX)
        h = b.hamiltonian(off, sites)
        h.close()
        s = c.basis(12, 9, bhx.ORDER_LEX)  # no room beside the spare block
        hs = s.hamiltonian(off, sites)
        assert hs.nnz == 24 * math.comb(19, 11)
        hs.close()
        s.close()
        h = b.hamiltonian(off, sites)
        assert np.array_equal(h.packed()[0], want)
        h.close()
        b.close()
