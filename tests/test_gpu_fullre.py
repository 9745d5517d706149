"""The full-reorthogonalisation step of the small sectors (one Gram-Schmidt pass over the stored vectors, a second
one where the first removed much), at the edges of its work split: one and several row chunks, the narrow and
the wide update (D B up to and over 65,536), coefficients that fit one staged block and that do not, frozen vectors
of several deflation passes, a Krylov space that ends."""
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


def sector(ctx, m, n, periodic=True):
    off, sites = O.chain_neighbours(m, periodic)
    b = ctx.basis(m, n)
    return b, b.hamiltonian(off, sites), O.hamiltonian(m, n, off, sites)


# FP64 solves: every value within the FP64 bar of the solver tests, 1e-9 of its magnitude (or of the lowest's)
@pytest.mark.parametrize("m,n,B,k", [(4, 3, 1, 2),      # D = 20: one chunk, the Krylov space ends at once
                                     (6, 6, 2, 6),      # D = 462: D B below a chunk
                                     (7, 6, 64, 4),     # D = 924, 64 lanes: 59,136 elements, narrow update
                                     (7, 7, 64, 3),     # D = 1,716, 64 lanes: 109,824 elements, wide update
                                     (7, 7, 5, 12)])    # k = 12: full reorthogonalisation with many frozen vectors
def test_levels(ctx, m, n, B, k):
    print(f"fullre levels m={m} n={n} B={B} k={k}", flush=True)
    b, h, ho = sector(ctx, m, n)
    J = 0.05 * 1.05 ** np.arange(B)
    r = h.lanczos(J, 1.0, k=k, prec=bhx.PREC_FP64)
    assert np.all(r.status == 0)
    for i in sorted({0, B // 2, B - 1}):
        want = np.linalg.eigvalsh(ho.dense(J[i], 1.0))[:k]
        assert np.all(np.abs(r.evals[i] - want) <= 1e-9 * np.maximum(np.abs(want), np.abs(want[0]))), (i, r.evals[i], want)
    h.close()
    b.close()


# products of D rounded terms: each entry of Q^T Q - 1 is at most D eps of the pass that made it orthogonal
@pytest.mark.parametrize("m,n,J,steps", [(6, 6, 0.005, 120), (8, 8, 0.3, 150), (9, 9, 0.05, 70)])
def test_basis_is_orthonormal(ctx, m, n, J, steps):
    print(f"fullre basis m={m} n={n} J={J}", flush=True)
    b, h, ho = sector(ctx, m, n)
    al, be, V = h.tridiag(J, 1.0, steps, basis=True)
    assert len(al) == steps
    assert np.abs(V @ V.T - np.eye(steps)).max() <= ho.D * 2.3e-16
    # T is the projection of H on the basis
    for t in (0, 1, steps // 2, steps - 1):
        hv = O.spmv(ho, J, 1.0, V[t].copy())
        assert abs(V[t] @ hv - al[t]) <= 1e-12 * np.abs(al).max()
        if t:
            assert abs(V[t - 1] @ hv - be[t]) <= 1e-12 * np.abs(al).max()
    h.close()
    b.close()


def test_krylov_space_ends(ctx):
    """U = 0 on a ring of four sites: few distinct levels, so that every pass exhausts its Krylov space"""
    m, n, J = 4, 14, 0.5
    b, h, ho = sector(ctx, m, n)
    one = [-2 * J * math.cos(2 * math.pi * q / m) for q in range(m)]
    want = sorted(sum(one[i] * c for i, c in enumerate((x, y, z, n - x - y - z)))
                  for x in range(n + 1) for y in range(n + 1 - x) for z in range(n + 1 - x - y))[:6]
    r = h.lanczos(J, 0.0, k=6, prec=bhx.PREC_FP64)
    assert r.status[0] == 0 and np.allclose(r.evals[0], want, rtol=0, atol=1e-9 * 2 * J * n)
    h.close()
    b.close()
