"""The selectively orthogonalised FP64 step where the partial sums of the operator pass and of the update are added up by the
kernels that use them (few lanes) and by launches of their own (more lanes), with no, few and many locked vectors."""
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


# FP64 solves: every value within the FP64 bar of the solver tests, 1e-9 of its magnitude (or of the lowest's)
@pytest.mark.parametrize("m,n,B,k", [(6, 4, 1, 2),     # D = 126: one workgroup of each kernel
                                     (7, 6, 4, 4),     # the most lanes summed directly
                                     (7, 6, 5, 4),     # eight lanes: launches of their own
                                     (7, 7, 1, 6)])    # D = 1,716: deflation passes, eight and sixteen locked vectors
def test_levels(ctx, m, n, B, k):
    print(f"step sums m={m} n={n} B={B} k={k}", flush=True)
    off, sites = O.chain_neighbours(m, True)
    b = ctx.basis(m, n)
    h = b.hamiltonian(off, sites)
    ho = O.hamiltonian(m, n, off, sites)
    J = 0.08 * 1.1 ** np.arange(B)
    r = h.lanczos(J, 1.0, k=k, prec=bhx.PREC_FP64, fullre_d=-1)
    assert np.all(r.status == 0)
    for i in sorted({0, B // 2, B - 1}):
        want = np.linalg.eigvalsh(ho.dense(J[i], 1.0))[:k]
        assert np.all(np.abs(r.evals[i] - want) <= 1e-9 * np.maximum(np.abs(want), np.abs(want[0]))), (i, r.evals[i], want)
    h.close()
    b.close()
