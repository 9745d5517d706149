"""The selectively orthogonalised FP64 step where the partial sums of the operator pass and of the update are added up by the
kernels that use them (up to four lanes) against the step with launches of their own (eight lanes): the same levels."""
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


# sectors just above the 16,384 states of full reorthogonalisation; both sides within the FP64 bar of the solver
# tests, 1e-9 of a value's magnitude (or of the lowest's), so within twice that of each other
@pytest.mark.parametrize("m,n,B", [(8, 10, 1),    # D = 19,448
                                   (8, 10, 3),    # four lanes, one of them idle: the most summed directly
                                   (9, 9, 2)])    # D = 24,310
def test_few_lanes_match_many(ctx, m, n, B):
    print(f"step sums m={m} n={n} B={B}", flush=True)
    off, sites = O.chain_neighbours(m, True)
    b = ctx.basis(m, n)
    h = b.hamiltonian(off, sites)
    J = 0.1 * 1.05 ** np.arange(8)
    many = h.lanczos(J, 1.0, k=2, prec=bhx.PREC_FP64)
    few = h.lanczos(J[:B], 1.0, k=2, prec=bhx.PREC_FP64)
    assert np.all(many.status == 0) and np.all(few.status == 0)
    want = many.evals[:B]
    assert np.all(np.abs(few.evals - want) <= 2e-9 * np.maximum(np.abs(want), np.abs(want[:, :1]))), few.evals - want
    h.close()
    b.close()
