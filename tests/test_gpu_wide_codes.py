"""Products of a sector whose value table is the largest there is (code_bits = 12: 32 KB of LDS) and whose rows are long enough
for the largest row tile (32 KB more), beside the kernel's own LDS: more than 64 KB for a workgroup."""
import numpy as np
import pytest

import bhx
import oracle as O

pytestmark = pytest.mark.gpu


def test_largest_table_with_largest_tile():
    m, n, times = 7, 15, 6  # every pair of seven sites six times over: (6 w)^2 (n_i + 1) n_j up to 2,304; rows of 42
    lists = [[j for j in range(m) if j != i for _ in range(times)] for i in range(m)]
    off = np.concatenate([[0], np.cumsum([len(x) for x in lists])]).astype(np.int32)
    sites = np.array([j for x in lists for j in x], np.int32)
    ho = O.hamiltonian(m, n, off, sites)
    with bhx.Context(0) as c:
        b = c.basis(m, n)
        h = b.hamiltonian(off, sites)
        assert h.packed()[1] == 12 and np.diff(h.csr()[0]).max() == 42
        rng = np.random.default_rng(1)
        for B in (1, 2, 4):
            X = rng.standard_normal((h.D, B))
            J, U = rng.uniform(0.1, 1.0, B), rng.uniform(0.5, 2.0, B)
            for prec, tol in ((bhx.PREC_FP64, 1e-13), (bhx.PREC_MIXED, 2e-6)):
                x = X if prec == bhx.PREC_FP64 else X.astype(np.float32).astype(np.float64)
                want = np.stack([O.spmv(ho, J[i], U[i], x[:, i].copy()) for i in range(B)], axis=1)
                if not (B == 4 and prec == bhx.PREC_FP64):
                    h.set_tuned(1, prec, B, B)
                print(f"wide codes B={B} prec={prec}", flush=True)
                got = h.spmv(J, U, X, prec=prec)
                assert np.abs(got - want).max() <= tol * np.abs(want).max(), (B, prec)
        h.close()
        b.close()
