"""Small sectors at a server whose budget holds one of them with its engine: each is given up whole for the next, while the
pass over the small sectors goes on."""
import numpy as np
import pytest

import bhx

pytestmark = pytest.mark.gpu

SECTORS = [(8, 6), (8, 7), (8, 8), (7, 7)]  # D = 1,716, 3,432, 6,435, 1,716


def serve(ctx, budget, requests):
    with bhx.Server(ctx, lanes=1, hbm_budget=budget) as srv:
        out = [srv.wait(srv.submit("chain", n, J, 1.0, 0.0, m=m), 60.0) for m, n, J in requests]
    assert all(r is not None for r in out)
    return out


def test_idle_sectors_are_given_up_whole():
    with bhx.Context(0) as ctx:
        lo, hi = 1 << 20, 64 << 20  # the smallest budget (within 16 KB) that holds the largest sector with its engine
        assert serve(ctx, hi, [(8, 8, 0.2)])[0].status == 0
        while hi - lo > 16 << 10:
            mid = (lo + hi) // 2
            if serve(ctx, mid, [(8, 8, 0.2)])[0].status == 0:
                hi = mid
            else:
                lo = mid
        requests = [(m, n, 0.1 + 0.01 * i) for i in range(4) for m, n in (SECTORS if i % 2 == 0 else SECTORS[::-1])]
        print(f"server eviction, budget {hi}", flush=True)
        got = serve(ctx, hi, requests)
        for (m, n, J), r in zip(requests, got):
            assert r.status == 0, (m, n, J)
            b = ctx.basis(m, n, bhx.ORDER_LEX)
            h = b.hamiltonian(*bhx.lattice("chain", m=m))
            want = h.lanczos(J, 1.0, k=4, prec=bhx.PREC_FP64).evals[0]
            assert np.all(np.abs(np.array(r.evals[:4]) - want) <= 1e-9 * np.maximum(np.abs(want), abs(want[0])))
            h.close()
            b.close()
