"""Handles released while a stream is being captured: where the capture's mode lets the calling thread free device memory, it
goes on, also for a matrix large enough (40 MB) that its block is kept for the next one of its size."""
import ctypes as C
import math
import threading

import numpy as np
import pytest

import bhx
import oracle as O

pytestmark = pytest.mark.gpu

THREAD_LOCAL, RELAXED = 1, 2


@pytest.mark.parametrize("mode,other", [(RELAXED, False), (RELAXED, True), (THREAD_LOCAL, True)])
def test_release_during_capture(mode, other):
    print(f"release during capture: mode {mode}, from another thread: {other}", flush=True)
    hip = bhx.lib()  # the HIP runtime it is linked to
    off, sites = O.chain_neighbours(12, True)
    with bhx.Context(0) as c:
        b = c.basis(12, 11, bhx.ORDER_LEX)
        base = c.memory()[0]
        h = b.hamiltonian(off, sites)
        assert c.memory()[0] - base > 32 << 20
        want = h.packed()[0]
        s, g = C.c_void_p(), C.c_void_p()
        assert hip.hipStreamCreateWithFlags(C.byref(s), C.c_uint(1)) == 0
        assert hip.hipStreamBeginCapture(s, C.c_int(mode)) == 0
        if other:
            t = threading.Thread(target=h.close)
            t.start()
            t.join()
        else:
            h.close()
        assert hip.hipStreamEndCapture(s, C.byref(g)) == 0
        assert hip.hipGraphDestroy(g) == 0 and hip.hipStreamDestroy(s) == 0
        h = b.hamiltonian(off, sites)  # in the block given back
        assert h.nnz == 24 * math.comb(21, 10) and np.array_equal(h.packed()[0], want)
        h.close()
        b.close()
