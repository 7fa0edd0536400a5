"""A tuple call with a row id out of range is refused: the id is found by the
kernel that gathers the rows, and nothing of the call reaches the caller's
buffers, the tables or the gradients.  Sizes: the ways the logits take to the
host (the context's pinned memory, a plain copy, and after enough good calls the
ring), the bad id first, in the middle and last, as center, context and negative."""

import ctypes

import numpy as np
import pytest

import distger
from distger import ffi

pytestmark = pytest.mark.gpu

ROWS, DIM, K = 1000, 128, 5


@pytest.mark.parametrize("n,where,good_calls", [(8, 0, 0), (20000, 7 * 1000 + 1, 0),
                                                (200000, 7 * 200000 - 1, 0), (200000, 7 * 200000 - 1, 9)])
@pytest.mark.parametrize("bf16", [0, 1])
def test_refused_call_writes_nothing(n, where, good_calls, bf16):
    print(f"[tuple-refused] n {n} id {where} after {good_calls} bf16 {bf16}", flush=True)
    r = np.random.default_rng(n)
    tables = [r.standard_normal((ROWS, DIM), dtype=np.float32) for _ in range(2)]
    good = r.integers(0, ROWS, (n, K + 2), dtype=np.uint32)
    bad = good.copy()
    bad.reshape(-1)[where] = ROWS
    vp = ctypes.c_void_p
    with distger.Context(0) as c:
        c.sgns_tables_create(*tables)
        logits = np.full((n, K + 1), 7.0, np.float32)
        loss = ctypes.c_double(7.0)

        def call(step, t):
            if step:
                return c.L.dg_sgns_tuples_step(c.h, t.ctypes.data_as(vp), n, K, bf16, ctypes.c_float(0.01), 1,
                                               logits.ctypes.data_as(vp), ctypes.byref(loss))
            return c.L.dg_sgns_tuples_forward(c.h, t.ctypes.data_as(vp), n, K, bf16, logits.ctypes.data_as(vp),
                                              ctypes.byref(loss))

        for _ in range(good_calls):
            assert call(0, good) == ffi.DG_OK
        logits[:], loss.value = 7.0, 7.0
        for step in (0, 1):
            assert call(step, bad) == ffi.DG_ERR_ARG
            assert (logits == 7.0).all() and loss.value == 7.0
            with pytest.raises(distger.DgError):
                c.grad_rows(0, good[:1, 1], DIM)
        for have, was in zip(c.sgns_tables(DIM), tables):
            assert np.array_equal(have, was)
        # the same call with ids in range is not held back
        for step in (0, 1):
            assert call(step, good) == ffi.DG_OK
            assert not (logits == 7.0).any() and loss.value != 7.0
        assert not np.array_equal(c.sgns_tables(DIM)[0], tables[0])
