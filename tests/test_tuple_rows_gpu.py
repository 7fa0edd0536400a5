"""Row ids are checked on the device as the gathering kernel reads them: a bad
id anywhere in a batch fails the call with its tuple's index, leaves the
tables and the next call as they were."""

import numpy as np
import pytest

import distger
from distger import ffi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,K,dim,bf16", [(1, 1, 64, False), (5, 5, 128, True), (257, 5, 128, False), (300, 15, 64, True),
                                          (9000, 6, 256, False)])
def test_bad_row_fails_the_call(ctx, n, K, dim, bf16):
    rng = np.random.default_rng(n)
    rows = 500
    s0, s1 = (rng.normal(0, 0.1, (rows, dim)).astype(np.float32) for _ in range(2))
    ctx.sgns_tables_create(s0, s1)
    good = rng.integers(0, rows, (n, K + 2)).astype(np.uint32)
    want = ctx.tuples_forward(good, K, bf16=bf16)
    for t, j, bad in ((0, 0, rows), (n - 1, 1, rows + 7), (n // 2, K + 1, 0xFFFFFFFF)):
        print(f"[tuple-rows] n={n} K={K} dim={dim} bf16={bf16} tuple {t} id {j} = {bad}", flush=True)
        x = good.copy()
        x[t, j] = bad
        for call in (lambda: ctx.tuples_forward(x, K, bf16=bf16),
                     lambda: ctx.tuples_backward(x, K, bf16=bf16, lr=0.1, apply=True),
                     lambda: ctx.tuples_step(x, K, bf16=bf16, lr=0.1, apply=True)):
            with pytest.raises(distger.DgError) as e:
                call()
            assert e.value.code == ffi.DG_ERR_ARG and f"tuple {t}: row {bad} " in str(e.value)
        with pytest.raises(distger.DgError) as e:
            ctx.grad_rows(0, [0], dim)
        assert e.value.code == ffi.DG_ERR_STATE
        got0, got1 = ctx.sgns_tables(dim)
        assert np.array_equal(got0, s0) and np.array_equal(got1, s1)
        again = ctx.tuples_forward(good, K, bf16=bf16)
        assert np.array_equal(again[0], want[0]) and again[1] == want[1]
