"""A backward with a bad id that also finds no memory for its gradients, and the
call after it: the failed check must not hold the next update back.  The device
is filled with another library's buffers first, down to less than the gradient
rows of the call need and more than the rest of it does."""

import numpy as np
import pytest
import torch

import distger

pytestmark = pytest.mark.gpu

ROWS, DIM, K, N = 1000, 256, 15, 1 << 18
MB = 1 << 20
GRAD = N * (K + 2) * DIM * 4            # the gradient rows: 4.5 GB
REST = N * (DIM * 4 + (K + 2) * 5 * 4)  # staged rows, tuples, sort pairs: 0.4 GB, and some more
LEFT = 2048 * MB


def test_update_after_a_call_without_room():
    assert REST + 512 * MB < LEFT < GRAD - 512 * MB
    r = np.random.default_rng(5)
    good = r.integers(0, ROWS, (N, K + 2), dtype=np.uint32)
    bad = good.copy()
    bad[3, 0] = ROWS
    small = good[:64]
    tables = [0.1 * r.standard_normal((ROWS, DIM), dtype=np.float32) for _ in range(2)]
    with distger.Context(0) as c:
        c.sgns_tables_create(*tables)
        held = []
        try:
            for size in (8192 * MB, 512 * MB, 64 * MB):
                while torch.cuda.mem_get_info()[0] > LEFT + size:
                    held.append(torch.empty(size, dtype=torch.uint8, device="cuda"))
            print(f"[tuple-no-room] {torch.cuda.mem_get_info()[0] // MB} MB left", flush=True)
            with pytest.raises(distger.DgError) as e:
                c.tuples_backward(bad, K, lr=0.05, apply=True)
            assert e.value.code == -3  # DG_ERR_NOMEM
        finally:
            held.clear()
            torch.cuda.empty_cache()
        c.tuples_step(small, K, lr=0.05, apply=True)
        after = c.sgns_tables(DIM)
    for have, was, rows in zip(after, tables, (small[:, 1], small[:, 0])):
        moved = np.abs(have - was).max(axis=1) > 0
        assert moved[rows].all()
