"""Results read back to pageable buffers take one of three ways by their size (up
to 64 KB, up to 4 MB, above it), and above 4 MB the ring once enough has been
copied without it.  Tables at the edges of those sizes come back whole, again
and again, into fresh buffers, and from two threads with a context each."""

import threading

import numpy as np
import pytest

import distger

pytestmark = pytest.mark.gpu

DIM = 64  # 256 bytes a row
ROWS = [1, 255, 256, 257, 16383, 16384, 16385, 20001, 69633]


def tables(rows, seed):
    r = np.random.default_rng(seed)
    return [r.standard_normal((rows, DIM), dtype=np.float32) for _ in range(2)]


@pytest.mark.parametrize("rows", ROWS)
def test_tables_come_back(rows):
    print(f"[host-reads] {rows} rows", flush=True)
    want = tables(rows, rows)
    with distger.Context(0) as c:
        c.sgns_tables_create(*want)
        for _ in range(6):
            for have, was in zip(c.sgns_tables(DIM), want):
                assert np.array_equal(have, was)


def test_two_threads():
    wrong = []

    def work(seed):
        try:
            with distger.Context(0) as c:
                for k, rows in enumerate([20001, 16384, 69633, 300, 20001, 69633]):
                    want = tables(rows, 100 * seed + k)
                    c.sgns_tables_create(*want)
                    for _ in range(4):
                        if not all(np.array_equal(a, b) for a, b in zip(c.sgns_tables(DIM), want)):
                            wrong.append((seed, rows))
        except Exception as e:
            wrong.append((seed, e))

    threads = [threading.Thread(target=work, args=(s,)) for s in (1, 2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
