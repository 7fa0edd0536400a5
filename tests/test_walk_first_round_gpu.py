"""The first round of a context, whose buffers are not there yet: how often it is
walked, and that the walks are the oracle's whichever way it gets its room.
Walks of the reference's parameters fit a lane's share of the LDS.  Longer ones
need spill space, which is there from the start where min_length or the
threshold says so (then only a token buffer that turns out too small is a second
walk), and is fetched by a second walk where neither does."""

import numpy as np
import pytest

import dgoracle
import distger
from distger import ffi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kw,walks,longer", [
    (dict(), 1, False),                                  # the reference's: 22 vertices
    (dict(mu=0.9, length_limit=4096), 2, True),          # low threshold: once more for the tokens
    (dict(min_length=23, max_length=25), 2, True),       # every walk past 24 vertices
    (dict(mu=0.9, max_length=24), 1, False),             # none past them
    (dict(mu=0.96), None, True),                         # a few, which nothing says beforehand
])
def test_first_round(c1_edges, kw, walks, longer):
    v = 10000
    with distger.Context(0) as c:
        c.graph_from_edges(v, c1_edges, undirected=True, cn_mode=ffi.DG_CN_COMPUTE)
        p = c.default_walk_params(seed=12, **kw)
        g = dgoracle.OracleGraph.from_csr(*c.graph_csr())
        c.walk_reset()
        for rnd, n in ((1, 5 * v), (2, v)):
            c.timing_reset()
            c.walk_round(p, rnd, 0, n)
            launches = c.timing("walk")[0]
            print(f"[walk-first] {kw} round {rnd}: walked {launches} times", flush=True)
            tok, off = g.walk_round(g.cfg(p.seed, p.min_length, p.max_length, p.mu), rnd, 0, n, threads=8,
                                    tok_cap=n * 4096 // 8)
            dtok, doff = c.corpus()
            assert np.array_equal(doff, off) and np.array_equal(dtok, tok)
            if rnd == 2:
                assert launches == 1
                break
            assert (np.diff(off).max() > 24) == longer
            if walks is None:
                assert launches > 1
            else:
                assert launches <= walks
