"""A DSGL step's distinct contexts fill one to four tiles of 16, and the rows of
its gradient buffer hold as many tiles as its window can (windows up to 4, 8,
12 and 15).  Walks of 40 vertices that never turn back (weights that saturate
the acceptance) on a complete graph reach every number of tiles each window
allows (checked on the host from the corpus and the window draws), with K on both sides of six, against the FP64 restatement: in the
one-wavefront order, and with one worker as a concurrent launch runs it, where
nothing but the order of a wavefront's own accesses stands between a step's
stores and the next step's loads.

Tolerance: FP32 rows and MFMA accumulation against FP64, relative to the
largest update: 2^-24 per operation, below 2^10 operations on a row's path
that do not cancel (2^-14 = 6e-5), 1e-4 as in the other DSGL parity tests.
"""

import numpy as np
import pytest

import dgoracle
import dgsgns_oracle
import distger
from distger import ffi

pytestmark = pytest.mark.gpu

V, WALKS, SEED, TABLE = 90, 100, 13, 100_000
TAG_DSGL_WIN = 0x44535749


def tiles_of(tok, off, window):
    """Tiles of 16 distinct contexts of each step of one worker over the walks."""
    walks = [tok[off[w]:off[w + 1]] for w in range(len(off) - 1)]
    left = [w for w in walks if len(w) > 1]
    cur, pos, step, tiles = [None, None], [0, 0], 0, set()
    while True:
        for s in (0, 1):
            if cur[s] is None:
                if not left:
                    return tiles
                cur[s], pos[s] = left.pop(0), 0
        half = window - int(dgoracle.philox((0, 0, step, TAG_DSGL_WIN), (SEED, 0))[0]) % window
        step += 1
        e = 0
        for s in (0, 1):
            lo, hi = max(0, pos[s] - half), pos[s] + half + 1
            e += len(set(cur[s][lo:pos[s]].tolist()) | set(cur[s][pos[s] + 1:hi].tolist()))
            pos[s] += 1
            if pos[s] == len(cur[s]):
                cur[s] = None
        tiles.add((e + 15) // 16)


@pytest.mark.parametrize("deterministic", [1, 0])
@pytest.mark.parametrize("dim,K,window,tiles", [(64, 5, 4, 1), (128, 6, 8, 2), (64, 7, 9, 3), (128, 5, 9, 3),
                                               (128, 5, 10, 3), (256, 3, 10, 3), (128, 10, 10, 3), (128, 5, 12, 3),
                                               (64, 1, 12, 3), (128, 5, 13, 4), (64, 14, 15, 4), (256, 6, 15, 4)])
def test_contexts_vs_fp64(dim, K, window, tiles, deterministic):
    print(f"[dsgl-contexts] dim {dim} K {K} window {window} deterministic {deterministic}", flush=True)
    edges = np.zeros(V * (V - 1) // 2, dtype=distger.EDGE_DTYPE)
    edges["src"], edges["dst"] = np.triu_indices(V, 1)
    edges["data"] = 1e3
    with distger.Context(0) as c:
        c.graph_from_edges(V, edges, undirected=True, cn_mode=ffi.DG_CN_COMPUTE_WEIGHTED)
        c.walk_reset()
        c.walk_round(c.default_walk_params(seed=9, min_length=39, max_length=40), 1, 0, WALKS)
        tok, off = c.corpus()
        rp, _, _ = c.graph_csr()
        counts = 2 * np.diff(rp).astype(np.uint64)
        p = c.default_sgns_params(form=ffi.DG_SGNS_DSGL_FP32, dim=dim, window=window, negative=K, table_size=TABLE,
                                  alpha=0.0025, sample=0.0, alpha_schedule=ffi.DG_ALPHA_LINEAR, seed=SEED,
                                  deterministic=deterministic, exact_sigmoid=1, init_float_ops=1, workers=1,
                                  min_count=0)
        c.sgns_init(p)
        init0, _ = c.sgns_tables(dim)
        c.sgns_train(p, corpus=ffi.DG_CORPUS_ROUND)
        s0, s1 = c.sgns_tables(dim)
        vocab = c.sgns_vocab()
    assert tiles_of(tok, off, window) >= set(range(1, tiles + 1))
    o = dgsgns_oracle.Trainer(counts, dim, table_size=TABLE, sample=0.0, float_init=True)
    o.dsgl_setup(sample=0.0, table_size=TABLE)
    o.dsgl(tok, off, window, K, 0.0025, 1, SEED, exact=True)
    assert np.array_equal(vocab, o.vertex_of_rank)
    d0 = o.syn0.astype(np.float64) - init0
    e0 = np.abs((s0.astype(np.float64) - init0) - d0).max() / np.abs(d0).max()
    e1 = np.abs(s1.astype(np.float64) - o.syn1).max() / np.abs(o.syn1).max()
    print(f"[dsgl-contexts] relative error syn0 {e0:.3e} syn1 {e1:.3e}", flush=True)
    assert e0 < 1e-4 and e1 < 1e-4
