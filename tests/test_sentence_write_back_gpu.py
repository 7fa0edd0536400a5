"""The batched kernels add a sentence's input-row deltas to the table through
LDS, in columns of a pool tile's rows.  A launch of one sentence has one order
of updates, so Hogwild mode (16-row pools up to 16 distinct vertices, 32-row
ones past it) has to give the tables of the deterministic mode (32-row pools)
up to rounding.

The walk is one walk of a complete graph of n vertices: pools of fewer rows
than a tile, a full tile, and two tiles, at every width.  Tolerance against
the largest movement of the table: the two pool sizes sum the recursion's
terms in other orders, at most 2^-24 of them per operation over fewer than
100 positions x 16 operations (2^-13 in FP32); in BF16 such a difference can
flip the rounding of a staged element, 2^-8 of it, in a row of which one
position's update is a part (2^-6).
"""

import itertools

import numpy as np
import pytest

import distger
from distger import ffi

pytestmark = pytest.mark.gpu

FP32 = (ffi.DG_SGNS_BATCHED_FP32, 2.0**-13)
BF16 = (ffi.DG_SGNS_BATCHED_BF16, 2.0**-6)


@pytest.mark.parametrize("form_tol,dim", [(FP32, 64), (FP32, 128), (BF16, 64), (BF16, 128), (BF16, 256)])
@pytest.mark.parametrize("n,length", [(3, 24), (15, 60), (16, 60), (17, 90), (30, 90)])
def test_one_sentence_tables(form_tol, dim, n, length):
    form, tol = form_tol
    pairs = list(itertools.combinations(range(n), 2))
    e = np.zeros(len(pairs), dtype=ffi.EDGE_DTYPE)
    e["src"], e["dst"] = np.array(pairs, dtype=np.uint32).T
    e["data"] = 1.0
    with distger.Context(0) as c:
        c.graph_from_edges(n, e, undirected=True, cn_mode=ffi.DG_CN_COMPUTE)
        c.walk_reset()
        try:
            c.walk_round(c.default_walk_params(seed=5, min_length=length - 2, max_length=length), 1, 0, 1)
        except distger.DgError as err:  # vertices without a visit: relative entropy undefined
            assert err.code == -7
        tok, _ = c.corpus()
        print(f"[write-back] form {form} dim {dim}: {len(tok)} positions, {len(np.unique(tok))} distinct", flush=True)
        tables = []
        for det in (1, 0):
            p = c.default_sgns_params(form=form, dim=dim, window=5, negative=5, sample=0.0, min_count=0, alpha=0.025,
                                      table_size=10_000, seed=7, deterministic=det, iter=1)
            c.sgns_init(p)
            rows = len(c.sgns_vocab())
            r = np.random.default_rng(11)
            init = [r.normal(0.0, 0.2, (rows, dim)).astype(np.float32) for _ in range(2)]
            c.sgns_set_tables(*init)
            c.sgns_train(p, corpus=ffi.DG_CORPUS_ROUND)
            tables.append([a.astype(np.float64) - b for a, b in zip(c.sgns_tables(dim), init)])
        for name, a, b in zip(("syn0", "syn1"), *tables):
            scale = np.abs(a).max()
            worst = np.abs(a - b).max()
            print(f"[write-back] {name}: moved {scale:.3e}, differ {worst:.3e}", flush=True)
            assert scale > 1e-4
            assert worst <= tol * scale
