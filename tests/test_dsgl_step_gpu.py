"""The DSGL kernel loads a step's output rows during the step before, unless
that step moves one of them, a sentence ends or more than eight rows are held;
the negatives' rows of a batch are moved by stores.  On a graph of 60 vertices
consecutive steps share negatives and targets all the time, so every one of
these ways is taken, in the one-wavefront order, against the FP64 restatement.

Tolerance: FP32 rows and MFMA accumulation against FP64, relative to the
largest update: 2^-24 per operation, below 2^10 operations on a row's path
that do not cancel (2^-14 = 6e-5), 1e-4 as in the other DSGL parity tests.
"""

import numpy as np
import pytest

import dgsgns_oracle
import distger
from distger import ffi

pytestmark = pytest.mark.gpu

TABLE = 100_000


@pytest.mark.parametrize("dim,K,window,workers", [(64, 1, 10, 1), (64, 5, 3, 2), (128, 5, 10, 3), (128, 6, 15, 1),
                                                 (128, 7, 10, 2), (256, 5, 10, 1), (256, 14, 15, 2)])
def test_steps_vs_fp64(dim, K, window, workers):
    print(f"[dsgl-step] dim {dim} K {K} window {window} workers {workers}", flush=True)
    edges = distger.gen_chung_lu(60, 240, 2.5, 2, 3)
    with distger.Context(0) as c:
        c.graph_from_edges(60, edges, undirected=True, cn_mode=ffi.DG_CN_COMPUTE)
        c.walk_reset()
        c.walk_round(c.default_walk_params(seed=9, max_length=40), 1, 0, 300)
        tok, off = c.corpus()
        rp, _, _ = c.graph_csr()
        counts = 2 * np.diff(rp).astype(np.uint64)
        p = c.default_sgns_params(form=ffi.DG_SGNS_DSGL_FP32, dim=dim, window=window, negative=K, table_size=TABLE,
                                  alpha=0.0025, sample=0.0, alpha_schedule=ffi.DG_ALPHA_LINEAR, seed=13,
                                  deterministic=1, exact_sigmoid=1, init_float_ops=1, workers=workers, min_count=0)
        c.sgns_init(p)
        init0, _ = c.sgns_tables(dim)
        c.sgns_train(p, corpus=ffi.DG_CORPUS_ROUND)
        s0, s1 = c.sgns_tables(dim)
        vocab = c.sgns_vocab()
    o = dgsgns_oracle.Trainer(counts, dim, table_size=TABLE, sample=0.0, float_init=True)
    o.dsgl_setup(sample=0.0, table_size=TABLE)
    o.dsgl(tok, off, window, K, 0.0025, workers, 13, exact=True)
    assert np.array_equal(vocab, o.vertex_of_rank)
    d0 = o.syn0.astype(np.float64) - init0
    e0 = np.abs((s0.astype(np.float64) - init0) - d0).max() / np.abs(d0).max()
    e1 = np.abs(s1.astype(np.float64) - o.syn1).max() / np.abs(o.syn1).max()
    print(f"[dsgl-step] relative error syn0 {e0:.3e} syn1 {e1:.3e}", flush=True)
    assert e0 < 1e-4 and e1 < 1e-4
