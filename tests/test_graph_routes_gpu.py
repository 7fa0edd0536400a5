"""Which build a graph takes follows its entries and vertices together: the
host's below 32,768, the device's from there.  Both sides of the line, and the device build at the edges
of its sort's tiles (4,096 entries) and digits (8 bits of the source) above it,
against the oracle: the order of every row, the counts and the refusal of a bad
edge."""

import numpy as np
import pytest

import dgoracle
import distger
from distger import ffi
from test_graph_build_gpu import _random_edges

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("v,e,simple,undirected,mode", [
    (300, 16233, False, True, ffi.DG_CN_COMPUTE),     # 32,466 entries and 300 vertices
    (300, 16234, False, True, ffi.DG_CN_COMPUTE),     # 32,468
    (32767, 1, True, False, ffi.DG_CN_COMPUTE),
    (1, 32767, False, False, ffi.DG_CN_FROM_DATA),
    (2, 32765, False, False, ffi.DG_CN_COMPUTE),
    (255, 32769, False, False, ffi.DG_CN_FROM_DATA),
    (256, 36863, False, False, ffi.DG_CN_COMPUTE),
    (257, 36865, False, False, ffi.DG_CN_COMPUTE_WEIGHTED),
    (4096, 18432, False, True, ffi.DG_CN_FROM_DATA),  # 36,864
    (65536, 40000, True, True, ffi.DG_CN_COMPUTE_WEIGHTED),
    (65537, 40961, False, False, ffi.DG_CN_COMPUTE),
])
def test_both_builds_match_oracle(v, e, simple, undirected, mode):
    print(f"[graph-routes] V={v} E={e} simple={simple} undirected={undirected} mode={mode}", flush=True)
    edges = _random_edges(v, e, v + e, simple)
    with distger.Context(0) as c:
        c.graph_from_edges(v, edges, undirected=undirected, cn_mode=mode)
        g = dgoracle.OracleGraph(v, edges, undirected=undirected, cn="data" if mode == ffi.DG_CN_FROM_DATA else None)
        rp, nbr, cn = c.graph_csr()
        assert np.array_equal(rp, g.row_ptr)
        assert np.array_equal(nbr, g.nbr[: g.m])
        assert np.array_equal(cn, g.cn[: g.m])
        bad = edges.copy()
        bad["src"][len(bad) - 1] = v
        with pytest.raises(distger.DgError) as err:
            c.graph_from_edges(v, bad, undirected=undirected, cn_mode=mode)
        assert err.value.code == ffi.DG_ERR_ARG and f"edge {len(bad) - 1} " in str(err.value)
        assert np.array_equal(c.graph_csr()[1], nbr)
