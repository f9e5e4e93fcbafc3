"""Dense levels beyond the direct sweeps' size, whose movers meet each vertex by
dozens of edges (the neighbours' destinations are tested before they are reset):
clusterings and run counters equal the oracle's."""
import numpy as np
import pytest

from oracle import oracle as O
from pennsylvaniagpugraphclustering_amd import graphs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wmax,wide", [(None, False), (9, False), (9, True)])
def test_dense_blocks_match_oracle(gpu_ctx, wmax, wide):
    from pennsylvaniagpugraphclustering_amd import clustering as C
    rng = np.random.default_rng(1)
    n, block, m = 20000, 400, 2400000
    src = rng.integers(0, n, m)
    near = rng.random(m) < 0.45
    dst = np.where(near, src // block * block + rng.integers(0, block, m), rng.integers(0, n, m))
    w = None if wmax is None else rng.integers(1, wmax, m, endpoint=True)
    g = graphs.from_edges(n, src, dst, w)
    assert g.nnz > 1 << 22
    obj = "Mod" if wmax is None else "WMod"
    vw = g.vertex_weights(obj)
    dg = C.DeviceGraph(g.rp, g.col, g.w.astype(np.int64), vw) if wide else C.DeviceGraph.from_csr(g, obj)
    print(f"dense blocks nnz={g.nnz} wmax={wmax} wide={wide}", flush=True)
    q, p, info = C.cluster(dg, "louvain", obj, 1.0, 0, seed=0)
    oq, op, oi = O.cluster(g.rp, g.col, g.w, vw, obj, 1.0, "louvain", 0, seed=0)
    assert q == oq and np.array_equal(p.cpu().numpy(), op)
    for key in ["labels", "uncut", "levels", "sweeps", "moves"]:
        assert info[key] == oi[key], key
