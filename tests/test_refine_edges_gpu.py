"""Edge passes of the refinement at the edges of their tiles: rows cut by the
2048-edge chunks and as long as one, chunks that span more rows than are summed
in LDS (runs of vertices without neighbours), and the degrees where the choice of
a neighbour changes its lanes (128, 15000).  Own-cluster weights and refined
clusters equal the oracle's, bit for bit."""
import numpy as np
import pytest

from oracle import oracle as O
from pennsylvaniagpugraphclustering_amd import graphs

pytestmark = pytest.mark.gpu

DEGREES = [1, 7, 8, 9, 31, 33, 127, 128, 129, 2046, 2047, 2048, 2049, 4097, 14999, 15000, 15001, 40000]


def edge_graph(gap, wmax):
    """Hubs of those degrees and a ring over leaves; every gap-th id is used,
    the others have no neighbours."""
    rng = np.random.default_rng(gap)
    leaves = 41000
    src = [np.arange(leaves)]
    dst = [(np.arange(leaves) + 1) % leaves]
    for k, d in enumerate(DEGREES):
        src.append(np.full(d, leaves + k))
        dst.append(rng.permutation(leaves)[:d])
    src, dst = np.concatenate(src), np.concatenate(dst)
    n = (leaves + len(DEGREES)) * gap
    ids = np.sort(rng.permutation(n)[: leaves + len(DEGREES)])
    w = None if wmax is None else rng.integers(1, wmax, src.size, endpoint=True)
    return graphs.from_edges(n, ids[src], ids[dst], w)


@pytest.mark.parametrize("wmax,wide", [(None, False), (30, False), (30, True)])
@pytest.mark.parametrize("gap", [1, 40])
def test_refine_at_tile_edges(gpu_ctx, gap, wmax, wide):
    from pennsylvaniagpugraphclustering_amd import clustering as C
    from tests.test_gpu_parity import dgraph, npy, weights_for
    g = edge_graph(gap, wmax)
    obj = "Mod" if wmax is None else "WMod"
    w = weights_for(g, obj)
    if wide:
        w = w.astype(np.int64)
        dg = C.DeviceGraph(g.rp, g.col, w, g.vertex_weights(obj))
    else:
        dg = dgraph(g, obj)
    lab = np.random.default_rng(8).integers(0, 3, g.n).astype(np.int32)
    print(f"refine gap={gap} wmax={wmax} wide={wide} n={g.n}", flush=True)
    vw = g.vertex_weights(obj)
    own = O.own_weight(g.rp, g.col, w, lab)
    assert np.array_equal(npy(C.own_weight(dg, lab)), own)
    vw = g.vertex_weights(obj)
    vol, _, _ = O.evaluate(g.rp, g.col, weights_for(g, obj), vw, lab, 3)
    lam = 1.0 / (g.nnz if w is None else int(vw.sum()))
    for uniform in ([False, True] if w is None else [False]):
        m, nc = C.coarsen_leidenR(dg, lab, vol, lam, uniform, 5)
        om, onc = O.leiden_refine(g.rp, g.col, w, vw, lab, vol, lam, uniform, 5)
        assert nc == onc and np.array_equal(npy(m), om)
