"""Hubs whose neighbour clusters crowd one slice of the hash range: the slice
overflows its LDS table and is done in parts.  One sweep from singletons on the
table path, bit-identical to the oracle, with 32-bit and 64-bit sums."""
import numpy as np
import pytest

from oracle import oracle as O
from pennsylvaniagpugraphclustering_amd import graphs

pytestmark = pytest.mark.gpu


def mix32(x):
    x = x.astype(np.uint32)
    x ^= x >> np.uint32(16)
    x *= np.uint32(0x85ebca6b)
    x ^= x >> np.uint32(13)
    x *= np.uint32(0xc2b2ae35)
    x ^= x >> np.uint32(16)
    return x


@pytest.mark.parametrize("weights", [None, (1 << 27, 1 << 28)])
@pytest.mark.parametrize("degree,share", [(8193, 2), (13000, 2), (16000, 2), (30000, 4)])
def test_crowded_slice(gpu_ctx, weights, degree, share):
    from pennsylvaniagpugraphclustering_amd import clustering as C
    n = 40000 * share
    ids = np.arange(1, n)
    crowd = ids[mix32(ids) < (1 << 32) // share]  # the first slice of `share`
    assert len(crowd) >= degree
    rng = np.random.default_rng(degree)
    nb = rng.choice(crowd, degree, replace=False)
    src = np.concatenate([np.zeros(degree, np.int64), rng.integers(1, n, 50000)])
    dst = np.concatenate([nb, rng.integers(1, n, 50000)])
    w = None if weights is None else rng.integers(weights[0], weights[1] + 1, len(src))
    g = graphs.from_edges(n, src, dst, w)
    obj = "Mod" if w is None else "WMod"
    vw = g.vertex_weights(obj)
    part = np.arange(n, dtype=np.int32)
    dest = np.full(n, -1, np.int32)
    gain = np.zeros(n, np.float32)
    lam = 1.0 / float(vw.sum())
    print(f"crowded slice degree={degree} share={share} weights={weights}", flush=True)
    mv, d2, g2, nc = C.sweep(C.DeviceGraph.from_csr(g, obj), part, vw, lam, 0.75, False, dest, gain)
    rmv, rd, rg, rnc = O.sweep(g.rp, g.col, g.w, vw, part, vw, lam, 0.75, False, dest, gain)
    assert nc == rnc
    assert np.array_equal(d2.cpu().numpy(), rd)
    assert np.array_equal(g2.cpu().numpy().view(np.int32), rg.view(np.int32))
    assert np.array_equal(mv.cpu().numpy(), rmv)
