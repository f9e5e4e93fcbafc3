"""The table kernels of the single degree classes (64 < degree <= 2048), which
levels of more than 8,192 such rows use: rows one below, at and one above every
class bound, for each value of the table knobs, unit weights, small ones and
weights whose row sums exceed 32 bits, bit-identical to the oracle."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.graphcases import many_table_rows

pytestmark = pytest.mark.gpu

DEGREES = [63, 64, 65, 66, 127, 128, 129, 255, 256, 257, 511, 512, 513, 1023, 1024, 1025, 2047, 2048, 2049, 4096, 4097]
GRAPHS = {"unit": (None, "Mod"), "w10": ((1, 10), "WMod"), "wbig": ((1 << 29, (1 << 30) - 1), "WMod")}


@pytest.fixture(scope="module")
def cases():
    """Per weights: the graph, a sweep's inputs (a third of the vertices in 500
    clusters, the others in clusters of two or three) and the oracle's answers."""
    out = {}
    for name, (weights, obj) in GRAPHS.items():
        g = many_table_rows(DEGREES, weights=weights)
        assert ((g.degrees() > 64) & (g.degrees() <= 2048)).sum() > 8192
        w = g.w if obj == "WMod" else None
        vw = g.vertex_weights(obj)
        rng = np.random.default_rng(13)
        L = 30000
        part = np.where(rng.random(g.n) < 1 / 3, rng.integers(0, 500, g.n), rng.integers(500, L, g.n)).astype(np.int32)
        part[:L] = np.arange(L)
        vol, uncut, sq = O.evaluate(g.rp, g.col, w, vw, part, L)
        dest = np.where(rng.random(g.n) < 0.1, -3, -1).astype(np.int32)
        gain = np.zeros(g.n, np.float32)
        lam = 1.0 / float(vw.sum())
        obj0 = float(uncut) - lam * float(sq)
        out[name] = (g, obj, part, vol, L, uncut, lam, obj0, dest, gain,
                     O.sweep(g.rp, g.col, w, vw, part, vol, lam, 0.75, False, dest, gain),
                     O.local_move(g.rp, g.col, w, vw, part, vol, L, uncut, lam, obj0, False))
    return out


@pytest.mark.parametrize("name", list(GRAPHS))
@pytest.mark.parametrize("threads", [64, 128, 256])
@pytest.mark.parametrize("spe", [2, 4])
def test_classes_at_their_bounds(gpu_ctx, cases, name, threads, spe):
    from pennsylvaniagpugraphclustering_amd import clustering as C
    g, obj, part, vol, L, uncut, lam, obj0, dest, gain, ref, move = cases[name]
    dg = C.DeviceGraph.from_csr(g, obj)
    print(f"table classes {name} threads={threads} slots={spe}", flush=True)
    try:
        gpu_ctx.set_knob("table_threads", threads)
        gpu_ctx.set_knob("table_slots_per_edge", spe)
        mv, d2, g2, nc = C.sweep(dg, part, vol, lam, 0.75, False, dest, gain)
        st, volt = C.make_state(vol, L, uncut, lam, obj0, cap=g.n)
        out = C.local_move(dg, part, st, False)
    finally:
        gpu_ctx.set_knob("table_threads", 64)
        gpu_ctx.set_knob("table_slots_per_edge", 2)
    rmv, rd, rg, rnc = ref
    assert nc == rnc
    assert np.array_equal(d2.cpu().numpy(), rd)
    assert np.array_equal(g2.cpu().numpy().view(np.int32), rg.view(np.int32))
    assert np.array_equal(mv.cpu().numpy(), rmv)
    rpart, rv, rL, ru, ro = move
    assert np.array_equal(out.cpu().numpy(), rpart)
    assert st.label_count == rL and st.uncut == ru and st.obj == ro
