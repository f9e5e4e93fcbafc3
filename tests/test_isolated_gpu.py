"""The renumbered copy with vertices without neighbours: left out of a local
move while they are alone in their clusters, and scored like any other vertex
when the input clustering puts them with others.  Equal to the run on the
caller's order, bit for bit."""
import numpy as np
import pytest

from pennsylvaniagpugraphclustering_amd import graphs

pytestmark = pytest.mark.gpu


def sparse_graph(weights):
    """3,000 vertices, every third one isolated."""
    rng = np.random.default_rng(2)
    n = 3000
    pool = np.flatnonzero(np.arange(n) % 3)
    src, dst = rng.choice(pool, 9000), rng.choice(pool, 9000)
    w = None if weights is None else rng.integers(1, 20, len(src))
    return graphs.from_edges(n, src, dst, w)


@pytest.mark.parametrize("objective", ["Mod", "CPM", "WMod"])
@pytest.mark.parametrize("labels", ["alone", "paired", "mixed"])
@pytest.mark.parametrize("plus", [False, True])
def test_improve_with_isolated_vertices(gpu_ctx, objective, labels, plus):
    from pennsylvaniagpugraphclustering_amd import clustering as C
    g = sparse_graph((1, 20) if objective == "WMod" else None)
    n = g.n
    iso = np.flatnonzero(g.degrees() == 0)
    assert len(iso) > n // 4
    rng = np.random.default_rng(4)
    part = rng.integers(0, 200, n).astype(np.int32)
    if labels == "alone":      # isolated vertices in clusters of their own
        part[iso] = 200 + np.arange(len(iso))
    elif labels == "paired":   # two by two, away from the others
        part[iso] = 200 + np.arange(len(iso)) // 2
    part = np.unique(part, return_inverse=True)[1].astype(np.int32)
    L = int(part.max()) + 1
    dg = C.DeviceGraph.from_csr(g, objective)
    res = []
    for knob in (0, 1):
        gpu_ctx.set_knob("renumber", knob)
        try:
            st, vol = C.state_init(dg, objective, 0.2 if objective == "CPM" else 1.0)
            v, uncut, sq = C.evaluate(dg, part, L)
            vol[:L] = v
            st.uncut, st.label_count = uncut, L
            st.obj = float(uncut) - st.lambda_ * float(sq)
            print(f"improve {objective} {labels} plus={plus} renumber={knob}", flush=True)
            C.check(gpu_ctx.lib.pggc_ctx_set_seed(gpu_ctx.h, 5, 0))  # the refinement's draws
            out = C.leiden_part(dg, st, plus=plus, improve=True, input=part)
            res.append((out.cpu().numpy(), st.obj, st.uncut, st.label_count))
        finally:
            gpu_ctx.set_knob("renumber", 2)
    assert np.array_equal(res[0][0], res[1][0])
    assert res[0][1:] == res[1][1:]


@pytest.mark.parametrize("objective", ["Mod", "CPM", "WMod"])
@pytest.mark.parametrize("groups", [1, 40, 3000])
def test_constrained_pass_with_isolated_vertices(gpu_ctx, objective, groups):
    """A constrained pLouvain pass from singletons, where the isolated vertices
    are left out and the others gather 16-byte records with their constraint: in
    one group, in a few that mix isolated and other vertices, and with every
    vertex a group of its own (no move under the constraint, so the strict local
    move runs, and then the passes without the constraint)."""
    import torch
    from pennsylvaniagpugraphclustering_amd import clustering as C
    g = sparse_graph((1, 20) if objective == "WMod" else None)
    dg = C.DeviceGraph.from_csr(g, objective)
    cons = np.random.default_rng(8).permutation(g.n) % groups
    res = []
    for knob in (0, 1):
        gpu_ctx.set_knob("renumber", knob)
        try:
            st, vol = C.state_init(dg, objective, 0.2 if objective == "CPM" else 1.0)
            print(f"constrained {objective} groups={groups} renumber={knob}", flush=True)
            c = torch.from_numpy(cons.astype(np.int32)).cuda()
            out = C.louvain_part(dg, st, constrained=True, constraint=c)
            res.append((out.cpu().numpy(), st.obj, st.uncut, st.label_count))
        finally:
            gpu_ctx.set_knob("renumber", 2)
    assert np.array_equal(res[0][0], res[1][0])
    assert res[0][1:] == res[1][1:]
