"""Vertex following on the device (vertexFollowing.cpp:46-258 and the driver
hook driverForGraphClustering.cpp:112-132) against the oracle, through the
C ABI: labels and counts bit for bit, the folded graph in canonical form with
exact (integer) weights."""
import numpy as np
import pytest

import oracle
from grappolo_amd import driver, engine
from grappolo_amd.graph import Graph

from graphs import catalog, pendants

pytestmark = pytest.mark.gpu

GRAPHS = dict(catalog(), pendants_w=pendants(seed=5), pendants=pendants(seed=6, weighted=False),
              edgeless=Graph(np.zeros(9, np.int64), np.zeros(0, np.int64), np.zeros(0)))
NAMES = list(GRAPHS)


def _expected(g):
    C, n = oracle.vertex_following(g)
    Cr, k = oracle.renumber(C)
    return C, n, Cr, k


def _same_graph(got, exp):
    np.testing.assert_array_equal(got.edgeListPtrs, exp.edgeListPtrs)
    np.testing.assert_array_equal(got.tails, exp.tails)
    np.testing.assert_array_equal(got.weights, exp.weights)
    assert got.numEdges == exp.numEdges


@pytest.mark.parametrize("name", NAMES)
def test_vertex_following_labels(name):
    import torch
    g = GRAPHS[name]
    C, n, _, _ = _expected(g)
    got, gn = engine.vertexFollowing(g)  # host form
    assert gn == n
    np.testing.assert_array_equal(got, C)
    dg = engine.DeviceGraph(g)
    dC = torch.empty(max(g.numVertices, 1), dtype=torch.int64, device="cuda")[:g.numVertices]
    assert engine.vertex_following_dev(dg, dC) == n
    np.testing.assert_array_equal(dC.cpu().numpy(), C)


@pytest.mark.parametrize("name", NAMES)
def test_build_vf(name):
    import torch
    g = GRAPHS[name]
    _, n, Cr, k = _expected(g)
    exp = oracle.build_vf(g, Cr, k)
    _same_graph(engine.buildNewGraphVF(g, Cr, k), exp)
    dg = engine.DeviceGraph(g)
    _same_graph(engine.coarsen_dev(dg, torch.from_numpy(Cr).cuda(), k, vf=True), exp)


@pytest.mark.parametrize("name", NAMES)
def test_prepass_equals_restated_hook(name):
    g = GRAPHS[name]
    _, n, Cr, k = _expected(g)
    dg = engine.DeviceGraph(g)
    out, gn = engine.vertex_following_prepass_dev(dg)
    assert gn == n
    if n == 0:
        assert out is dg
        return
    assert out.numVertices == k
    _same_graph(out.to_host(), oracle.build_vf(g, Cr, k))


def test_driver_with_vf_clusters_the_folded_graph(tmp_path):
    """driverForGraphClustering.cpp:112-189 with -v -c 1: the run sees the
    folded graph, exactly as the restated hook builds it."""
    g = pendants(seed=8, nv=20000)
    _, n, Cr, k = _expected(g)
    folded = oracle.build_vf(g, Cr, k)
    opts = driver.ClusteringParameters(VF=True, coloring=1, output=True, minGraphSize=1000)
    C, st, dg = driver.cluster(g, opts, inFile=str(tmp_path / "pend"))
    assert st["vertices_folded"] == n and C.shape[0] == k
    C2, st2 = engine.runMultiPhaseColoring(folded, coloring=1, minGraphSize=1000, threshold=1e-6,
                                           C_threshold=0.01)
    np.testing.assert_array_equal(C, C2)
    assert st["final_modularity"] == st2["final_modularity"]
    np.testing.assert_array_equal(driver.read_communities(tmp_path / "pend_clustInfo"), C)


def test_build_vf_with_empty_clusters():
    """Caller-chosen labels may give clusters without any entry (a valid id on
    an isolated vertex): their rows are empty, first, in the middle and last,
    and a contraction with no entries at all yields all-zero offsets."""
    import torch
    g = pendants(seed=9, nv=4000)
    _, _, Cr, k = _expected(g)
    iso = np.flatnonzero(g.degrees() == 0)
    C = Cr.copy()
    C[C >= 0] += 1  # frees id 0
    mid = k // 2 + 1
    C[C >= mid] += 1  # frees id mid; the others now lie in [1, k + 1]
    C[iso[0]], C[iso[1]], C[iso[2]] = 0, mid, k + 2
    k2 = k + 3
    exp = oracle.build_vf(g, C, k2)
    d = np.diff(exp.edgeListPtrs)
    assert d[0] == 0 and d[mid] == 0 and d[-1] == 0 and np.count_nonzero(d == 0) == 3
    _same_graph(engine.buildNewGraphVF(g, C, k2), exp)
    dg = engine.DeviceGraph(g)
    _same_graph(engine.coarsen_dev(dg, torch.from_numpy(C).cuda(), k2, vf=True), exp)
    e = Graph(np.zeros(4, np.int64), np.zeros(0, np.int64), np.zeros(0))
    out = engine.buildNewGraphVF(e, np.array([0, 1, 2], np.int64), 3)
    np.testing.assert_array_equal(out.edgeListPtrs, [0, 0, 0, 0])
    assert out.nnz == 0 and out.numEdges == 0


@pytest.mark.parametrize("hubs", [[0], [2999], [0, 15, 31, 48, 65, 129, 194, 800, 2999]])
def test_contraction_with_runs_of_keys_left_out(hubs):
    """Rows whose pairs all lie with a few others leave runs of keys out of the
    sorted pairs (15 to 17, 63 to 65, hundreds, thousands of them, at the start
    and at the end), which one thread or a wavefront fills: stars around `hubs`
    contracted with every vertex its own cluster equal the oracle's graphs,
    seeded and not."""
    nv = 3000
    rng = np.random.default_rng(len(hubs))
    leaves = np.setdiff1d(np.arange(nv), hubs)
    g = Graph.from_pairs(nv, np.stack([np.array(hubs)[rng.integers(0, len(hubs), len(leaves))], leaves], 1))
    C = np.arange(nv, dtype=np.int64)
    _same_graph(engine.buildNextLevelGraphOpt(g, C, nv), oracle.coarsen(g, C, nv))
    _same_graph(engine.buildNewGraphVF(g, C, nv), oracle.build_vf(g, C, nv))
