"""The whole-GPU persistent colored iteration (engine/wide.hip): graphs above
15,360 vertices, and smaller ones with large color classes, sweep every color
step of an iteration in one launch, with light, mid, heavy and giant vertices as
work items of wavefronts and workgroups.  Phases of few, light and large classes
take launches per color instead.  Checked against the oracle's restatement of
the colored sweep (Coloring/parallelLouvainWithColoring.cpp:154-218) and
multi-phase driver (Coloring/runMultiPhaseColoring.cpp:51-238): bit-identical
on unit weights, at least 99.9 % of the moves of an iteration on FP64 weights."""
import hashlib
import json
import os
import subprocess
import sys

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "wide_rmat19.json")
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _sha(*arrays):
    h = hashlib.sha256()
    for a in arrays:
        h.update(np.ascontiguousarray(a).tobytes())
    return h.hexdigest()


def test_rmat19_run_equals_oracle():
    """RMAT scale 19 (hubs of up to ~2e4 entries: giants split over
    workgroups, heavy vertices in LDS tables, mid and light vertices per
    wavefront): labels, final modularity and iterations per phase equal the
    oracle's (golden/wide_rmat19.json, written by make_wide_fixture.py); the
    first phase ran on the whole-GPU sweep."""
    import torch
    from grappolo_amd import engine
    from grappolo_amd.graph import gen_rmat
    with open(GOLDEN) as f:
        gold = json.load(f)
    g = gen_rmat(19, seed=3)
    assert _sha(g.edgeListPtrs, g.tails, g.weights) == gold["graph_sha256"]
    dg = engine.DeviceGraph(g, "cuda")
    C = torch.empty(g.numVertices, dtype=torch.int64, device="cuda")
    engine.profile_reset()
    engine.profile_enable(True)
    try:
        st = engine.run_colored_dev(dg, C, minGraphSize=1000, threshold=1e-9, C_threshold=1e-6)
    finally:
        engine.profile_enable(False)
    prof = engine.profile_read()
    assert prof["sweep_wide_iteration"][2] == gold["phase_iters"][0]
    assert _sha(C.cpu().numpy()) == gold["labels_sha256"]
    assert st["final_modularity"] == gold["final_modularity"]
    assert st["per_phase"]["phase_iters"].tolist() == gold["phase_iters"]
    assert st["moves"] > 0


@pytest.mark.parametrize("weighted", [False, True])
def test_one_iteration_agrees_with_oracle(weighted):
    """One colored iteration from singletons with the same coloring: every
    move equal to the oracle's on unit weights, at least 99.9 % on FP64
    weights U[0.5, 2] (per-community sums of vertices above 64 entries are
    formed in another order), and the modularity within 1e-12 relative of
    the oracle's on the engine's own labels."""
    import torch
    from grappolo_amd import engine
    from grappolo_amd.graph import gen_lfr
    g = gen_lfr(300000, seed=21, wlo=0.5 if weighted else 1.0, whi=2.0 if weighted else 1.0)
    dg = engine.DeviceGraph(g, "cuda")
    colors = torch.empty(g.numVertices, dtype=torch.int32, device="cuda")
    mc, _ = engine.color_dev(dg, colors)
    C = torch.full((g.numVertices,), -1, dtype=torch.int64, device="cuda")
    engine.profile_reset()
    engine.profile_enable(True)
    try:
        q, it = engine.colored_phase_dev(dg, C, colors, mc + 1, -1.0, 1e9)
    finally:
        engine.profile_enable(False)
    assert engine.profile_read()["sweep_wide_iteration"][2] == 1
    assert it == 1
    qo, Co, ito, _ = oracle.louvain_colored(g, colors.cpu().numpy(), mc + 1, -1.0, 1e9, frozen=True)
    assert ito == 1
    got = C.cpu().numpy()
    agree = np.mean(got == Co)
    if weighted:
        assert agree >= 0.999, agree
        assert abs(q - qo) <= 1e-6
    else:
        assert agree == 1.0
        assert q == qo
    qg = oracle.modularity(g, got)
    assert abs(engine.modularity_dev(dg, C) - qg) <= 1e-12 * abs(qg)


@pytest.mark.parametrize("valid", [True, False])
@pytest.mark.parametrize("nv", [15360, 15361, 20000])
def test_phase_on_both_sides_of_the_dense_limit(nv, valid):
    """A whole colored phase at the vertex count where the whole-GPU sweep
    takes over from the dense persistent one (15,360), with self-loops and
    isolated vertices, a proper coloring and one whose classes hold edges:
    labels, iterations and modularity equal the oracle's frozen color steps
    (integer weights, so sums are exact in any order)."""
    from grappolo_amd import engine
    from grappolo_amd.graph import Graph, gen_planted
    core = gen_planted(nv - 50, 20, 12, 0.25, seed=nv)
    rows = np.repeat(np.arange(core.numVertices), core.degrees())
    keep = rows < core.tails
    loops = np.arange(0, core.numVertices, 11)
    pairs = np.concatenate([np.stack([rows[keep], core.tails[keep]], 1), np.stack([loops, loops], 1)])
    w = np.concatenate([np.ones(int(keep.sum())), np.full(len(loops), 2.0)])
    g = Graph.from_pairs(nv, pairs, w)
    colors, mc = oracle.color_greedy(g)
    if not valid:
        colors = (np.arange(nv) * 7 % 5).astype(np.int32)
        mc = 4
    q, C, it = engine.algoLouvainWithDistOneColoring(g, colors, mc + 1, -1.0, 1e-6)
    qo, Co, ito, _ = oracle.louvain_colored(g, colors, mc + 1, -1.0, 1e-6, frozen=True)
    assert it == ito and q == qo
    np.testing.assert_array_equal(C, Co)


@pytest.mark.parametrize("conflicts", [0, 1])
def test_phase_with_a_callers_colors(conflicts):
    """The stage entry point finds out whether the colors it is given are
    proper: then one full modularity pass serves the phase, with a single edge
    inside a class (of the hub, whose row a workgroup scans) every iteration
    takes one; labels, iterations and modularity equal the oracle's either way."""
    from grappolo_amd import engine
    from grappolo_amd.graph import Graph, gen_planted
    nv = 20000
    core = gen_planted(nv, 20, 12, 0.25, seed=1)
    rows = np.repeat(np.arange(nv), core.degrees())
    keep = (rows < core.tails) & (rows > 0)
    hub = np.stack([np.zeros(6000, np.int64), np.arange(1, 6001)], 1)
    g = Graph.from_pairs(nv, np.concatenate([hub, np.stack([rows[keep], core.tails[keep]], 1)]))
    colors, mc = oracle.color_greedy(g)
    colors = colors.astype(np.int32)
    if conflicts:  # neighbour 6000 of the hub takes the hub's color, which none of its other neighbours has
        mc += 1
        colors[[0, 6000]] = mc
    engine.profile_reset()
    engine.profile_enable(True)
    try:
        q, C, it = engine.algoLouvainWithDistOneColoring(g, colors, mc + 1, -1.0, 1e-6)
    finally:
        engine.profile_enable(False)
    assert it > 2
    assert engine.profile_read()["modularity"][2] == (it if conflicts else 1)
    qo, Co, ito, _ = oracle.louvain_colored(g, colors, mc + 1, -1.0, 1e-6, frozen=True)
    assert it == ito and q == qo
    np.testing.assert_array_equal(C, Co)


@pytest.mark.parametrize("kind,route", [("ring", "launches"), ("ring_of_257", "wide"), ("planted", "wide"),
                                        ("proper_100", "wide"), ("edges_inside_100", "dense"),
                                        ("edges_inside_128", "wide")])
def test_route_of_a_phase(kind, route):
    """Per-color launches keep the phases above the dense limit whose classes
    take a launch or two each and hold no vertex above 256 entries; the dense
    sweep keeps classes of fewer than 64 vertices, of fewer than 128 when they
    hold edges.  The profile tells the routes apart (the whole-GPU sweep takes a
    modularity pass, the dense one none); all equal the oracle's color steps."""
    from grappolo_amd import engine
    from grappolo_amd.graph import Graph, gen_planted
    if kind.startswith("ring"):
        nv = 20000
        i = np.arange(nv)
        pairs = [np.stack([i, (i + s) % nv], 1) for s in range(1, 21)]
        if kind != "ring":  # one vertex of 40 + 217 entries
            pairs.append(np.stack([np.zeros(217, np.int64), 100 + 7 * np.arange(217)], 1))
        g = Graph.from_pairs(nv, np.concatenate(pairs))
        assert g.degrees().max() == (40 if kind == "ring" else 257)
    else:
        g = gen_planted(20000 if kind == "planted" else 1600, 16, 8, 0.25, seed=2)
    nv = g.numVertices
    if kind.startswith("edges_inside"):
        classes = nv // int(kind[-3:])
        colors, mc = (np.arange(nv) * 7 % classes).astype(np.int32), classes - 1
    elif kind == "proper_100":  # greedy colors, the largest classes split
        colors, _ = oracle.color_greedy(g)
        colors = np.unique(colors * 2 + (np.arange(nv) % 2), return_inverse=True)[1].astype(np.int32)
        mc = int(colors.max())
        assert 64 <= nv / (mc + 1) < 128
    else:
        colors, mc = oracle.color_greedy(g)
    engine.profile_reset()
    engine.profile_enable(True)
    try:
        q, C, it = engine.algoLouvainWithDistOneColoring(g, colors, mc + 1, -1.0, 1e-6)
    finally:
        engine.profile_enable(False)
    prof = engine.profile_read()
    persistent, passes = prof["sweep_persistent_iteration"][2], prof["modularity"][2]
    assert (persistent, passes > 0) == {"launches": (0, True), "wide": (it, True), "dense": (it, False)}[route]
    qo, Co, ito, _ = oracle.louvain_colored(g, colors, mc + 1, -1.0, 1e-6, frozen=True)
    assert it == ito and q == qo
    np.testing.assert_array_equal(C, Co)


@pytest.mark.parametrize("stage", ["run", "phase"])
def test_degrees_at_the_item_bounds(stage):
    """Vertices whose entries sit at the bounds of the sweep's work items
    (light / mid 64, mid / heavy 512 by way of bin 7's 256, heavy / giant
    8192, one and several chunks of 4096, a table round past each) on a
    planted background: the run's labels (labels pushed in the step; the
    giants merged once few communities are left) and the stage entry point's
    (with one edge inside a class, so that labels are pushed after the step)
    equal the oracle's."""
    import torch
    from grappolo_amd import engine
    from grappolo_amd.graph import Graph, gen_planted
    degrees = [64, 65, 255, 256, 257, 511, 512, 513, 1024, 1025, 4096, 4097, 8191, 8192, 8193, 12288, 12289, 20481]
    nh, nv = len(degrees), 30000
    core = gen_planted(nv - nh, 24, 8, 0.3, seed=4)
    rows = np.repeat(np.arange(core.numVertices), core.degrees())
    keep = rows < core.tails
    pairs = [np.stack([rows[keep] + nh, core.tails[keep] + nh], 1)]
    rng = np.random.default_rng(9)
    for h, d in enumerate(degrees):
        others = nh + rng.choice(nv - nh, size=d, replace=False)
        pairs.append(np.stack([np.full(d, h), others], 1))
    g = Graph.from_pairs(nv, np.concatenate(pairs))
    assert g.degrees()[:nh].tolist() == degrees
    if stage == "run":
        dg = engine.DeviceGraph(g, "cuda")
        C = torch.empty(nv, dtype=torch.int64, device="cuda")
        st = engine.run_colored_dev(dg, C, minGraphSize=100, threshold=1e-9, C_threshold=1e-6)
        Co, so = oracle.run_colored(g, coloring="jp", frozen=True, minGraphSize=100, threshold=1e-9, C_threshold=1e-6)
        assert st["final_modularity"] == so["final_modularity"]
        np.testing.assert_array_equal(C.cpu().numpy(), Co)
    else:
        colors, mc = oracle.color_greedy(g)
        v = int(g.edgeListPtrs[nh])  # the first planted vertex takes its first neighbour's color
        colors[nh] = colors[g.tails[v]]
        q, C, it = engine.algoLouvainWithDistOneColoring(g, colors, mc + 1, -1.0, 1e-6)
        qo, Co, ito, _ = oracle.louvain_colored(g, colors, mc + 1, -1.0, 1e-6, frozen=True)
        assert it == ito and q == qo
        np.testing.assert_array_equal(C, Co)


def test_two_threads_on_two_streams():
    """Two threads of a program cluster two graphs at a time, each on a stream of
    its own: kernels with grid barriers take turns on the device, so both finish
    with the results that each has alone."""
    import threading
    import torch
    from grappolo_amd import engine
    from grappolo_amd.graph import gen_lfr
    dgs = [engine.DeviceGraph(gen_lfr(nv, seed=nv)) for nv in (200003, 150001)]
    out = [[], []]

    def work(i, runs):
        with torch.cuda.stream(torch.cuda.Stream()):
            C = torch.empty(dgs[i].numVertices, dtype=torch.int64, device="cuda")
            for _ in range(runs):
                st = engine.run_colored_dev(dgs[i], C)
                torch.cuda.current_stream().synchronize()
                out[i].append((st["final_modularity"], st["total_iterations"], C.cpu().numpy()))

    torch.cuda.synchronize()
    work(0, 1)
    work(1, 1)
    threads = [threading.Thread(target=work, args=(i, 4)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for alone, *runs in out:
        assert len(runs) == 4
        for r in runs:
            assert r[:2] == alone[:2]
            np.testing.assert_array_equal(r[2], alone[2])


_LITTLE_MEMORY = """
import numpy as np
import torch
import oracle
from grappolo_amd import engine
from grappolo_amd.graph import gen_planted
for nv, degree in ((20000, 24), (4096, 128)):
    g = gen_planted(nv, 4, degree, 0.3, seed=3)
    colors, mc = oracle.color_greedy(g)
    C = torch.empty(nv, dtype=torch.int64, device="cuda")
    q, it = engine.colored_phase_dev(engine.DeviceGraph(g), C, torch.from_numpy(colors).int().cuda(), mc + 1)
    qo, Co, ito, _ = oracle.louvain_colored(g, colors, mc + 1, -1.0, 1e-6, frozen=True)
    assert it == ito and q == qo and np.array_equal(C.cpu().numpy(), Co)
print("same", flush=True)
"""


@pytest.mark.parametrize("limit,routes", [(None, ["wide persistent sweep", "wide persistent sweep"]),
                                          (1 << 20, ["per-color launches", "persistent sweep"])])
def test_phase_without_the_memory_for_the_sweep(limit, routes):
    """A phase whose entry labels and positions do not fit the device's memory
    (blocks above `limit` bytes are refused) takes the per-color launches, a
    dense one the dense sweep, instead of failing: the oracle's labels,
    iterations and modularity either way.  In a process of its own, which reads
    the limit."""
    env = dict(os.environ, GLV_TRACE="1")
    if limit:
        env["GLV_MAX_BLOCK"] = str(limit)
    r = subprocess.run([sys.executable, "-c", _LITTLE_MEMORY], cwd=ROOT, capture_output=True, text=True, timeout=100,
                       env=env)
    assert r.returncode == 0 and r.stdout.strip().endswith("same"), r.stderr[-2000:]
    took = [line.split(": ")[-1].split(" (")[0] for line in r.stderr.splitlines() if "colored phase nv" in line]
    assert took == routes


_RUN_AND_STAGE = """
import sys
import numpy as np
import oracle
from grappolo_amd import engine
from grappolo_amd.graph import Graph, gen_planted
nv = int(sys.argv[1])
if nv < 50000:
    g = gen_planted(nv, 16, 60, 0.25, seed=2)  # bins of 33 to 64 and 65 to 256 entries
else:
    i = np.arange(nv)
    g = Graph.from_pairs(nv, np.concatenate([np.stack([i, (i + s) % nv], 1) for s in range(1, 21)]))
C, st = engine.runMultiPhaseColoring(g, minGraphSize=nv + 1)
Co, so = oracle.run_colored(g, coloring="jp", frozen=True, minGraphSize=nv + 1)
assert st["final_modularity"] == so["final_modularity"] and np.array_equal(C, Co)
colors, mc, _ = oracle.color_jp(g)
q, C, it = engine.algoLouvainWithDistOneColoring(g, colors.astype(np.int32), mc + 1, -1.0, 1e-6)
qo, Co, ito, _ = oracle.louvain_colored(g, colors, mc + 1, -1.0, 1e-6, frozen=True)
assert it == ito and q == qo and np.array_equal(C, Co)
print("same", nv / (mc + 1), flush=True)
"""


@pytest.mark.parametrize("nv,run", [(20000, "wide persistent sweep"), (30000, "wide persistent sweep"),
                                    (50000, "per-color launches")])
def test_route_of_a_run_and_of_a_callers_colors(nv, run):
    """A run's coloring is known to be proper: classes of up to 1,024 vertices, or
    of more than one and a half launches each, take the whole-GPU sweep there,
    where the stage call with the same colors takes the launches (952 and 1,400
    vertices a class, 1.7 launches; 1,500 and one launch: both take them).  All
    equal the oracle."""
    r = subprocess.run([sys.executable, "-c", _RUN_AND_STAGE, str(nv)], cwd=ROOT, capture_output=True, text=True,
                       timeout=100, env=dict(os.environ, GLV_TRACE="1"))
    assert r.returncode == 0 and r.stdout.startswith("same"), r.stderr[-2000:]
    took = [line.split(": ")[-1].split(" (")[0] for line in r.stderr.splitlines() if f"colored phase nv {nv}" in line]
    assert took == [run, "per-color launches"]


_MANY_ENTRIES = """
import hashlib
import torch
from grappolo_amd import engine
n, k = 256 * 34000, 255  # vertex v beside v - k .. v + k, colors v mod (k + 1)
step = torch.cat([torch.arange(-k, 0, device="cuda"), torch.arange(1, k + 1, device="cuda")])
tails = torch.empty(n * 2 * k, dtype=torch.int64, device="cuda")
assert tails.shape[0] > 1 << 32
for r in range(0, n, 1 << 18):
    rows = torch.arange(r, min(n, r + (1 << 18)), device="cuda")
    tails[r * 2 * k:(r + rows.shape[0]) * 2 * k] = ((rows[:, None] + step) % n).reshape(-1)
w = torch.ones(tails.shape[0], dtype=torch.float64, device="cuda")
dg = engine.DeviceGraph.from_tensors(torch.arange(n + 1, device="cuda") * (2 * k), tails, w, n * k)
torch.cuda.empty_cache()
colors = (torch.arange(n, device="cuda") % (k + 1)).int()
C = torch.empty(n, dtype=torch.int64, device="cuda")
print("built", flush=True)
q, it = engine.colored_phase_dev(dg, C, colors, k + 1, -1.0, 1e-2)
print(repr(q), it, hashlib.sha256(C.cpu().numpy().tobytes()).hexdigest(), flush=True)
"""


def test_more_entries_than_a_word_counts():
    """4.4 billion entries: positions beyond 32 bits take a byte more, and a
    phase of the whole-GPU sweep gives the labels and modularity of the
    per-color launches (unit weights).  In processes of their own, one after the
    other; needs about 180 GB of device memory."""
    import torch
    torch.cuda.empty_cache()
    if torch.cuda.mem_get_info()[0] < 220 << 30:
        pytest.skip("device memory")
    res = []
    for wide in ("1", "0"):
        r = subprocess.run([sys.executable, "-c", _MANY_ENTRIES], cwd=ROOT, capture_output=True, text=True, timeout=110,
                           env=dict(os.environ, GLV_TRACE="1", GLV_WIDE=wide))
        assert r.returncode == 0, r.stderr[-2000:]
        assert ("wide persistent sweep" in r.stderr) == (wide == "1")
        res.append(r.stdout.splitlines()[-1])
    assert res[0] == res[1]
