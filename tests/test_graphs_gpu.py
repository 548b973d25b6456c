"""Graph workloads on the GPU ("cc", "bfs", "pagerank", "sssp" executors and gp_launch_graph) against
the numpy oracle and scipy, and preempt-then-resume of their host loops (reference
src/workloads/graphcompute.tr.cu; BLPExecutor::execute graph branch, src/executor.cpp:226-228).

Component labels, BFS levels and SSSP distances are integers with a unique answer: compared
bit-exactly.  PageRank adds fp32 residuals with atomics in arrival order, so two runs differ in the
last bits and may stop one iteration apart: compared to the linear system's solution within 0.02
(values are of order 1; the residual-push iteration leaves up to 0.001 per vertex unpushed, which
the oracle's own run turns into an error of 0.008 on this graph)."""
import ctypes as C
import threading
import time

import numpy as np
import pytest

from oracle import graphs as G

pytestmark = pytest.mark.gpu

N, DEG = 30000, 5
PR_TOL = 0.02


@pytest.fixture(scope="module")
def ex_mod(gp):
    from gpreempt_amd import executor
    return executor


@pytest.fixture(scope="module")
def graph(ex_mod, tmp_path_factory):
    base = str(tmp_path_factory.mktemp("graph") / "g")
    assert ex_mod.lib().gpx_write_synthetic_graph(base.encode(), C.c_ulonglong(N), DEG, C.c_ulonglong(7)) == 0
    indptr, indices, w = G.read_graph(base, weights=True)
    return base, indptr, indices, w


def expected(kind, graph):
    _, indptr, indices, w = graph
    if kind == "bfs":
        return "label", np.uint32, G.bfs(indptr, indices)[0]
    if kind == "cc":
        return "comp", np.uint64, G.cc(indptr, indices)[0]
    if kind == "sssp":
        return "cost", np.uint32, G.sssp(indptr, indices, w)[0]
    return "value", np.float32, G.pagerank_exact(indptr, indices)


def check(kind, got, want):
    if kind == "pagerank":
        assert np.abs(got - want).max() < PR_TOL
    else:
        assert np.array_equal(got, want)


@pytest.mark.parametrize("kind", ["bfs", "cc", "sssp", "pagerank"])
@pytest.mark.parametrize("blp", [False, True])
def test_workload_matches_oracle(gp, ex_mod, graph, kind, blp):
    ex = ex_mod.Executor(kind, blp=blp, graph_path=graph[0])
    if blp:
        ex.set_flag(gp.Flag())
    stream = gp.Stream(1)
    key, dt, want = expected(kind, graph)
    for _ in range(2):  # a second execute starts from scratch
        ex.execute(stream)
        check(kind, ex.graph_result(key, dt), want)
    info = ex.graph_info()
    assert info["vertices"] == N and info["edges"] == len(graph[2]) and info["preemptions"] == 0
    assert info["iterations"] >= 3


def test_synthetic_default_and_bad_names(gp, ex_mod):
    ex = ex_mod.Executor("bfs@n=5000,deg=4,seed=3")
    ex.execute()
    label = ex.graph_result("label", np.uint32)
    assert label[0] == 0 and (label != G.INF).sum() > 4000
    assert ex.kernel_num() == 0
    with pytest.raises(ex_mod.StatusError):
        ex.graph_result("cost", np.uint32)
    with pytest.raises(ex_mod.StatusError):
        ex_mod.Executor("bfs@n=1")
    with pytest.raises(ex_mod.StatusError):
        ex_mod.Executor("bfs", graph_path="/nonexistent/graph")


# (iteration, kernel, claim): -1 = PageRank's set-up kernel.  An injected stop is the stepwise loop's; the launches that a
# run queues are stopped in test_queued_launches_stopped_again_and_again.
INJECT = {"bfs": [(0, 0, 0), (2, 0, 900), (4, 0, 1500)],
          "cc": [(-1, 0, 5), (0, 0, 1500), (1, 0, 10), (2, 0, 1800)],
          "sssp": [(1, 0, 100), (3, 1, 60), (6, 0, 1700)],
          "pagerank": [(-1, 0, 50), (0, 0, 1000), (1, 1, 20), (5, 0, 1600)]}


@pytest.mark.parametrize("kind", ["bfs", "cc", "sssp", "pagerank"])
def test_injected_preemption_then_resume(gp, ex_mod, graph, kind):
    key, dt, want = expected(kind, graph)
    ex = ex_mod.Executor(kind, blp=True, graph_path=graph[0])
    flag = gp.Flag()
    ex.set_flag(flag)
    stream = gp.Stream(1)
    total = 0
    for it, kernel, claim in INJECT[kind]:
        flag.set(0)
        ex.graph_inject_preempt(it, kernel, claim)
        ex.execute(stream)
        info = ex.graph_info()
        assert flag.get() == 0  # raised by the kernel, lowered by the loop after the stop was seen
        # (a flag raised by the last claims of a short kernel is first seen by the next kernel)
        assert info["preemptions"] == total + 1, (it, kernel, claim, info)
        total = info["preemptions"]
        check(kind, ex.graph_result(key, dt), want)


def test_pagerank_push_runs_every_tile_exactly_once(gp):
    """The push kernel is not idempotent: with residual increments of 0.5 (exact in fp32 in any
    order) the residual of a vertex must equal half its in-degree, also when the launch is stopped
    half-way and continued."""
    rng = np.random.default_rng(0)
    n, deg = 20000, 8
    indices = rng.integers(0, n, n * deg).astype(np.uint64)
    indptr = (np.arange(n + 1) * deg).astype(np.uint64)
    want = np.bincount(indices.astype(np.int64), minlength=n).astype(np.float32) * 0.5
    bufs = dict(vl=gp.DevBuf.from_array(indptr), el=gp.DevBuf.from_array(indices),
                active=gp.DevBuf.from_array(np.ones(n, np.uint8)), delta=gp.DevBuf.from_array(np.full(n, 0.5, np.float32)),
                residual=gp.DevBuf.from_array(np.zeros(n, np.float32)), value=gp.DevBuf.from_array(np.zeros(n, np.float32)),
                changed=gp.DevBuf.from_array(np.zeros(1, np.uint32)))
    p = gp.GraphParams(3, 0, n, bufs["vl"].ptr, bufs["el"].ptr, None, None, bufs["active"].ptr, None, None,
                       bufs["delta"].ptr, bufs["residual"].ptr, bufs["value"].ptr, 0.85, 0.001, None, None, bufs["changed"].ptr, 0)
    flag = gp.Flag()
    st = gp.BlpState(1, flag)
    info = gp.launch("gp_launch_graph", p, st.ctx(0, inject_at=40))
    gp.check(gp.lib().gp_stream_sync(None))
    assert info.total_tiles >= n // 4 // 16
    assert st.stop_index() == 0 and flag.get() == 1
    part = bufs["residual"].download(np_dtype=np.float32)
    assert not np.array_equal(part, want)
    flag.set(0)
    st.clear_stop()
    gp.launch("gp_launch_graph", p, st.ctx(0))
    gp.check(gp.lib().gp_stream_sync(None))
    assert st.stop_index() == -1
    assert np.array_equal(bufs["residual"].download(np_dtype=np.float32), want)
    assert not bufs["active"].download(np_dtype=np.uint8).any()


@pytest.mark.parametrize("lanes", [16, 32, 64])
def test_bfs_step_lane_widths(gp, graph, lanes):
    """one BFS level through the C ABI at each lane-group width, against the oracle's frontier"""
    _, indptr, indices, _ = graph
    label = np.full(N, G.INF, np.uint32)
    label[0] = 0
    want, _ = G.bfs(indptr, indices)
    bufs = dict(vl=gp.DevBuf.from_array(indptr.astype(np.uint64)), el=gp.DevBuf.from_array(indices.astype(np.uint64)),
                label=gp.DevBuf.from_array(label), changed=gp.DevBuf.from_array(np.zeros(1, np.uint32)))
    for level in range(3):
        p = gp.GraphParams(0, level, N, bufs["vl"].ptr, bufs["el"].ptr, None, bufs["label"].ptr, None, None, None,
                           None, None, None, 0, 0, None, None, bufs["changed"].ptr, lanes)
        info = gp.launch("gp_launch_graph", p)
        assert info.total_tiles == (N + 256 // lanes - 1) // (256 // lanes)
    gp.check(gp.lib().gp_stream_sync(None))
    got = bufs["label"].download(np_dtype=np.uint32)
    assert np.array_equal(got[want <= 3], want[want <= 3]) and (got[want > 3] == G.INF).all()
    p = gp.GraphParams(0, 0, N, bufs["vl"].ptr, bufs["el"].ptr, None, bufs["label"].ptr, None, None, None,
                       None, None, None, 0, 0, None, None, bufs["changed"].ptr, 8)
    with pytest.raises(gp.GpError):
        gp.launch("gp_launch_graph", p)


@pytest.mark.parametrize("kind", ["cc", "pagerank"])
def test_host_timed_preemption(gp, ex_mod, kind):
    """The flag goes up whenever the host gets to it, several times per run, while the count of
    active latency-critical tasks is non-zero (the reference's lc_tasks); the result is the same."""
    wl = f"{kind}@n=400000,deg=6,seed=11"
    base = ex_mod.Executor(wl)
    base.execute()
    key, dt = ("comp", np.uint64) if kind == "cc" else ("value", np.float32)
    want = base.graph_result(key, dt).copy()
    ex = ex_mod.Executor(wl, blp=True)
    flag = gp.Flag()
    ex.set_flag(flag)
    stream = gp.Stream(1)
    preempted = 0
    for _ in range(4):
        done = threading.Event()

        def run():
            ex.execute(stream)
            done.set()
        t = threading.Thread(target=run)
        t.start()
        while not done.is_set():
            ex.set_lc_tasks(1)
            flag.set(1)
            time.sleep(0.0003)
            flag.set(0)
            ex.set_lc_tasks(0)
            time.sleep(0.0005)
        t.join()
        got = ex.graph_result(key, dt)
        if kind == "cc":
            assert np.array_equal(got, want)
        else:
            assert np.abs(got - want).max() < 2 * PR_TOL
        preempted = ex.graph_info()["preemptions"]
    assert preempted > 0


def test_golden_graph_on_the_gpu(gp, ex_mod):
    """tests/golden/tiny_graph (10 vertices, answers worked out by hand) through the executors"""
    import json
    import os
    base = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "tiny_graph")
    want = json.load(open(base + ".expected.json"))
    for kind, key, dt, field in (("bfs", "label", np.uint32, "bfs_levels"), ("cc", "comp", np.uint64, "components"), ("sssp", "cost", np.uint32, "distances")):
        ex = ex_mod.Executor(kind, blp=True, graph_path=base)
        ex.set_flag(gp.Flag())
        ex.execute()
        assert ex.graph_result(key, dt).tolist() == want[field], kind


def test_ragged_graph_with_sinks_and_isolated_vertices(gp, ex_mod, tmp_path):
    """directed edges, a sink (no out-edges), an isolated vertex, a self-contained pair, and a
    vertex whose neighbour list is longer than a wavefront"""
    import os
    import struct
    n = 200
    adj = {v: [] for v in range(n)}
    for v in range(1, 150):
        adj[0].append(v)          # a hub with 149 out-edges
    for v in range(1, 100):
        adj[v].append(v + 1)      # a directed chain 1 -> 2 -> ... -> 100
    adj[150].append(151)
    adj[151].append(150)          # a pair on its own
    # 100..149 are sinks; 152..199 are isolated
    indptr, indices = [0], []
    for v in range(n):
        indices += sorted(adj[v])
        indptr.append(len(indices))
    w = [1 + (i * 7) % 13 for i in range(len(indices))]
    base = str(tmp_path / "ragged")
    for ext, arr, fmt, size in ((".col", indptr, "Q", 8), (".dst", indices, "Q", 8), (".val", w, "I", 4)):
        with open(base + ext, "wb") as f:
            f.write(struct.pack("<QQ", len(arr), size))
            f.write(struct.pack("<%d%s" % (len(arr), fmt), *arr))
    ip, ix, ww = G.read_graph(base, weights=True)
    for kind, key, dt, want in (("bfs", "label", np.uint32, G.bfs(ip, ix)[0]), ("cc", "comp", np.uint64, G.cc(ip, ix)[0]),
                                ("sssp", "cost", np.uint32, G.sssp(ip, ix, ww)[0])):
        ex = ex_mod.Executor(kind, blp=True, graph_path=base)
        ex.set_flag(gp.Flag())
        ex.execute()
        assert np.array_equal(ex.graph_result(key, dt), want), kind
    ex = ex_mod.Executor("pagerank", blp=True, graph_path=base)
    ex.set_flag(gp.Flag())
    ex.execute()
    value = ex.graph_result("value", np.float32)
    ref, _ = G.pagerank(ip, ix)
    assert np.isfinite(value).all() and np.abs(value - ref).max() < 5e-3
    assert np.allclose(value[152:], 0.15)  # nobody points at the isolated vertices
    # a malformed file is refused, not launched
    with open(base + ".dst", "r+b") as f:
        f.seek(16)
        f.write(struct.pack("<Q", 10 ** 6))
    with pytest.raises(ex_mod.StatusError):
        ex_mod.Executor("bfs", graph_path=base)


def _write_directed(base, n, edges, rng):
    edges = edges[np.lexsort((edges[:, 1], edges[:, 0]))]
    indptr = np.zeros(n + 1, np.uint64)
    indptr[1:] = np.cumsum(np.bincount(edges[:, 0], minlength=n))
    w = rng.integers(1, 1000, len(edges)).astype(np.uint32)
    for ext, arr in ((".col", indptr), (".dst", edges[:, 1].astype(np.uint64)), (".val", w)):
        with open(base + ext, "wb") as f:
            np.array([arr.size, arr.itemsize], np.uint64).tofile(f)
            arr.tofile(f)


@pytest.mark.parametrize("symmetric", [False, True])
@pytest.mark.parametrize("n,m", [(1, 0), (2, 1), (63, 200), (257, 900), (1025, 3000), (20000, 90000), (300000, 700000)])
def test_queued_iterations_at_the_edges_of_tiles(gp, ex_mod, tmp_path, n, m, symmetric):
    """sizes around the 64 vertices of a wavefront and the 256 of a tile, several tiles per claim, directed graphs
    (PageRank pulls along the transpose), self-loops, double edges and a hub whose list a whole wavefront walks"""
    rng = np.random.default_rng(n)
    edges = np.stack([rng.integers(0, n, m), rng.integers(0, n, m)], 1)
    hub = np.stack([np.full(min(n, 1500), n // 2), rng.permutation(n)[:1500]], 1)
    chain = np.stack([np.zeros(1, int), np.full(1, n // 2)], 1)
    edges = np.concatenate([edges, hub, chain])
    if symmetric:
        edges = np.concatenate([edges, edges[:, ::-1]])
    base = str(tmp_path / "g")
    _write_directed(base, n, edges, rng)
    ip, ix, w = G.read_graph(base, weights=True)
    for blp in (False, True):
        for kind, key, dt in (("bfs", "label", np.uint32), ("sssp", "cost", np.uint32), ("cc", "comp", np.uint64), ("pagerank", "value", np.float32)):
            if kind == "cc" and not symmetric:
                continue  # labels of a directed graph depend on the order of arrival in the reference's scheme
            ex = ex_mod.Executor(kind, blp=blp, graph_path=base)
            if blp:
                ex.set_flag(gp.Flag())
            for _ in range(2):
                ex.execute()
                got = ex.graph_result(key, dt)
                if kind == "pagerank":
                    want = G.pagerank(ip, ix)[0]
                    assert np.abs(got - want).max() < 5e-3 * max(1, want.max()), n
                else:
                    want = {"bfs": lambda: G.bfs(ip, ix)[0], "sssp": lambda: G.sssp(ip, ix, w)[0], "cc": lambda: G.cc(ip, ix)[0]}[kind]()
                    assert np.array_equal(got, want), (kind, n)


@pytest.mark.parametrize("bridge", [3, 1000, 10 ** 6, 0x70000000])
@pytest.mark.parametrize("n", [300, 40000])
def test_one_heavy_edge_in_a_light_graph(gp, ex_mod, tmp_path, n, bridge):
    """the second half of the vertices hangs on the first by one edge: the iterations do not grow with its weight"""
    rng = np.random.default_rng(n)
    half = n // 2
    u = np.arange(half - 1)
    near = np.concatenate([np.stack([u, u + 1], 1)[:50], np.stack([rng.integers(0, 51, half), np.arange(half)], 1)])
    edges = np.concatenate([near, near + half, [[half - 1, half]]])
    base = str(tmp_path / "g")
    _write_directed(base, n, edges, rng)
    ip, ix, _ = G.read_graph(base, weights=True)
    w = np.where(ix == half, bridge, 1).astype(np.uint32)  # (the bridge, and an edge or two back to its far end)
    with open(base + ".val", "wb") as f:
        np.array([w.size, 4], np.uint64).tofile(f)
        w.tofile(f)
    want = G.sssp(ip, ix, w)[0]
    assert want[half:].min() >= bridge
    ex = ex_mod.Executor("sssp", blp=True, graph_path=base)
    ex.set_flag(gp.Flag())
    for _ in range(2):
        ex.execute()
        assert np.array_equal(ex.graph_result("cost", np.uint32), want)
        # at most 52 hops to either side: three iterations for each, and those of the gap
        assert ex.graph_info()["iterations"] <= 3 * 2 * 53 + 10


@pytest.mark.parametrize("kind", ["bfs", "sssp", "cc", "pagerank"])
@pytest.mark.parametrize("n,deg", [(60000, 6), (1 << 20, 8)])
def test_queued_launches_stopped_again_and_again(gp, ex_mod, kind, n, deg):
    """The launches a user's run queues, under a flag that goes up and down faster than an iteration: short launches that
    are finished and long ones that give their claims back.  The result is the undisturbed run's."""
    wl = f"{kind}@n={n},deg={deg},seed=3"
    key, dt = {"bfs": ("label", np.uint32), "sssp": ("cost", np.uint32), "cc": ("comp", np.uint64), "pagerank": ("value", np.float32)}[kind]
    base = ex_mod.Executor(wl)
    base.execute()
    want = base.graph_result(key, dt).copy()
    ex = ex_mod.Executor(wl, blp=True)
    flag, stream = gp.Flag(), gp.Stream(1)
    ex.set_flag(flag)
    for pause in (20e-6, 60e-6, 150e-6, 400e-6):
        done = threading.Event()

        def run():
            ex.execute(stream)
            done.set()
        before = ex.graph_info()["preemptions"]
        t = threading.Thread(target=run)
        t.start()
        ups = 0
        while not done.is_set():
            flag.set(ups < 300 and ups % 2 == 0)  # (not for ever: a run that is stopped faster than it starts would never end)
            ups += 1
            until = time.perf_counter() + pause
            while time.perf_counter() < until:
                pass
        flag.set(0)
        t.join()
        got = ex.graph_result(key, dt)
        if kind == "pagerank":
            # shares that are taken in another order stop an iteration apart; the bound is the module's own
            assert np.abs(got - want).max() < PR_TOL, pause
        else:
            assert np.array_equal(got, want), pause
        if pause >= 150e-6 and n == 1 << 20:
            assert ex.graph_info()["preemptions"] > before, pause


@pytest.mark.parametrize("n,deg", [(300, 3), (4099, 8), (30000, 5), (200000, 16)])
@pytest.mark.parametrize("blp", [False, True])
def test_pagerank_of_a_generated_graph_pushes(gp, ex_mod, tmp_path, n, deg, blp):
    """A generated graph has every edge both ways, so that the last iterations push along the edges out where a file's
    graph pulls along those in.  A run ends with residuals between nothing and the tolerance t everywhere: the values
    are low by (I - alpha P^T)^-1 of these, which is t / (1 - alpha) times the solution x at most, vertex by vertex.
    (1e-5: some forty fp32 additions per vertex.)"""
    base = str(tmp_path / "g")
    assert ex_mod.lib().gpx_write_synthetic_graph(base.encode(), C.c_ulonglong(n), deg, C.c_ulonglong(13)) == 0
    x = G.pagerank_exact(*G.read_graph(base)[:2])
    launches = []
    for wl, path in ((f"pagerank@n={n},deg={deg},seed=13", None), ("pagerank", base)):
        ex = ex_mod.Executor(wl, blp=blp, graph_path=path)
        if blp:
            ex.set_flag(gp.Flag())
        for _ in range(2):
            before = ex.graph_info()["kernels_launched"]
            ex.execute()
            got = ex.graph_result("value", np.float32)
            assert (got <= x * (1 + 1e-5)).all() and (got >= x * (1 - 0.001 / 0.15 - 1e-5)).all(), wl
            info = ex.graph_info()
            launches.append(info["kernels_launched"] - before - info["iterations"])
    if n >= 30000:  # (going over to the push takes a launch; a small graph's sample of its vertices may miss the moment)
        assert min(launches[:2]) > max(launches[2:]), launches


class IterParams(C.Structure):
    vp = C.c_void_p
    _fields_ = [("kernel", C.c_int), ("level", C.c_uint), ("vertex_count", C.c_uint), ("row_end", C.c_uint)] + [(n, C.c_void_p) for n in (
        "row", "ids", "weights", "label", "cost", "parent", "active", "next_active", "comp", "share", "degree", "next_share", "residual",
        "value", "gained", "next_gained")] + [("alpha", C.c_float), ("tolerance", C.c_float), ("step", C.c_uint), ("changed", C.c_void_p),
        ("prev_changed", C.c_void_p), ("started", C.c_void_p), ("seq", C.c_uint), ("sets", C.c_uint), ("relay", C.c_void_p)]


IN_SETS = 0x53455453


@pytest.mark.parametrize("sets", [0, IN_SETS, 1])  # (1: what an older caller may have left in the gap)
@pytest.mark.parametrize("gap", [1, 1000])
def test_progress_words_in_one_set_and_in_eight(gp, sets, gap):
    """Shortest paths over 3000 vertices (twelve workgroups) launch by launch through the C ABI: the words of an iteration say how the
    next one goes on, whether they come in one set or in one per XCD.  gap: the weight of the one edge in the middle of the path
    behind the random part, so that the limit has to be looked for where it is large."""
    rng = np.random.default_rng(11)
    n, random_part = 3000, 2900
    edges = [(int(u), int(v), int(w)) for u, v, w in zip(rng.integers(0, random_part, 6000), rng.integers(0, random_part, 6000), rng.integers(1, 9, 6000)) if u != v]
    edges += [(v - 1, v, gap if v == 2950 else 1) for v in range(1, n)]
    edges += [(v, u, w) for u, v, w in edges]
    lists = [[] for _ in range(n)]
    for u, v, w in edges:
        lists[u].append((v, w))
    row, ids, weights = [0], [], []
    for l in lists:
        l = l + [(n, 0)] * (-len(l) % 4)
        ids += [v for v, _ in l]
        weights += [w for _, w in l]
        row.append(len(ids) // 4)
    ids += [n] * 4

    def dev(x):
        d = gp.DevBuf(x.nbytes)
        d.upload(x)
        return d

    d_row, d_ids, d_w = dev(np.array(row, np.uint32)), dev(np.array(ids, np.uint32)), dev(np.array(weights + [0] * 4, np.uint32))
    cost, active, next_active = dev(np.zeros(n + 1, np.uint32)), dev(np.zeros(n + 8, np.uint8)), dev(np.zeros(n + 8, np.uint8))
    slot = 8 * 32 if sets == IN_SETS else 32
    rounds = 400
    words = dev(np.zeros((rounds, slot), np.uint32))
    s = gp.Stream(0)
    p = IterParams(kernel=3, vertex_count=n, row_end=row[-1], row=d_row.ptr, ids=d_ids.ptr, weights=d_w.ptr, cost=cost.ptr, active=active.ptr,
                   next_active=next_active.ptr, step=5, changed=words.ptr, sets=sets)
    gp.launch("gp_launch_graph_iter", p, None, s)
    p.kernel = 2
    for i in range(rounds):
        p.changed = words.ptr + 4 * slot * i
        p.prev_changed = words.ptr + 4 * slot * (i - 1) if i else None
        p.active, p.next_active = (active.ptr, next_active.ptr) if i % 2 == 0 else (next_active.ptr, active.ptr)
        gp.launch("gp_launch_graph_iter", p, None, s)
    s.sync()
    said = words.download(np_dtype=np.uint8).view(np.uint32).reshape(rounds, -1, 32)
    ran = said[:, :, 0].any(axis=1)
    assert ran[0] and not ran[-1] and not ran[int(np.argmin(ran)):].any()  # it converged, and nothing ran behind that
    assert (said[:int(np.argmin(ran)), 1:, :5].any() if sets == IN_SETS else True)    # (the other sets are used)
    indptr = np.cumsum([0] + [len(l) for l in lists])
    indices = np.array([v for l in lists for v, _ in l])
    want = G.sssp(indptr, indices, np.array([w for l in lists for _, w in l], np.uint32))[0]
    assert np.array_equal(cost.download(np_dtype=np.uint8).view(np.uint32)[:n], want)
    if sets not in (0, IN_SETS):
        s.destroy()  # (the streams of a process share four hardware queues; tests that hold one of two streams up count on their share)
