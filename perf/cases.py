"""What is timed when the speed of this framework is compared between two trees.

A case is a dict of plain values.  There are four kinds, each the work of one sort of user:

  request      a model served through Executor / BLPExecutor: the input comes from host memory, the model's
               kernels run, the output goes back to host memory.  `blp`: the tenant is preemptible.  `stop`: a
               higher level's request arrives right behind the submission: the flag goes up, the tenant leaves
               the GPU, the flag comes down and the tenant resumes.
  gemm         one matrix product on operands in device memory through the C ABI, plainly or as a preemptible
               launch with its claim counters (and, for long tiles, its checkpoint workspace) cleared first.
  miniweather  a stretch of the weather simulation between two outputs of its state.
  graph        one run of a graph algorithm to convergence and its result.
"""
import math
import os
import tempfile

import numpy as np
import torch

from gpreempt_amd import capi as gp
from gpreempt_amd import executor as gx

ES = {"f32": 4, "f16": 2, "bf16": 2}
TORCH = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
VOCAB = 30522
FUSED_BERT = ("f16", "bf16")
# multiply-adds of one image (224 x 224; Inception-v3 299 x 299) and weights
CNN = {"resnet50": (3.9e9, 25.6e6), "resnet101": (7.6e9, 44.5e6), "resnet152": (11.3e9, 60.2e6), "vgg16": (15.5e9, 138.4e6),
       "densenet201": (4.3e9, 20.0e6), "inception": (5.7e9, 23.8e6)}
GRAPH_RESULT = {"bfs": ("label", np.uint32), "cc": ("comp", np.uint64), "sssp": ("cost", np.uint32), "pagerank": ("value", np.float32)}


def listed():
    return [
        # the smallest request: one element-wise kernel and a copy, what the 500 req/s latency probe of the ResNet-50 scenario asks for
        {"name": "probe_64x64", "kind": "request", "model": "toy", "rows": 64, "cols": 64, "dtype": "f32", "blp": False, "stop": False},
        # the headline's high-priority request
        {"name": "bert_b1_s128_f16", "kind": "request", "model": "bert", "b": 1, "s": 128, "dtype": "f16", "blp": False, "stop": False},
        # a small batch of requests of odd length, in the other 16-bit type
        {"name": "bert_b2_s211_bf16", "kind": "request", "model": "bert", "b": 2, "s": 211, "dtype": "bf16", "blp": False, "stop": False},
        # the best-effort tenants of the two-, three- and ten-tenant scenarios
        {"name": "resnet50_b1_f32", "kind": "request", "model": "resnet50", "b": 1, "dtype": "f32", "blp": True, "stop": False},
        {"name": "resnet152_b8_f16", "kind": "request", "model": "resnet152", "b": 8, "dtype": "f16", "blp": True, "stop": False},
        {"name": "densenet201_b4_f16", "kind": "request", "model": "densenet201", "b": 4, "dtype": "f16", "blp": True, "stop": False},
        {"name": "vgg16_b16_f16", "kind": "request", "model": "vgg16", "b": 16, "dtype": "f16", "blp": True, "stop": False},
        # ... and one of them stopped by a request of a higher level and resumed
        {"name": "inception_b1_f16_stopped", "kind": "request", "model": "inception", "b": 1, "dtype": "f16", "blp": True, "stop": True},
        # the smallest scenario of all: C = relu(A B + bias) of 1024^3 in fp32
        {"name": "gemm_1024_f32", "kind": "gemm", "m": 1024, "n": 1024, "k": 1024, "dtype": "f32", "bias": True, "act": gp.ACT_RELU, "blp": True},
        # the heaviest best-effort tenant
        {"name": "gemm_8192_bf16", "kind": "gemm", "m": 8192, "n": 8192, "k": 8192, "dtype": "bf16", "bias": False, "act": gp.ACT_NONE, "blp": True},
        # the simulation at the size of the reference's configuration, an output every 20 executes
        {"name": "miniweather_3200x1600", "kind": "miniweather", "nx": 3200, "nz": 1600, "steps": 20},
        # the longest of the four graph tenants at the size of their scenario
        {"name": "pagerank_1m", "kind": "graph", "algorithm": "pagerank", "n": 1 << 20, "deg": 8},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["bert", "bert", "cnn", "cnn", "cnn", "gemm", "gemm", "toy", "miniweather", "graph", "graph"])
    if kind == "toy":
        return {"kind": "request", "model": "toy", "rows": _log(rng, 8, 1024), "cols": 8 * _log(rng, 1, 96), "dtype": rng.choice(["f32", "f16", "bf16"]), "blp": False, "stop": False}
    if kind == "bert":
        dtype, s = rng.choice(["f16", "f16", "bf16", "f32"]), _log(rng, 16, 512)
        if dtype not in FUSED_BERT:  # the three-launch form of attention multiplies over the sequence, in vectors of four
            s = max(16, s // 4 * 4)
        b = _log(rng, 1, max(1, min(8, 1024 // s)))
        blp = rng.random() < 0.3
        return {"kind": "request", "model": "bert", "b": b, "s": s, "dtype": dtype, "blp": blp, "stop": blp and rng.random() < 0.4}
    if kind == "cnn":
        dtype, blp = rng.choice(["f16", "f16", "bf16", "f32"]), rng.random() < 0.7
        return {"kind": "request", "model": rng.choice(sorted(CNN)), "b": _log(rng, 1, 16), "dtype": dtype, "blp": blp, "stop": blp and rng.random() < 0.3}
    if kind == "gemm":
        dtype = rng.choice(["f32", "f16", "bf16"])
        return {"kind": "gemm", "m": _log(rng, 1, 8192), "n": _log(rng, 32, 8192), "k": 8 * _log(rng, 8, 1024), "dtype": dtype,
                "bias": rng.random() < 0.7, "act": rng.choice([gp.ACT_NONE, gp.ACT_RELU, gp.ACT_GELU]), "blp": rng.random() < 0.5}
    if kind == "miniweather":
        return {"kind": "miniweather", "nx": _log(rng, 100, 3200), "nz": _log(rng, 50, 1600), "steps": rng.randint(5, 20)}
    return {"kind": "graph", "algorithm": rng.choice(sorted(GRAPH_RESULT)), "n": _log(rng, 1 << 12, 1 << 20), "deg": rng.randint(2, 8)}


def workload(case):
    """The executor's name for the case's model."""
    if case["model"] == "toy":
        return "toy@rows=%d,cols=%d,n=1,dtype=%s" % (case["rows"], case["cols"], case["dtype"])
    size = "b=%d,s=%d" % (case["b"], case["s"]) if case["model"] == "bert" else "b=%d" % case["b"]
    return "%s@%s,dtype=%s" % (case["model"], size, case["dtype"])


class Server:
    """A loaded model with its stream and flag.  A serving program loads it once and feeds it requests."""

    def __init__(self, case):
        self.ex = gx.Executor(workload(case), blp=case["blp"])
        self.stream = gp.Stream(1 if case["blp"] else 0)
        self.flag = gp.Flag()
        if case["blp"]:
            self.ex.set_flag(self.flag)
            self.ex.set_running(True)


_servers = {}


def _server(case):
    key = (workload(case), case["blp"])
    if key not in _servers:
        _servers[key] = Server(case)
    return _servers[key]


def _prepare_request(case, seed):
    rng = np.random.default_rng(seed)
    if case["model"] == "bert":
        data = rng.integers(0, VOCAB, (case["b"], case["s"]), np.int64)
    else:
        hw = 299 if case["model"] == "inception" else 224
        shape = (case["rows"], case["cols"]) if case["model"] == "toy" else (case["b"], 3, hw, hw)
        data = gp.to_storage(rng.standard_normal(shape, np.float32), gp.DTYPE_BY_NAME[case["dtype"]])
    return {"run": _run_request, "server": _server(case), "data": data, "dtype": TORCH[case["dtype"]], "stop": case["stop"]}


def _run_request(st):
    ex, stream, flag = st["server"].ex, st["server"].stream, st["server"].flag
    ex.set_input("data", st["data"], stream)
    ex.execute(stream)
    if st["stop"]:
        flag.set(1)
        stream.sync()
        flag.set(0)
        ex.resume(stream)
    return torch.from_numpy(ex.get_output("heads", stream)).view(st["dtype"])


def _prepare_gemm(case, seed):
    gp.init(0)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dtype, M, N, K = TORCH[case["dtype"]], case["m"], case["n"], case["k"]

    def uniform(*shape):
        return (torch.rand(shape, generator=gen, device="cuda") * 2 - 1).to(dtype)

    A, B, C = uniform(M, K), uniform(N, K), torch.empty((M, N), dtype=dtype, device="cuda")
    bias = uniform(N) if case["bias"] else None
    p = gp.GemmParams(dtype=gp.DTYPE_BY_NAME[case["dtype"]], M=M, N=N, K=K, A=A.data_ptr(), lda=K, B=B.data_ptr(), ldb=K, b_is_nk=1,
                      C=C.data_ptr(), ldc=N, bias=bias.data_ptr() if case["bias"] else None, alpha=1.0, act=case["act"], batch=1)
    state = {"run": _run_gemm, "p": p, "C": C, "keep": (A, B, bias), "stream": gp.Stream(1 if case["blp"] else 0), "blp": None}
    if case["blp"]:
        state["blp"] = gp.BlpState(1, gp.Flag(), 32)
        state["blp"].enable_checkpoints(p)
        state["ctx"] = state["blp"].ctx(fresh=2)
    torch.cuda.synchronize()
    return state


def _run_gemm(st):
    blp, ctx = st["blp"], None
    if blp is not None:
        ctx = st["ctx"]
        gp.check(gp.lib().gp_fill32_async(gp.vp(blp.executed.ptr), gp.C.c_uint32(0), gp.C.c_size_t(blp.ints_per_kernel), st["stream"].h))
        if blp.ckpt is not None:
            gp.check(gp.lib().gp_ckpt_reset_async(gp.vp(blp.ckpt.ptr), st["stream"].h))
    gp.launch("gp_launch_gemm", st["p"], ctx, st["stream"])
    return st["C"]


def _prepare_miniweather(case, seed):
    ex = gx.Executor("miniweather@nx=%d,nz=%d" % (case["nx"], case["nz"]), blp=True)
    stream, flag = gp.Stream(1), gp.Flag()
    ex.set_flag(flag)
    # the two colliding thermals the workload starts from, a little stronger or weaker and with noise on their temperature
    rng = np.random.default_rng(seed)
    x = ex.read_storage("state").view(np.float32).reshape(4, case["nz"] + 4, case["nx"] + 4)
    inside = x[3, 2:-2, 2:-2]
    inside *= rng.uniform(0.8, 1.2)
    inside += 0.01 * rng.standard_normal(inside.shape, np.float32)
    ex.set_input("state", x, stream)
    ex.set_input("state_tmp", x.copy(), stream)
    stream.sync()
    return {"run": _run_miniweather, "ex": ex, "stream": stream, "flag": flag, "steps": case["steps"]}


def _run_miniweather(st):
    for _ in range(st["steps"]):
        st["ex"].execute(st["stream"])
    return st["ex"].get_output("state", st["stream"]).view(np.float32)


def _write_communities(base, n, deg, seed):
    """An undirected graph of many components as the files a data set comes in (count, element size, values): every
    vertex has `deg` neighbours among the next 64, none across the borders between communities of random sizes."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    v = torch.arange(n, device="cuda").repeat_interleave(deg)
    u = v + torch.randint(1, 65, v.shape, generator=gen, device="cuda")
    community = (torch.rand(n, generator=gen, device="cuda") < 1 / 500).cumsum(0)
    u, v = u[u < n], v[u < n]
    same = community[u] == community[v]
    u, v = u[same], v[same]
    key = (torch.cat([u, v]) * n + torch.cat([v, u])).sort().values
    offsets = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    offsets[1:] = torch.bincount(key // n, minlength=n).cumsum(0)
    for suffix, values in ((".col", offsets), (".dst", key % n)):
        with open(base + suffix, "wb") as f:
            np.array([values.numel(), 8], np.uint64).tofile(f)
            values.cpu().numpy().tofile(f)


def _prepare_graph(case, seed):
    if case["algorithm"] == "cc":  # the built-in random graph is one component: its labels would all be 0
        with tempfile.TemporaryDirectory() as d:
            base = os.path.join(d, "graph")
            _write_communities(base, case["n"], case["deg"], seed)
            ex = gx.Executor("cc", blp=True, graph_path=base)
    else:
        ex = gx.Executor("%s@n=%d,deg=%d,seed=%d" % (case["algorithm"], case["n"], case["deg"], 1 + seed), blp=True)
    stream, flag = gp.Stream(1), gp.Flag()
    ex.set_flag(flag)
    return {"run": _run_graph, "ex": ex, "stream": stream, "flag": flag, "result": GRAPH_RESULT[case["algorithm"]]}


def _run_graph(st):
    st["ex"].execute(st["stream"])
    return st["ex"].graph_result(*st["result"])


PREPARE = {"request": _prepare_request, "gemm": _prepare_gemm, "miniweather": _prepare_miniweather, "graph": _prepare_graph}


def prepare(case, seed):
    return PREPARE[case["kind"]](case, seed)


def run(state):
    return state["run"](state)


def work(case):
    """Inputs, weights and results once; activations between the kernels are not counted."""
    if case["kind"] == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": ES[case["dtype"]] * (m * k + n * k + m * n), "flops": 2.0 * m * n * k}
    if case["kind"] == "miniweather":  # 12 stages of a time step pair read the state and write it; about 350 operations per cell and stage
        cells = float(case["nx"] * case["nz"])
        return {"bytes": case["steps"] * 12 * 2 * 4 * 4 * cells, "flops": case["steps"] * 12 * 350 * cells}
    if case["kind"] == "graph":  # neighbour lists (64-bit ids, both directions of every edge) once, a result of 4 bytes per vertex
        n, edges = case["n"], 2.0 * case["n"] * case["deg"]
        return {"bytes": 8 * (n + edges) + 4 * n, "flops": edges}
    es = ES[case["dtype"]]
    if case["model"] == "toy":
        return {"bytes": 2 * es * case["rows"] * case["cols"], "flops": case["rows"] * case["cols"]}
    if case["model"] == "bert":  # twelve layers of 7.1 million weights; the embedding rows of the tokens
        t = case["b"] * case["s"]
        return {"bytes": es * (85.0e6 + 2 * t * 768) + 8 * t, "flops": 2.0 * t * 85.0e6 + 12 * 4.0 * t * case["s"] * 768}
    macs, weights = CNN[case["model"]]
    hw = 299 if case["model"] == "inception" else 224
    return {"bytes": es * (weights + case["b"] * (3 * hw * hw + 1000)), "flops": 2.0 * macs * case["b"]}


def tolerance(case):
    if case["kind"] == "graph":
        # the other three count in whole numbers; PageRank adds fp32 contributions in order of arrival and stops with up to 0.001 per vertex undistributed
        return {"rel": 1e-3} if case["algorithm"] == "pagerank" else "exact"
    if case["kind"] == "miniweather":
        # fp32; the pressure terms are small differences of values near 1e5
        return {"rel": 1e-4}
    if case["kind"] == "gemm":
        return {"rel": {"f32": 1e-5, "f16": 1e-3, "bf16": 5e-3}[case["dtype"]]}
    if case["model"] == "toy":
        return "exact"
    # dozens of layers that each round their output to the type
    return {"rel": {"f32": 1e-4, "f16": 1e-2, "bf16": 2e-2}[case["dtype"]]}
