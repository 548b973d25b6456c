"""Models that merge launches (DenseNet's scale-shift layers, Inception's branches), stopped at, launched at and recorded with the kernels that
another kernel's launch does.  (What a caller sees of their storages: tests/test_fusion_cpu.py.)"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_a_dense_block_in_a_graph_and_stopped_at_its_scale_shift_layers(gp, monkeypatch):
    """... every storage is there behind every replay, whatever the model has run in between, and a preemption injected at a
    layer that is otherwise left to its convolution fires and resumes to the same bits"""
    from gpreempt_amd import executor as ex_mod
    monkeypatch.setenv("GPREEMPT_USE_HIPGRAPH", "1")
    wl = "densenet201@b=2,hw=64,l1=2,l2=2,l3=2,l4=2,dtype=f16"
    inputs = [gp.to_storage(np.random.default_rng(s).standard_normal((2, 3, 64, 64), np.float32), gp.F16) for s in range(3)]
    shown = ("block1.layer1.norm1.out", "block2.layer2.norm1.out", "heads")

    def model(fuse):
        monkeypatch.setenv("GPREEMPT_FUSE_LN", fuse)
        ex, stream, flag = ex_mod.Executor(wl, blp=True), gp.Stream(1), gp.Flag()
        ex.set_flag(flag)
        ex.set_running(True)
        return ex, stream, flag

    def see(ex, stream, x):
        ex.set_input("data", x, stream)
        ex.execute(stream)
        return [ex.get_output(k, stream).tobytes() for k in shown]

    apart, stream_a, _ = model("0")
    want = [see(apart, stream_a, x) for x in inputs]
    ex, stream, flag = model("1")
    assert [see(ex, stream, x) for x in inputs] == want  # launch by launch
    layers = [i for i, k in enumerate(ex.kernels()) if k["name"] == "eltwise"]
    ex.set_input("data", inputs[0], stream)
    for layer in layers[:6]:
        ex.inject_preempt(layer, 0)
        ex.execute(stream)
        stream.sync()
        assert flag.get() == 1
        flag.set(0)
        ex.inject_preempt(-1, -1)
        ex.resume(stream)
        stream.sync()
        assert ex.last_stop_index() in (layer, layer + 1)  # (a layer whose tiles were all claimed at once ends)
        assert [ex.get_output(k, stream).tobytes() for k in shown] == want[0]
    ex.capture_graph(stream)
    assert not ex.uses_program()
    for _ in range(2):
        assert [see(ex, stream, x) for x in inputs] == want
        for _ in range(3):  # stopped inside a replay, resumed kernel by kernel
            ex.execute(stream)
            flag.set(1)
            stream.sync()
            flag.set(0)
            ex.resume(stream)
            assert [ex.get_output(k, stream).tobytes() for k in shown] == want[2]


def test_a_preemption_injected_at_a_member_fires_and_a_member_launched_alone_runs(gp):
    from gpreempt_amd import executor as ex_mod
    x = gp.to_storage(np.random.default_rng(4).standard_normal((1, 3, 139, 139), np.float32), gp.F16)
    ex = ex_mod.Executor("inception@b=1,hw=139,dtype=f16", blp=True)
    stream, flag = gp.Stream(1), gp.Flag()
    ex.set_flag(flag)
    ex.set_running(True)
    ex.set_input("data", x, stream)
    ex.execute(stream)
    want = ex.get_output("heads", stream)
    members = [i for i, n in enumerate(ex.counters()) if n == 0]
    assert len(members) > 20
    for kernel in members[::6] + [members[0] - 1]:
        ex.inject_preempt(kernel, 0)
        ex.execute(stream)
        stream.sync()
        assert flag.get() == 1, kernel
        flag.set(0)
        ex.inject_preempt(-1, -1)
        ex.resume(stream)
        assert ex.last_stop_index() >= kernel and np.array_equal(ex.get_output("heads", stream), want)
        ex.reset_counters(stream)
        ex.launch_kernel(kernel, stream)
        stream.sync()
        assert ex.counters()[kernel] > 0


def test_inception_in_a_graph_stopped_and_resumed_kernel_by_kernel(gp, monkeypatch):
    """the recorded launches are the groups', and so are the relaunches, also when the model has been launched apart in between"""
    from gpreempt_amd import executor as ex_mod
    monkeypatch.setenv("GPREEMPT_USE_HIPGRAPH", "1")
    inputs = [gp.to_storage(np.random.default_rng(s).standard_normal((1, 3, 139, 139), np.float32), gp.F16) for s in range(2)]
    ex = ex_mod.Executor("inception@b=1,hw=139,dtype=f16", blp=True)
    stream, flag = gp.Stream(1), gp.Flag()
    ex.set_flag(flag)
    ex.set_running(True)

    def see(x):
        ex.set_input("data", x, stream)
        ex.execute(stream)
        return ex.get_output("heads", stream).tobytes()

    want = [see(x) for x in inputs]
    members = [i for i, n in enumerate(ex.counters()) if n == 0]
    ex.capture_graph(stream)
    assert not ex.uses_program()
    for k in range(6):
        assert [see(x) for x in inputs] == want
        ex.reset_counters(stream)  # kernel by kernel, one group apart
        ex.inject_preempt(members[5 * k], 1 << 20)
        for i in range(ex.kernel_num()):
            ex.launch_kernel(i, stream)
        ex.inject_preempt(-1, -1)
        assert ex.get_output("heads", stream).tobytes() == want[1]
        ex.execute(stream)
        flag.set(1)
        stream.sync()
        flag.set(0)
        ex.resume(stream)
        assert ex.get_output("heads", stream).tobytes() == want[1]
