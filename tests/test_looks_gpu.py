"""Launches whose tiles look at the stop word as they go (tile_loop.hpp: fixed claims, a front workgroup, counters of leavers), in the forms
of the matrix bodies with a scale and shift in front (gemm_pre.hpp) and with their input window in LDS (gemm_window.hpp): run
through, given up under a raised flag and resumed, to the bits of plain launches."""
import ctypes as C
import os
import subprocess
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def sweep(gp, launch, out, want):
    """launch(ctx) -> info; `out` is wiped between the launches"""
    flag = gp.Flag()
    st = gp.BlpState(1, flag, 32)
    st.enable_done_counters()

    def counted():
        return int(st.counters().reshape(32, 16)[:, 0].sum()), int(st.done.download(np_dtype=np.int32).reshape(32, 16)[:, 0].sum())

    for fresh, up in ((1, 0), (2, 0), (1, 1), (0, 1)):
        flag.set(up)
        st.reset(); st.clear_stop(); out.fill32(0x7E007E00)
        info = launch(st.ctx(fresh=fresh))
        made, left = counted()
        assert info.fixed_claims == 1 and info.front == 8  # the form that looks
        assert left == info.grid - info.front
        if not up:
            assert made == info.total_tiles and np.array_equal(out.download(), want)
        elif made == 0:
            assert (out.download().view(np.uint16) == 0x7E00).all()  # nothing claimed, nothing written
        flag.set(0); st.clear_stop()
        launch(st.ctx(done_launches=1))
        assert np.array_equal(out.download(), want) and counted()[0] == info.total_tiles


def scaled(gp, dt, case):
    """tests/test_eltwise_conv_gpu.py's layer and convolution"""
    import test_eltwise_conv_gpu as t
    e, c, mid, out, keep = t.setup(gp, dt, case, gp.ACT_RELU, residual=True)
    want = t.two_launches(gp, e, c, mid, out)
    sweep(gp, lambda ctx: t.fused(gp, e, c, ctx), out, want)


# fp32 layers whose tiles are long by the launcher's own rule: the 14 x 14 blocks of DenseNet-201 at batch 16
@pytest.mark.parametrize("case", [(16, 14, 576, 128, 576), (16, 14, 1760, 128, 1792), (12, 14, 1120, 128, 1120), (11, 14, 1188, 130, 1792)], ids=lambda c: "x".join(map(str, c)))
def test_scaled_layers_of_long_tiles(gp, case):
    scaled(gp, "f32", case)


def windowed(gp, dt, images, H, Cin, Cout, R):
    dtype, rng = gp.DTYPE_BY_NAME[dt], np.random.default_rng(H + Cin)
    x, w, b = (gp.DevBuf.from_array(rng.uniform(-1, 1, s).astype(np.float32), dtype) for s in ((images, H, H, Cin), (Cout, R, R, Cin), (Cout,)))
    out = gp.DevBuf((images * H * H * Cout * 2 + 3) // 4 * 4)
    p = gp.ConvParams(dtype=dtype, N=images, H=H, W=H, Cin=Cin, Cout=Cout, R=R, S=R, stride_h=1, stride_w=1, pad_h=R // 2, pad_w=R // 2, in_=x.ptr, in_pix_stride=Cin, weight=w.ptr,
                      bias=b.ptr, out=out.ptr, out_pix_stride=Cout, act=gp.ACT_RELU)
    name = C.create_string_buffer(64)
    gp.check(gp.lib().gp_conv2d_body(C.byref(p), name, C.c_size_t(len(name))))
    assert name.value == b"wide32x32_16 window"

    def launch(ctx):
        info = gp.launch("gp_launch_conv2d", p, ctx)
        gp.check(gp.lib().gp_stream_sync(None))
        return info
    out.fill32(0x7E007E00)
    launch(None)
    sweep(gp, launch, out, out.download().copy())


def child():
    from gpreempt_amd import capi as gp
    gp.init(0)
    n = 0
    for dt in ("f32", "f16", "bf16"):
        # 64 x 64 tiles of one K-step to nine; eight and sixteen wavefronts of one stage and more; fp32: 16 x 16 and 32 x 16 tiles
        for case in ((4, 28, 32, 128, 64), (4, 28, 256, 128, 256), (4, 28, 480, 128, 512), (2, 17, 576, 160, 608), (4, 14, 1024, 128, 1792), (4, 7, 1880, 130, 1920), (8, 14, 800, 250, 800)):
            print("scaled", dt, case, flush=True)
            scaled(gp, dt, case)
            n += 1
    for dt in ("f16", "bf16"):
        # 3 x 3 over one K-block of channels to twelve (3 to 27 stages), and 5 x 5
        for case in ((4, 7, 128, 32, 3), (8, 7, 512, 512, 3), (2, 14, 128, 32, 3), (5, 3, 768, 33, 3), (1, 28, 128, 128, 3), (1, 9, 192, 40, 5)):
            print("windowed", dt, case, flush=True)
            windowed(gp, dt, *case)
            n += 1
    print("OK", n)


def test_every_form_looks(gp):
    """The threshold that selects the form is read once per process, hence the child process with GPREEMPT_LONG_TILE_MACS=1."""
    code = "import sys; sys.path[:0] = sys.argv[1:]; import test_looks_gpu; test_looks_gpu.child()"
    out = subprocess.run([sys.executable, "-c", code, ROOT, os.path.join(ROOT, "tests")], capture_output=True, text=True, timeout=110, env={**os.environ, "GPREEMPT_LONG_TILE_MACS": "1"})
    assert out.returncode == 0 and out.stdout.strip().endswith("OK 33"), (out.stdout[-600:], out.stderr[-1500:])
