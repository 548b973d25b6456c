"""A scale-shift-ReLU layer and the pointwise convolution behind it as one launch (gp_launch_eltwise_conv2d): the bits of the two
launches, on every body that takes it, at the edges of its tiles and K-steps."""
import ctypes as C

import numpy as np
import pytest

from helpers import sync

pytestmark = pytest.mark.gpu
CASES = [
    # images, height, Cin, Cout, channels of the buffer the input is a slice of
    (1, 1, 8, 8, 8),           # one K-chunk of one row
    (1, 9, 72, 36, 96),        # K and N ragged
    (4, 56, 64, 128, 256),     # 64 x 64 tiles, ring of two stages
    (1, 28, 480, 128, 512),    # ... of four, K ends inside a K-step
    (2, 17, 576, 160, 608),    # 64 x 64 on eight wavefronts
    (4, 14, 1024, 128, 1792),  # 32 x 32 on sixteen
    (4, 7, 1880, 130, 1920),   # ... K ends inside a stage, N is no multiple of four
    (8, 14, 800, 250, 800),    # 64 x 32 on sixteen
]


def fused(gp, e, c, ctx=None):
    info = gp.LaunchInfo()
    gp.check(gp.lib().gp_launch_eltwise_conv2d(C.byref(e), C.byref(c), C.byref(ctx) if ctx is not None else None, None, C.byref(info)))
    sync(gp)
    return info


def setup(gp, dt, case, act, residual=False, special=False):
    images, H, Cin, Cout, wide = case
    dtype, rows = gp.DTYPE_BY_NAME[dt], images * H * H
    rng = np.random.default_rng(sum(case))
    buf = rng.standard_normal((rows, wide), np.float32)
    if special:  # not numbers and infinities, in the operand and where only the two together make one
        buf[0, 0], buf[rows // 2, 1], buf[-1, 2] = np.nan, np.inf, -np.inf
    scale, shift = rng.uniform(0.5, 1.5, Cin).astype(np.float32), rng.uniform(-1, 1, Cin).astype(np.float32)
    if special:
        scale[1] = 0.0
    w = rng.uniform(-1, 1, (Cout, Cin)).astype(np.float32) / np.sqrt(Cin)
    keep = [gp.DevBuf.from_array(v, dtype) for v in (buf, scale, shift, w, rng.uniform(-1, 1, Cout).astype(np.float32), rng.standard_normal((rows, Cout), np.float32))]
    mid, out = gp.DevBuf(rows * Cin * gp.DTYPE_SIZE[dtype]), gp.DevBuf(rows * Cout * gp.DTYPE_SIZE[dtype] + 64)
    e = gp.EltwiseParams(dtype, rows, Cin, keep[0].ptr, wide, None, 0, keep[1].ptr, keep[2].ptr, mid.ptr, Cin, act)
    c = gp.ConvParams(dtype=dtype, N=images, H=H, W=H, Cin=Cin, Cout=Cout, R=1, S=1, stride_h=1, stride_w=1, in_=mid.ptr, in_pix_stride=Cin, weight=keep[3].ptr, bias=keep[4].ptr,
                      residual=keep[5].ptr if residual else None, res_pix_stride=Cout, out=out.ptr, out_pix_stride=Cout, act=gp.ACT_RELU)
    return e, c, mid, out, keep


def two_launches(gp, e, c, mid, out):
    out.fill32(0x7E007E00)
    gp.launch("gp_launch_eltwise", e)
    gp.launch("gp_launch_conv2d", c)
    sync(gp)
    want = out.download().copy()
    out.fill32(0x7E007E00)
    mid.fill32(0x55AA55AA)
    return want


@pytest.mark.parametrize("dt", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c)))
def test_one_launch_has_the_bits_of_two(gp, dt, case):
    vec = 4 if dt == "f32" else 8
    case = case[:2] + (case[2] // vec * vec,) + case[3:]
    for act, residual, special in ((gp.ACT_RELU, False, False), (gp.ACT_NONE, True, False), (gp.ACT_RELU, False, True)):
        e, c, mid, out, keep = setup(gp, dt, case, act, residual, special)
        want = two_launches(gp, e, c, mid, out)
        assert gp.lib().gp_eltwise_conv2d_supported(C.byref(e), C.byref(c)) == 1
        fused(gp, e, c)
        assert np.array_equal(out.download(), want)
        assert (mid.download().view(np.uint32) == 0x55AA55AA).all()  # the layer's output is not written
        # a first preemptible launch, eager and not, and one that is stopped at its first claim and resumed
        flag = gp.Flag()
        for fresh, inject in ((2, -1), (1, -1), (0, 0)):
            st = gp.BlpState(1, flag, 32)
            out.fill32(0x7E007E00)
            fused(gp, e, c, st.ctx(fresh=fresh, inject_at=inject))
            flag.set(0)
            st.stop.upload(np.array([-1], np.int32))
            info = fused(gp, e, c, st.ctx())
            assert np.array_equal(out.download(), want)
            assert not info.fixed_claims or st.counters().reshape(32, 16)[:, 0].sum() == info.total_tiles


@pytest.mark.parametrize("dt", ["f16", "bf16", "f32"])
@pytest.mark.parametrize("case", [(1, 9, 72, 36, 96), (4, 14, 1024, 128, 1792)], ids=["64x64", "32x32"])
def test_products_at_the_ends_of_the_range_round_as_in_two_launches(gp, dt, case):
    """products beyond the largest float whose sum with the shift is not (bf16, fp32), and ones below the smallest normal float"""
    e, c, mid, out, keep = setup(gp, dt, case, gp.ACT_NONE)
    dtype, (images, H, Cin, Cout, wide) = gp.DTYPE_BY_NAME[dt], case
    big, tiny = (2.0 ** 15, 2.0 ** -24) if dt == "f16" else (2.0 ** 64, 1.5 * 2.0 ** -70)
    x, scale, shift = np.ones((images * H * H, wide), np.float32), np.ones(Cin, np.float32), np.zeros(Cin, np.float32)
    x[0::2, 0], x[1::2, 0], scale[0], shift[0] = 1.5 * big, 0.0, big, -1.984375 * 2.0 ** (15 if dt == "f16" else 127)
    x[:, 2:6], scale[2:6], shift[2:6] = tiny * 1.0078125, tiny * 1.0078125, np.array([0, 1, -1, 8], np.float32) * 2.0 ** (-24 if dt == "f16" else -133)
    for buf, v in zip(keep, (x, scale, shift, np.eye(Cout, Cin, dtype=np.float32), np.zeros(Cout, np.float32))):
        buf.upload(gp.to_storage(v, dtype))
    c.act = gp.ACT_NONE
    want = two_launches(gp, e, c, mid, out)
    fused(gp, e, c)
    assert np.array_equal(out.download(), want)


def test_what_one_launch_does_not_take(gp):
    """other activations, an addend, another input, a window, a table that does not fit, a body that does not take it"""
    e, c, mid, out, keep = setup(gp, "f16", (4, 14, 1024, 128, 1792), gp.ACT_RELU)
    ok = lambda: gp.lib().gp_eltwise_conv2d_supported(C.byref(e), C.byref(c))
    assert ok() == 1
    for obj, field, value in ((e, "act", gp.ACT_GELU), (e, "b", e.a), (e, "scale", None), (e, "shift", None), (e, "rows", e.rows - 1), (c, "in_", e.a), (c, "in_pix_stride", 1032),
                              (c, "stride_h", 2), (c, "pad_h", 1), (c, "out", e.a), (c, "residual", mid.ptr), (c, "tile_m", 64), (c, "variant", gp.MAT_PIPE), (c, "dtype", gp.BF16)):
        was = getattr(obj, field)
        setattr(obj, field, value)
        if field == "tile_m":
            c.tile_n = value
        assert ok() == 0, field
        with pytest.raises(gp.GpError):
            fused(gp, e, c)
        setattr(obj, field, was)
        c.tile_n = 0
    assert ok() == 1
    for dt, case in (("f16", (1, 7, 6152, 64, 6152)), ("f32", (1, 7, 3076, 64, 3076)),  # more than 24 KB of scales and shifts
                     ("f16", (16, 56, 160, 128, 160))):                                    # tiles of 128 x 128
        e, c, mid, out, keep = setup(gp, dt, case, gp.ACT_RELU)
        assert ok() == 0, case


def test_a_dense_block_shows_the_layers_it_does_not_launch(gp, monkeypatch):
    """DenseNet: the scale-shift layers in front of pointwise convolutions are not launched, their outputs are there for whoever
    reads them, and the output has the bits of a model that launches every kernel"""
    from gpreempt_amd import executor as ex_mod
    wl = "densenet201@b=2,hw=64,l1=2,l2=2,l3=2,l4=2,dtype=f16"
    x = gp.to_storage(np.random.default_rng(3).standard_normal((2, 3, 64, 64), np.float32), gp.F16)
    got = {}
    for fuse in ("1", "0"):
        monkeypatch.setenv("GPREEMPT_FUSE_LN", fuse)
        ex = ex_mod.Executor(wl, blp=True)
        stream, flag = gp.Stream(1), gp.Flag()
        ex.set_flag(flag)
        ex.set_running(True)
        ex.set_input("data", x, stream)
        ex.execute(stream)
        stream.sync()
        counts = ex.counters()
        got[fuse] = [ex.get_output(k, stream) for k in ("heads", "block2.layer2.norm1.out")] + [ex.read_storage("block3.layer1.norm1.out")]
        assert (np.array(counts) == 0).sum() >= (8 if fuse == "1" else 0) and (fuse == "1" or (np.array(counts) > 0).all())
    for a, b in zip(got["1"], got["0"]):
        assert np.array_equal(a.view(np.uint16), b.view(np.uint16)) and a.view(np.uint16).any()
