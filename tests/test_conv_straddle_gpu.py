"""Convolutions whose K-blocks straddle filter taps (channels no multiple of a block) on the wide and narrow bodies: the bits of the
four-wavefront split-K body, which divides for every chunk, plain, preempted and resumed."""
import numpy as np
import pytest

from helpers import sync

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", ["f16", "bf16", "f32"])
@pytest.mark.parametrize("N,H,W,Cin,Cout,R,S,stride,ph,pw", [
    (1, 17, 17, 160, 160, 1, 7, 1, 0, 3),   # Inception-v3's factorised layers
    (1, 17, 17, 160, 192, 7, 1, 1, 3, 0),
    (1, 35, 35, 48, 64, 5, 5, 1, 2, 2),
    (2, 35, 35, 96, 96, 3, 3, 1, 1, 1),
    (1, 35, 35, 288, 384, 3, 3, 2, 0, 0),
    (1, 9, 7, 24, 33, 5, 6, 1, 2, 3),       # a stage covers ten taps, rows and columns ragged, thirty taps
    (3, 6, 6, 200, 40, 3, 3, 1, 2, 2),      # more padding than the window needs
    (1, 8, 8, 72, 24, 4, 8, 2, 3, 4),       # the last of 32 taps
    (8, 14, 14, 104, 136, 3, 3, 1, 1, 1),   # tiles of 64 x 32 or 64 x 64
])
def test_blocks_that_straddle_taps(gp, dt, N, H, W, Cin, Cout, R, S, stride, ph, pw):
    dtype = gp.DTYPE_BY_NAME[dt]
    rng = np.random.default_rng(H + Cin + Cout)
    Ho, Wo = (H + 2 * ph - R) // stride + 1, (W + 2 * pw - S) // stride + 1
    x, w = rng.uniform(-1, 1, (N, H, W, Cin + 16)).astype(np.float32), rng.uniform(-1, 1, (Cout, R, S, Cin)).astype(np.float32)
    dx, dw, db = (gp.DevBuf.from_array(v, dtype) for v in (x, w, rng.uniform(-1, 1, Cout).astype(np.float32)))
    out = gp.DevBuf((N * Ho * Wo * Cout * gp.DTYPE_SIZE[dtype] + 3) // 4 * 4)
    p = gp.ConvParams(dtype=dtype, N=N, H=H, W=W, Cin=Cin, Cout=Cout, R=R, S=S, stride_h=stride, stride_w=stride, pad_h=ph, pad_w=pw, in_=dx.ptr, in_pix_stride=Cin + 16,
                      weight=dw.ptr, bias=db.ptr, out=out.ptr, out_pix_stride=Cout, act=gp.ACT_RELU, tile_m=32, tile_n=32, variant=gp.MAT_PIPE_SPLITK)
    out.fill32(0x7E007E00)
    gp.launch("gp_launch_conv2d", p)
    sync(gp)
    want = out.download().copy()
    p.tile_m = p.tile_n = p.variant = 0
    flag = gp.Flag()
    for ctx_of in (None, lambda st: st.ctx(fresh=2), lambda st: st.ctx(inject_at=0)):
        st = gp.BlpState(1, flag, 32)
        out.fill32(0x7E007E00)
        info = gp.launch("gp_launch_conv2d", p, ctx_of(st) if ctx_of else None)
        sync(gp)
        assert info.block in (512, 1024), "not a wide body"
        flag.set(0)
        st.stop.upload(np.array([-1], np.int32))
        if ctx_of:
            gp.launch("gp_launch_conv2d", p, st.ctx())
            sync(gp)
        assert np.array_equal(out.download(), want)
    for variant in (gp.MAT_WIDE, gp.MAT_WIDE8):  # asked for by name, a wide body is refused here as it always was
        if Cin % (32 if dt == "f32" else 64):
            p.tile_m = p.tile_n = 32
            p.variant = variant
            with pytest.raises(gp.GpError):
                gp.launch("gp_launch_conv2d", p)


@pytest.mark.parametrize("dt", ["f16", "bf16", "f32"])
@pytest.mark.parametrize("N,H,W,Cin,Cout,R,S,stride,ph,pw,tile", [
    (1, 20, 20, 8, 64, 3, 3, 1, 1, 1, 64),    # a first layer: two K-steps, the second one mostly past K
    (1, 41, 39, 8, 64, 7, 7, 2, 3, 3, 64),    # 49 taps
    (2, 13, 9, 40, 24, 1, 7, 1, 0, 3, 64),
    (1, 12, 10, 24, 33, 5, 6, 1, 4, 5, 64),   # windows mostly outside the image, ragged columns
    (2, 15, 15, 104, 136, 3, 3, 1, 1, 1, 128),
    (1, 517, 523, 8, 64, 3, 3, 1, 1, 1, 0),   # tiles of 128 x 64, the last one partly past the rows
    (1, 519, 521, 64, 40, 3, 3, 1, 1, 1, 0),  # ... whose K-steps lie within a tap, ragged columns
])
def test_pipelined_bodies_that_straddle_taps_or_take_tall_tiles(gp, dt, N, H, W, Cin, Cout, R, S, stride, ph, pw, tile):
    """Against fp64, plain and stopped and resumed; where the launcher picks, with the bits of 64 x 64 tiles.  The largest error is that of K
    products summed in fp32 (K roundings of half a unit of the sum of their magnitudes at most) and one rounding to the type."""
    import torch
    dtype = gp.DTYPE_BY_NAME[dt]
    rng = np.random.default_rng(H + Cin + Cout)
    Ho, Wo = (H + 2 * ph - R) // stride + 1, (W + 2 * pw - S) // stride + 1
    x, w, b = rng.uniform(-1, 1, (N, H, W, Cin + 8)).astype(np.float32), rng.uniform(-1, 1, (Cout, R, S, Cin)).astype(np.float32), rng.uniform(-1, 1, Cout).astype(np.float32)
    dx, dw, db = (gp.DevBuf.from_array(v, dtype) for v in (x, w, b))
    x, w, b = (torch.from_numpy(v.download(dtype, a.shape)).double() for v, a in ((dx, x), (dw, w), (db, b)))
    x = x[..., :Cin].permute(0, 3, 1, 2)
    conv = lambda x, w, b: torch.nn.functional.conv2d(x, w.permute(0, 3, 1, 2), b, stride, (ph, pw)).permute(0, 2, 3, 1).numpy()
    ref, size = conv(x, w, b), conv(x.abs(), w.abs(), b.abs())
    out = gp.DevBuf((N * Ho * Wo * Cout * gp.DTYPE_SIZE[dtype] + 3) // 4 * 4)
    p = gp.ConvParams(dtype=dtype, N=N, H=H, W=W, Cin=Cin, Cout=Cout, R=R, S=S, stride_h=stride, stride_w=stride, pad_h=ph, pad_w=pw, in_=dx.ptr, in_pix_stride=Cin + 8,
                      weight=dw.ptr, bias=db.ptr, out=out.ptr, out_pix_stride=Cout, act=gp.ACT_NONE, tile_m=tile, tile_n=tile, variant=gp.MAT_PIPE if tile else 0)
    out.fill32(0x7E007E00)
    info = gp.launch("gp_launch_conv2d", p)
    sync(gp)
    want = out.download().copy()
    rows = N * Ho * Wo
    assert info.total_tiles == -(-rows // (tile or (64 if dt == "f32" else 128))) * -(-Cout // (tile or 64))
    got = out.download(dtype)[: rows * Cout].reshape(ref.shape)
    eps = {"f32": 0.0, "f16": 2.0 ** -11, "bf16": 2.0 ** -8}[dt]
    assert (np.abs(got - ref) <= R * S * Cin * 2.0 ** -24 * size * 2 + eps * np.abs(ref) * 1.01).all()
    flag = gp.Flag()
    st = gp.BlpState(1, flag, 32)
    out.fill32(0x7E007E00)
    gp.launch("gp_launch_conv2d", p, st.ctx(inject_at=0))
    sync(gp)
    flag.set(0)
    st.clear_stop()
    gp.launch("gp_launch_conv2d", p, st.ctx())
    sync(gp)
    assert np.array_equal(out.download(), want)
    if not tile:
        p.tile_m = p.tile_n = 64
        p.variant = gp.MAT_PIPE
        out.fill32(0x7E007E00)
        gp.launch("gp_launch_conv2d", p)
        sync(gp)
        assert np.array_equal(out.download(), want)
