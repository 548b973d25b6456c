"""Convolutions that keep their input window in LDS (gemm_window.hpp): the bits of the body that gathers every tap, plain, preempted
and resumed."""
import ctypes as C

import numpy as np
import pytest

from helpers import sync

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", ["f16", "bf16"])
@pytest.mark.parametrize("N,H,W,Cin,Cout,R,S,tile", [
    (1, 14, 14, 256, 256, 3, 3, 32),   # ResNet's third stage
    (8, 7, 7, 512, 512, 3, 3, 32),     # tiles that span images
    (4, 14, 14, 128, 32, 3, 3, 32),    # DenseNet's growth layers
    (1, 8, 8, 448, 384, 3, 3, 32),
    (1, 17, 17, 192, 192, 1, 7, 32),   # no rows above or below
    (1, 17, 17, 128, 192, 7, 1, 32),   # ... none to the sides
    (5, 3, 5, 768, 33, 3, 3, 32),      # images smaller than a tile, ragged columns
    (1, 1, 1, 832, 40, 3, 3, 32),      # one pixel: eight taps of nine outside
    (1, 35, 3, 192, 24, 5, 3, 32),     # a narrow image, one window over most of it
    (1, 28, 28, 128, 128, 3, 3, 32),
    (1, 9, 40, 1024, 64, 3, 3, 32),    # the window does not fit: gathered
    (8, 14, 14, 256, 256, 3, 3, 64),   # tiles of 64 x 32: gathered
])
def test_a_window_gives_the_bits_of_the_gather(gp, dt, N, H, W, Cin, Cout, R, S, tile):
    dtype = gp.DTYPE_BY_NAME[dt]
    rng = np.random.default_rng(H + Cin + Cout)
    x, w = rng.uniform(-1, 1, (N, H, W, Cin + 24)).astype(np.float32), rng.uniform(-1, 1, (Cout, R, S, Cin)).astype(np.float32)
    x[:, :, :, Cin:] = np.nan  # the channels beside the slice that is read
    dx, dw, db, dr = (gp.DevBuf.from_array(v, dtype) for v in (x, w, rng.uniform(-1, 1, Cout).astype(np.float32), rng.uniform(-1, 1, (N, H, W, Cout)).astype(np.float32)))
    out = gp.DevBuf((N * H * W * Cout * 2 + 3) // 4 * 4)
    p = gp.ConvParams(dtype=dtype, N=N, H=H, W=W, Cin=Cin, Cout=Cout, R=R, S=S, stride_h=1, stride_w=1, pad_h=R // 2, pad_w=S // 2, in_=dx.ptr, in_pix_stride=Cin + 24, weight=dw.ptr,
                      bias=db.ptr, residual=dr.ptr, res_pix_stride=Cout, out=out.ptr, out_pix_stride=Cout, act=gp.ACT_RELU, tile_m=32, tile_n=32, variant=gp.MAT_WIDE)
    out.fill32(0x7E007E00)
    gp.launch("gp_launch_conv2d", p)
    sync(gp)
    want = out.download().copy()
    assert np.isfinite(gp.from_storage(want[:N * H * W * Cout * 2].copy(), dtype)).all()
    p.tile_m = p.tile_n = p.variant = 0
    name = C.create_string_buffer(64)
    gp.check(gp.lib().gp_conv2d_body(C.byref(p), name, C.c_size_t(len(name))))
    assert name.value == (b"wide64x32_16 taps" if tile == 64 else b"wide32x32_16 taps" if (H, W) == (9, 40) else b"wide32x32_16 window")
    flag = gp.Flag()
    for ctx_of in (None, lambda st: st.ctx(fresh=2), lambda st: st.ctx(inject_at=0), lambda st: st.ctx(max_workgroups=8)):
        st = gp.BlpState(1, flag, 32)
        out.fill32(0x7E007E00)
        info = gp.launch("gp_launch_conv2d", p, ctx_of(st) if ctx_of else None)
        sync(gp)
        assert info.block == 1024 and info.total_tiles == -(-N * H * W // tile) * -(-Cout // 32)
        flag.set(0)
        st.stop.upload(np.array([-1], np.int32))
        if ctx_of:
            gp.launch("gp_launch_conv2d", p, st.ctx())
            sync(gp)
        assert np.array_equal(out.download(), want)

