"""The fp32 bodies with 16 x 16 and 32 x 16 tiles (gemm_narrow.hpp) against the four-wavefront split-K body, whose sums they make in
the same order: equal bits, plain, preempted and resumed."""
import numpy as np
import pytest

from helpers import rel_err, sync
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def launches(gp, name, p, out, want):
    """plainly, as an eager first launch, and stopped at the first claim and resumed"""
    out.fill32(0x7FC00000)
    info = gp.launch(name, p)
    sync(gp)
    assert np.array_equal(out.download(), want)
    flag = gp.Flag()
    for fresh, inject in ((2, -1), (0, 0)):
        st = gp.BlpState(1, flag, 32)
        st.enable_done_counters()
        out.fill32(0x7FC00000)
        gp.launch(name, p, st.ctx(fresh=fresh, inject_at=inject))
        sync(gp)
        flag.set(0)
        st.stop.upload(np.array([-1], np.int32))
        gp.launch(name, p, st.ctx(done_launches=1))
        sync(gp)
        assert np.array_equal(out.download(), want)
    return info


@pytest.mark.parametrize("M,N,K,tile", [(1, 16, 512, 16), (17, 33, 516, 16), (49, 512, 2048, 16), (196, 250, 1028, 16), (1, 1000, 2048, 16), (64, 1024, 25088, 16),
                                        (100, 1000, 768, 32), (392, 256, 2304, 32), (33, 2040, 772, 32)])
def test_narrow_gemm_has_the_bits_of_the_split_k_body(gp, M, N, K, tile):
    rng = np.random.default_rng(M + N + K)
    A, B = (rng.uniform(-1, 1, s).astype(np.float32) for s in ((M, K), (N, K)))
    bias, res = rng.uniform(-1, 1, N).astype(np.float32), rng.uniform(-1, 1, (M, N)).astype(np.float32)
    dA, dB, db, dr = (gp.DevBuf.from_array(v, gp.F32) for v in (A, B, bias, res))
    out = gp.DevBuf(M * N * 4)
    p = gp.GemmParams(dtype=gp.F32, M=M, N=N, K=K, A=dA.ptr, lda=K, B=dB.ptr, ldb=K, b_is_nk=1, C=out.ptr, ldc=N, bias=db.ptr, residual=dr.ptr, alpha=1.0, act=gp.ACT_RELU, batch=1,
                      tile_m=32, tile_n=32, variant=gp.MAT_PIPE_SPLITK)
    gp.launch("gp_launch_gemm", p)
    sync(gp)
    want = out.download().copy()
    assert rel_err(gp.from_storage(want, gp.F32).reshape(M, N), O.gemm_bias_act(A, B, bias, res, O.ACT_RELU, b_is_nk=True)) < 1e-4
    p.tile_m = p.tile_n = p.variant = 0
    info = launches(gp, "gp_launch_gemm", p, out, want)
    assert info.total_tiles == -(-M // tile) * -(-N // 16)


@pytest.mark.parametrize("N,H,W,Cin,Cout,R,stride,pad,tile", [(1, 7, 7, 512, 512, 3, 1, 1, 16), (1, 14, 14, 256, 256, 3, 1, 1, 16), (1, 9, 5, 64, 24, 5, 2, 2, 16), (3, 8, 8, 96, 40, 3, 1, 0, 16),
                                                              (1, 28, 28, 128, 128, 3, 1, 1, 32), (2, 17, 17, 160, 160, 3, 1, 1, 32), (1, 15, 15, 1024, 136, 1, 2, 0, 16)])
def test_narrow_convolution_has_the_bits_of_the_split_k_body(gp, N, H, W, Cin, Cout, R, stride, pad, tile):
    rng = np.random.default_rng(H + Cin + Cout)
    Ho, Wo = (H + 2 * pad - R) // stride + 1, (W + 2 * pad - R) // stride + 1
    x, w = rng.uniform(-1, 1, (N, H, W, Cin + 8)).astype(np.float32), rng.uniform(-1, 1, (Cout, R, R, Cin)).astype(np.float32)
    dx, dw, db = (gp.DevBuf.from_array(v, gp.F32) for v in (x, w, rng.uniform(-1, 1, Cout).astype(np.float32)))
    out = gp.DevBuf(N * Ho * Wo * Cout * 4)
    p = gp.ConvParams(dtype=gp.F32, N=N, H=H, W=W, Cin=Cin, Cout=Cout, R=R, S=R, stride_h=stride, stride_w=stride, pad_h=pad, pad_w=pad, in_=dx.ptr, in_pix_stride=Cin + 8,
                      weight=dw.ptr, bias=db.ptr, out=out.ptr, out_pix_stride=Cout, act=gp.ACT_RELU, tile_m=32, tile_n=32, variant=gp.MAT_PIPE_SPLITK)
    gp.launch("gp_launch_conv2d", p)
    sync(gp)
    want = out.download().copy()
    p.tile_m = p.tile_n = p.variant = 0
    info = launches(gp, "gp_launch_conv2d", p, out, want)
    assert info.total_tiles == -(-N * Ho * Wo // tile) * -(-Cout // 16)
