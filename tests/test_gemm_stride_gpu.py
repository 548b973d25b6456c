"""The pipelined bodies fetch through descriptors of 2 GB (256 x 256 tiles, 16-bit tiles of 64 x 64 and less, 16-bit convolutions of whole
taps, convolutions whose K-steps straddle taps; the others by pointers) that begin at a tile's first row, and work out addresses of 64 bits
where a tile's rows span more (16-bit 256 x 256 tiles over a deep K, whose loop has no such form: the loop of the shallower ones).  Rows just inside and just outside of that span, of either operand, give the bits of packed rows, and
those the oracle's values; K with a remainder, and tiles with rows and columns past the last one."""
import numpy as np
import pytest

from helpers import rel_err, sync
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def spread(gp, rows, stride_bytes):
    """the rows, `stride_bytes` apart"""
    buf = gp.DevBuf((len(rows) - 1) * stride_bytes + rows[0].nbytes)
    for i, row in enumerate(rows):
        gp.check(gp.lib().gp_memcpy_h2d(gp.vp(buf.ptr + i * stride_bytes), row.ctypes.data_as(gp.vp), gp.C.c_size_t(row.nbytes)))
    return buf


@pytest.mark.parametrize("outside", [False, True])
@pytest.mark.parametrize("dtype_name,tile,variant,K,far_operand", [("bf16", 256, "MAT_PIPE", 2056, "A"), ("f16", 256, "MAT_PIPE", 2176, "B"), ("bf16", 256, "MAT_PIPE", 200, "A"), ("bf16", 256, "MAT_PIPE", 128, "B"), ("f32", 256, "MAT_PIPE", 68, "A"),
                                                                   ("f16", 128, "MAT_PIPE", 136, "B"), ("f32", 64, "MAT_PIPE", 36, "A"), ("bf16", 64, "MAT_PIPE_SPLITK", 72, "B")])
def test_far_rows(gp, dtype_name, tile, variant, K, far_operand, outside):
    dtype, es, vec = gp.DTYPE_BY_NAME[dtype_name], 4 if dtype_name == "f32" else 2, 4 if dtype_name == "f32" else 8
    M = N = tile + 4
    rng = np.random.default_rng(tile + K)
    A, B = (gp.to_storage(rng.uniform(-1, 1, (s, K)).astype(np.float32), dtype).view(np.uint8).reshape(s, K * es) for s in (M, N))
    dA, dB, out = gp.DevBuf.from_array(A), gp.DevBuf.from_array(B), gp.DevBuf(M * N * es)
    p = gp.GemmParams(dtype=dtype, M=M, N=N, K=K, A=dA.ptr, lda=K, B=dB.ptr, ldb=K, b_is_nk=1, C=out.ptr, ldc=N, alpha=1.0, act=gp.ACT_NONE, batch=1,
                      tile_m=tile, tile_n=tile, variant=getattr(gp, variant))
    gp.launch("gp_launch_gemm", p)
    sync(gp)
    want = out.download().copy()
    A32, B32 = (gp.from_storage(v.reshape(-1), dtype).reshape(-1, K) for v in (A, B))
    # fp32 sums of K products, the result rounded to the type: half a unit in its last place
    assert rel_err(gp.from_storage(want, dtype).reshape(M, N), O.gemm_bias_act(A32, B32, None, None, O.ACT_NONE, b_is_nk=True)) < {"f32": 1e-5, "f16": 1e-3, "bf16": 8e-3}[dtype_name]
    ld = ((1 << 31) // es - K) // tile // vec * vec + (vec if outside else 0)
    far = spread(gp, A if far_operand == "A" else B, ld * es)
    if far_operand == "A":
        p.A, p.lda = far.ptr, ld
    else:
        p.B, p.ldb = far.ptr, ld
    out.fill32(0x7FC00000)
    info = gp.launch("gp_launch_gemm", p)
    sync(gp)
    assert info.total_tiles == (-(-M // tile)) ** 2
    assert np.array_equal(out.download(), want)
    if variant == "MAT_PIPE":  # and the preemptible form
        st = gp.BlpState(1, gp.Flag(), 32)
        st.enable_checkpoints(p)
        out.fill32(0x7FC00000)
        gp.launch("gp_launch_gemm", p, st.ctx(fresh=2))
        sync(gp)
        assert np.array_equal(out.download(), want)


@pytest.mark.parametrize("dtype_name,N,H,W,Cin,Cout,R,stride,pad,tile,variant", [
    ("f16", 2, 9, 11, 64, 70, 3, 1, 1, 64, "MAT_PIPE"), ("bf16", 3, 8, 7, 128, 133, 3, 2, 1, 128, "MAT_PIPE"), ("f32", 2, 7, 9, 32, 64, 5, 1, 2, 64, "MAT_PIPE"),
    # K-steps that straddle taps: found by multiplication and through descriptors, and by division and through pointers
    ("f16", 2, 9, 11, 40, 70, 3, 1, 1, 64, "MAT_PIPE"), ("bf16", 1, 12, 10, 72, 133, 5, 2, 2, 128, "MAT_PIPE"), ("f32", 2, 7, 9, 20, 130, 3, 1, 1, 128, "MAT_PIPE"), ("f32", 1, 13, 9, 4, 40, 7, 2, 3, 64, "MAT_PIPE"),
    ("f16", 1, 12, 12, 192, 40, 1, 2, 0, 64, "MAT_PIPE_SPLITK"), ("f16", 2, 9, 5, 128, 36, 3, 1, 0, 32, "MAT_PIPE_SPLITK"), ("f32", 3, 13, 3, 64, 130, 3, 1, 1, 128, "MAT_PIPE")])
def test_far_pixels(gp, dtype_name, N, H, W, Cin, Cout, R, stride, pad, tile, variant):
    """a convolution's form for buffers of 2 GB, where K-steps lie within a tap and where they straddle taps, and the general one behind
    pixels that span more"""
    dtype, es = gp.DTYPE_BY_NAME[dtype_name], 4 if dtype_name == "f32" else 2
    rng = np.random.default_rng(H * Cin + R)
    x, w = rng.uniform(-1, 1, (N, H, W, Cin)).astype(np.float32), rng.uniform(-1, 1, (Cout, R, R, Cin)).astype(np.float32)
    dx, dw, db = (gp.DevBuf.from_array(v, dtype) for v in (x, w, rng.uniform(-1, 1, Cout).astype(np.float32)))
    Ho, Wo = (H + 2 * pad - R) // stride + 1, (W + 2 * pad - R) // stride + 1
    out = gp.DevBuf(N * Ho * Wo * Cout * es)
    p = gp.ConvParams(dtype=dtype, N=N, H=H, W=W, Cin=Cin, Cout=Cout, R=R, S=R, stride_h=stride, stride_w=stride, pad_h=pad, pad_w=pad, in_=dx.ptr, in_pix_stride=Cin,
                      weight=dw.ptr, bias=db.ptr, out=out.ptr, out_pix_stride=Cout, act=gp.ACT_RELU, tile_m=tile, tile_n=tile, variant=getattr(gp, variant))

    def bits():
        out.fill32(0x7FC00000)
        gp.launch("gp_launch_conv2d", p)
        sync(gp)
        return out.download().copy()

    packed = bits()
    stride_elems = ((1 << 31) // es // (N * H * W) // 8 + 1) * 8
    rows = gp.to_storage(x, dtype).reshape(N * H * W, Cin).view(np.uint8)
    far = spread(gp, list(rows), stride_elems * es)
    p.in_, p.in_pix_stride = far.ptr, stride_elems
    assert np.array_equal(bits(), packed)


@pytest.mark.parametrize("form", ["plain", "claims", "checkpoints"])
@pytest.mark.parametrize("dtype_name", ["f16", "bf16"])
def test_256_tiles_of_few_k_steps(gp, dtype_name, form):
    """The 16-bit 256 x 256 body asks for two K-steps ahead of the one it multiplies, also where there are fewer: from a part of one
    K-step to five, with and without a remainder, give the bits of 128 x 128 tiles (the same products in the same order), and so do both sides of the
    lines from which on a K-step is taken in phases (1024; with checkpoints 1792); tiles with one row and one column of the problem."""
    dtype = gp.DTYPE_BY_NAME[dtype_name]
    for M, N, K in [(256, 256, 8), (257, 260, 64), (300, 520, 72), (256, 512, 128), (513, 256, 136), (260, 257, 192), (256, 256, 256), (300, 300, 328),
                    (300, 257, 1016), (257, 300, 1024), (256, 260, 1032), (513, 256, 1088), (260, 300, 1784), (300, 260, 1792), (256, 513, 1800), (257, 257, 1864)]:
        rng = np.random.default_rng(M + N + K)
        dA, dB, dbias = (gp.DevBuf.from_array(O.round_to(rng.uniform(-1, 1, s).astype(np.float32), dtype_name), dtype) for s in ((M, K), (N, K), (N,)))
        outs = []
        for tile in (128, 256):
            out = gp.DevBuf(M * N * 2)
            out.fill32(0x7E007E00)
            p = gp.GemmParams(dtype=dtype, M=M, N=N, K=K, A=dA.ptr, lda=K, B=dB.ptr, ldb=K, b_is_nk=1, C=out.ptr, ldc=N, bias=dbias.ptr, alpha=0.5, act=gp.ACT_RELU,
                              batch=1, tile_m=tile, tile_n=tile, variant=gp.MAT_PIPE)
            ctx = None
            if form != "plain":
                blp = gp.BlpState(1, gp.Flag(), 32)
                if form == "checkpoints":
                    blp.enable_checkpoints(p)
                ctx = blp.ctx()
            gp.launch("gp_launch_gemm", p, ctx)
            sync(gp)
            outs.append(out.download().copy())
        assert np.array_equal(*outs), (M, N, K)
