"""Which GEMMs and convolutions the planner accepts around the 2 GB that a buffer descriptor spans (no GPU: the plan alone)."""
import ctypes as C

import pytest

from gpreempt_amd import capi as gp


def _rc(params):
    lib = C.CDLL(gp.LIB_PATH)
    fn = lib.gp_conv_ckpt_bytes if isinstance(params, gp.ConvParams) else lib.gp_gemm_ckpt_bytes
    n = C.c_size_t(0)
    return fn(C.byref(params), C.byref(n))


def _gemm(dtype, M, N, K, lda, ldb, variant, tm, tn):
    return gp.GemmParams(dtype=dtype, M=M, N=N, K=K, A=4096, lda=lda, B=8192, ldb=ldb, b_is_nk=1, C=12288, ldc=N, alpha=1.0, batch=1, tile_m=tm, tile_n=tn, variant=variant)


@pytest.mark.parametrize("dtype", [gp.F32, gp.F16, gp.BF16])
@pytest.mark.parametrize("variant,tm,tn", [(gp.MAT_WIDE, 32, 32), (gp.MAT_WIDE8, 32, 32), (gp.MAT_WIDE, 64, 32), (gp.MAT_WIDE8, 64, 64)])
@pytest.mark.parametrize("bytes_a,bytes_b", [(1 << 20, 1 << 20), (2 << 30, 1 << 20), (1 << 20, 5 << 30), (3 << 30, 3 << 30)])
def test_a_wide_variant_takes_operands_of_any_size(dtype, variant, tm, tn, bytes_a, bytes_b):
    M = N = 64
    es = gp.DTYPE_SIZE[dtype]
    assert _rc(_gemm(dtype, M, N, 512, max(512, bytes_a // (es * M)), max(512, bytes_b // (es * N)), variant, tm, tn)) == gp.SUCC


def test_what_a_wide_variant_refuses_is_still_refused():
    assert _rc(_gemm(gp.F16, 64, 64, 512, 512, 512, gp.MAT_WIDE, 128, 128)) == gp.OUTOFRANGE
    assert _rc(_gemm(gp.F16, 64, 64, 512, 1 << 25, 512, gp.MAT_WIDE, 32, 64)) == gp.OUTOFRANGE
    p = _gemm(gp.F16, 64, 64, 512, 512, 512, gp.MAT_WIDE, 32, 32)
    p.b_is_nk = 0
    assert _rc(p) == gp.OUTOFRANGE


@pytest.mark.parametrize("images,rc", [(1, gp.SUCC), (1200, gp.SUCC)])
def test_wide_convolution_over_two_gigabytes_of_images(images, rc):
    p = gp.ConvParams(dtype=gp.F16, N=images, H=112, W=112, Cin=128, Cout=64, R=3, S=3, stride_h=1, stride_w=1, pad_h=1, pad_w=1, in_=4096, in_pix_stride=128,
                      weight=8192, out=12288, out_pix_stride=64, tile_m=32, tile_n=32, variant=gp.MAT_WIDE)
    assert _rc(p) == rc


@pytest.mark.parametrize("dtype", [gp.F32, gp.F16, gp.BF16])
@pytest.mark.parametrize("channels", [21760, 21888, 65536])
def test_wide_convolution_of_any_number_of_channels(dtype, channels):
    """(K + 1) * Cin passes 2^32 between the first two: only blocks that straddle taps divide by the channels"""
    p = gp.ConvParams(dtype=dtype, N=1, H=5, W=5, Cin=channels, Cout=32, R=3, S=3, stride_h=1, stride_w=1, pad_h=1, pad_w=1, in_=4096, in_pix_stride=channels,
                      weight=8192, out=12288, out_pix_stride=32, tile_m=32, tile_n=32, variant=gp.MAT_WIDE)
    assert _rc(p) == gp.SUCC
    p.Cin = p.in_pix_stride = channels + 8  # blocks that straddle taps: a wide body asked for by name is refused, as ever
    assert _rc(p) == gp.OUTOFRANGE


@pytest.mark.parametrize("ldb", [768, 1 << 22, (1 << 24) - 8])
def test_layernorm_prologue_over_any_number_of_rows_of_b(ldb):
    """the buffer starts at the tile's first row of B, so only a tile's rows have to fit"""
    p = _gemm(gp.F16, 128, 3072, 768, 768, ldb, gp.MAT_AUTO, 0, 0)
    p.ln_gamma, p.ln_beta, p.ln_out, p.ln_eps = 16384, 20480, 24576, 1e-5
    assert _rc(p) == gp.SUCC
