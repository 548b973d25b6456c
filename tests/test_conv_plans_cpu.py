"""Which convolutions the planner takes into one launch with others (no GPU: the plan alone)."""
import ctypes as C
import os
import subprocess
import sys

import pytest

from gpreempt_amd import capi as gp


def _scaled(dtype, a_stride, images=4, H=14, Cin=1024, Cout=128):
    e = gp.EltwiseParams(dtype, images * H * H, Cin, 1 << 20, a_stride, None, 0, 4096, 8192, 1 << 30, Cin, gp.ACT_RELU)
    c = gp.ConvParams(dtype=dtype, N=images, H=H, W=H, Cin=Cin, Cout=Cout, R=1, S=1, stride_h=1, stride_w=1, in_=1 << 30, in_pix_stride=Cin, weight=1 << 16, out=1 << 31, out_pix_stride=Cout)
    return C.CDLL(gp.LIB_PATH).gp_eltwise_conv2d_supported(C.byref(e), C.byref(c))


@pytest.mark.parametrize("dtype", [gp.F32, gp.F16, gp.BF16])
@pytest.mark.parametrize("a_stride,ok", [(1024, 1), (1792, 1), (512, 1), (0, 1), (-1024, 0)])
def test_a_scale_and_shift_in_front_of_a_convolution_takes_rows_that_do_not_run_backwards(dtype, a_stride, ok):
    """the element-wise kernel alone takes any distance between rows; the matrix bodies' offsets are unsigned"""
    assert _scaled(dtype, a_stride) == ok


def _conv(Cin=1280, Cout=192, H=8, dtype=gp.F16, R=1, S=1):
    return gp.ConvParams(dtype=dtype, N=1, H=H, W=H, Cin=Cin, Cout=Cout, R=R, S=S, stride_h=1, stride_w=1, pad_h=R // 2, pad_w=S // 2, in_=1 << 30, in_pix_stride=Cin, weight=1 << 16,
                         out=1 << 31, out_pix_stride=Cout)


def test_a_question_leaves_the_last_error_as_it_was():
    lib = C.CDLL(gp.LIB_PATH)
    lib.gp_last_error.restype = C.c_char_p
    assert lib.gp_launch_conv2d(None, None, None, None) == gp.OUTOFRANGE
    said = lib.gp_last_error()
    assert said
    assert _scaled(gp.F16, -1024) == 0
    two = (gp.ConvParams * 2)(_conv(), _conv(dtype=gp.F32))
    assert lib.gp_conv2d_group_supported(two, 2) == 0 and lib.gp_conv2d_group_supported(two, 5) == 0
    g = gp.GemmParams(dtype=gp.F16, M=128, N=768, K=768, A=4096, lda=768, B=8200, ldb=768, b_is_nk=1, C=12288, ldc=768, alpha=1.0, batch=1)
    assert lib.gp_gemm_ln_supported(C.byref(g)) == 0  # B is not aligned
    assert lib.gp_last_error() == said


@pytest.mark.parametrize("macs,Cin,dtype,ok", [
    ("", 2048, gp.F16, 1), ("", 17568, gp.F16, 1), ("", 17600, gp.F16, 0),  # 32 x 32 tiles: 1.8e7 from K = 17579 on
    ("", 2048, gp.F32, 1), ("", 8784, gp.F32, 1), ("", 8800, gp.F32, 0),    # 16 x 16, eight times the weight: from 8790 on
    ("1000000", 960, gp.F16, 1), ("1000000", 992, gp.F16, 0), ("1000000", 512, gp.F32, 0)])
def test_a_group_takes_no_layer_whose_tiles_are_given_up_on_a_stop(macs, Cin, dtype, ok):
    """alone such a layer looks at the stop word inside its tiles, in a group it would not (the variable is read once per process, hence the child)"""
    code = (f"import sys; sys.path.insert(0, {os.path.dirname(os.path.abspath(__file__))!r}); import ctypes as C, test_conv_plans_cpu as t; from gpreempt_amd import capi as gp; "
            f"print(C.CDLL(gp.LIB_PATH).gp_conv2d_group_supported((gp.ConvParams * 2)(*[t._conv({Cin}, 64, 7, {dtype})] * 2), 2))")
    r = subprocess.run([sys.executable, "-c", code], cwd=os.path.dirname(os.path.dirname(os.path.abspath(__file__))), capture_output=True, text=True, timeout=120,
                       env={**os.environ, "GPREEMPT_LONG_TILE_MACS": macs})
    assert r.returncode == 0 and r.stdout.strip() == str(ok), r.stdout + r.stderr


@pytest.mark.parametrize("dtype,step", [(gp.F16, 32), (gp.F32, 16)])
def test_two_layers_of_larger_tiles_are_more_than_a_group_takes(dtype, step):
    """... whatever their shape, so that a group's kernel needs only the smallest tiles"""
    lib = C.CDLL(gp.LIB_PATH)
    for H in range(1, 70):
        for columns in (1, 2, 3, 5, 8, 16, 40):
            both = [_conv(1280, step * columns, H, dtype) for _ in range(2)]
            tiles = -(-H * H // step) * columns  # of one of them
            assert lib.gp_conv2d_group_supported((gp.ConvParams * 2)(*both), 2) == (1 if 2 * tiles <= 256 else 0), (H, columns)


@pytest.mark.parametrize("dt,N,H,Cin,Cout,R,stride,tile,variant,want", [
    ("f16", 16, 224, 64, 64, 3, 1, 0, "MAT_AUTO", "pipe128x64 taps"), ("bf16", 16, 224, 8, 64, 3, 1, 0, "MAT_AUTO", "pipe128x64 straddling"),
    ("f16", 4, 224, 64, 64, 3, 1, 0, "MAT_AUTO", "pipe64 taps"), ("f32", 16, 224, 64, 64, 3, 1, 0, "MAT_AUTO", "pipe64 gathered"),
    ("f16", 16, 224, 64, 64, 3, 1, 64, "MAT_PIPE", "pipe64 taps"), ("f32", 16, 73, 80, 192, 3, 1, 0, "MAT_AUTO", "pipe128 straddling"),
    ("f16", 1, 35, 48, 64, 5, 1, 0, "MAT_AUTO", "wide32x32_16 straddling"), ("f16", 1, 35, 48, 64, 5, 1, 64, "MAT_PIPE_SPLITK", "pipe64_splitk divided"),
    ("f16", 3, 9, 23176, 64, 9, 1, 64, "MAT_PIPE", "pipe64 divided"),  # (too deep for the inverse of the channels)
    ("f16", 1, 56, 64, 256, 1, 1, 0, "MAT_AUTO", "pipe64")])
def test_the_body_that_is_named_is_the_one_that_runs(dt, N, H, Cin, Cout, R, stride, tile, variant, want):
    p = gp.ConvParams(dtype=gp.DTYPE_BY_NAME[dt], N=N, H=H, W=H, Cin=Cin, Cout=Cout, R=R, S=R, stride_h=stride, stride_w=stride, pad_h=R // 2, pad_w=R // 2, in_=4096,
                      in_pix_stride=Cin, weight=8192, bias=12288, out=16384, out_pix_stride=Cout, tile_m=tile, tile_n=tile, variant=getattr(gp, variant))
    name = C.create_string_buffer(64)
    assert C.CDLL(gp.LIB_PATH).gp_conv2d_body(C.byref(p), name, C.c_size_t(64)) == gp.SUCC
    assert name.value.decode() == want
