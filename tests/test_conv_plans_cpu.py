"""Which convolutions the planner takes into one launch with others (no GPU: the plan alone)."""
import ctypes as C

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
