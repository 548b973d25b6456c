"""Convolutions side by side in one launch (gp_launch_conv2d_group): the bits of launches of their own, plain, eager, stopped in every
member and resumed; and the models whose kernel lists pair them up."""
import ctypes as C

import numpy as np
import pytest

from helpers import sync

pytestmark = pytest.mark.gpu
# (H, W, Cin, Cout, R, S, stride, pad_h, pad_w), one image each member: pointwise, factorised, straddling taps, ragged rows and columns
GROUPS = [
    [(17, 17, 768, 192, 1, 1, 1, 0, 0), (17, 17, 768, 160, 1, 1, 1, 0, 0)],
    [(17, 17, 160, 160, 1, 7, 1, 0, 3), (17, 17, 160, 160, 7, 1, 1, 3, 0), (17, 17, 768, 192, 1, 1, 1, 0, 0)],
    [(8, 8, 384, 384, 1, 3, 1, 0, 1), (8, 8, 384, 384, 3, 1, 1, 1, 0), (8, 8, 448, 384, 3, 3, 1, 1, 1), (8, 8, 1280, 190, 1, 1, 1, 0, 0)],
    [(17, 17, 192, 320, 3, 3, 2, 0, 0), (17, 17, 192, 192, 1, 7, 1, 0, 3)],
    [(8, 8, 384, 384, 1, 3, 1, 0, 1), (8, 8, 384, 384, 3, 1, 1, 1, 0)],
    [(9, 9, 104, 50, 3, 3, 1, 1, 1), (9, 9, 1024, 40, 1, 1, 1, 0, 0), (9, 9, 56, 33, 5, 5, 1, 2, 2)],
    [(7, 7, 8784, 40, 1, 1, 1, 0, 0), (7, 7, 968, 33, 3, 3, 1, 1, 1)],  # the deepest that fp32 takes
]


def members(gp, dt, group, images=1):
    dtype = gp.DTYPE_BY_NAME[dt]
    params, outs, keep = (gp.ConvParams * len(group))(), [], []
    for i, (H, W, Cin, Cout, R, S, stride, ph, pw) in enumerate(group):
        rng = np.random.default_rng(Cin + Cout + i)
        Ho, Wo = (H + 2 * ph - R) // stride + 1, (W + 2 * pw - S) // stride + 1
        x, w, b = (gp.DevBuf.from_array(rng.uniform(-1, 1, s).astype(np.float32), dtype) for s in ((images, H, W, Cin), (Cout, R, S, Cin), (Cout,)))
        out = gp.DevBuf((images * Ho * Wo * Cout * gp.DTYPE_SIZE[dtype] + 3) // 4 * 4)
        params[i] = gp.ConvParams(dtype=dtype, N=images, H=H, W=W, Cin=Cin, Cout=Cout, R=R, S=S, stride_h=stride, stride_w=stride, pad_h=ph, pad_w=pw, in_=x.ptr, in_pix_stride=Cin,
                                  weight=w.ptr, bias=b.ptr, out=out.ptr, out_pix_stride=Cout, act=gp.ACT_RELU)
        outs.append(out)
        keep += [x, w, b]
    return params, outs, keep


def launch(gp, params, ctx=None):
    info = gp.LaunchInfo()
    gp.check(gp.lib().gp_launch_conv2d_group(params, len(params), C.byref(ctx) if ctx is not None else None, None, C.byref(info)))
    sync(gp)
    return info


@pytest.mark.parametrize("dt,images", [("f16", 1), ("bf16", 1), ("f32", 1), ("f16", 2)])
@pytest.mark.parametrize("group", GROUPS, ids=range(len(GROUPS)))
def test_a_group_has_the_bits_of_its_members(gp, dt, images, group):
    params, outs, keep = members(gp, dt, group, images)
    supported = gp.lib().gp_conv2d_group_supported(params, len(group))
    want, tiles = [], []
    for i, out in enumerate(outs):
        out.fill32(0x7E007E00)
        tiles.append(gp.launch("gp_launch_conv2d", params[i]).total_tiles)
        sync(gp)
        want.append(out.download().copy())
    if supported != 1:  # members with different bodies, or too many tiles: refused, and nothing runs
        with pytest.raises(gp.GpError):
            launch(gp, params)
        assert all(np.array_equal(o.download(), w) for o, w in zip(outs, want))
        return

    def check():
        assert all(np.array_equal(o.download(), w) for o, w in zip(outs, want))

    def wipe():
        for o in outs:
            o.fill32(0x7E007E00)

    wipe()
    info = launch(gp, params)
    assert info.total_tiles == sum(tiles)
    check()
    flag = gp.Flag()
    for fresh, inject in [(2, -1), (1, -1)] + [(0, sum(tiles[:i])) for i in range(len(group))] + [(0, sum(tiles) - 1)]:
        st = gp.BlpState(1, flag, 32)
        wipe()
        launch(gp, params, st.ctx(fresh=fresh, inject_at=inject))
        flag.set(0)
        st.stop.upload(np.array([-1], np.int32))
        launch(gp, params, st.ctx())
        check()
        launch(gp, params, st.ctx())  # all made: nothing runs
        check()
    # the general loop: one claim counter, and fewer workgroups than tiles, each running members of different forms in turn
    for groups, workgroups in ((1, 0), (1, 3), (4, 4)):
        for inject in (-1, sum(tiles) // 2):
            st = gp.BlpState(1, flag, groups)
            wipe()
            info = launch(gp, params, st.ctx(inject_at=inject, max_workgroups=workgroups, poll_every=1))
            assert not info.fixed_claims or sum(tiles) <= 4
            flag.set(0)
            st.stop.upload(np.array([-1], np.int32))
            launch(gp, params, st.ctx(max_workgroups=workgroups))
            check()
    # a launch behind a stop leaves without writing
    st = gp.BlpState(1, flag, 32)
    st.stop.upload(np.array([0], np.int32))
    wipe()
    launch(gp, params, st.ctx(fresh=2))
    assert all((o.download().view(np.uint16) == 0x7E00).all() for o in outs)


def test_the_groups_of_the_test_above_are_groups(gp):
    for dt, group in (("f16", 0), ("f16", 1), ("f16", 2), ("bf16", 3), ("f32", 4), ("f32", 5), ("f32", 6), ("f16", 6)):
        params, outs, keep = members(gp, dt, GROUPS[group])
        assert gp.lib().gp_conv2d_group_supported(params, len(GROUPS[group])) == 1, (dt, group)
    params, outs, keep = members(gp, "f16", GROUPS[2])
    for n in (0, 1, 5):
        assert gp.lib().gp_conv2d_group_supported(params, n) == 0
    params[1].dtype = gp.BF16
    assert gp.lib().gp_conv2d_group_supported(params, 4) == 0
    params[1].dtype, params[1].variant, params[1].tile_m, params[1].tile_n = gp.F16, gp.MAT_WIDE, 32, 32
    assert gp.lib().gp_conv2d_group_supported(params, 4) == 0


@pytest.mark.parametrize("dt", ["f16", "f32"])
def test_inception_in_groups_has_the_bits_of_inception_kernel_by_kernel(gp, monkeypatch, dt):
    """... run through, stopped early and resumed, as a program and with every kernel launched"""
    from gpreempt_amd import executor as ex_mod
    x = gp.to_storage(np.random.default_rng(3).standard_normal((1, 3, 139, 139), np.float32), gp.DTYPE_BY_NAME[dt])
    got = []
    for fuse in ("1", "0"):
        monkeypatch.setenv("GPREEMPT_FUSE_LN", fuse)
        ex = ex_mod.Executor(f"inception@b=1,hw=139,dtype={dt}", blp=True)
        stream, flag = gp.Stream(1), gp.Flag()
        ex.set_flag(flag)
        ex.set_running(True)
        ex.set_input("data", x, stream)
        ex.execute(stream)
        got.append(ex.get_output("heads", stream))
        launched = (np.array(ex.counters()) > 0).sum()
        assert launched < ex.kernel_num() - 20 if fuse == "1" else launched == ex.kernel_num()
        for _ in range(3):
            ex.execute(stream)
            flag.set(1)
            stream.sync()
            flag.set(0)
            ex.resume(stream)
            got.append(ex.get_output("heads", stream))
    assert all(np.array_equal(g, got[0]) for g in got)
