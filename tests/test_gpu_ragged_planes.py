"""Channel-first planes of any length over the workgroups of an XCD (plane_fwd_ragged /
plane_bwd_ragged, and the kernels of planes that do not fill their threads): parity, the same bits
when every wait runs out at once or early (benchmark build), tensors off every alignment, in place."""
import numpy as np
import pytest

from tests import util
from tests.util import TOL, assert_close

pytestmark = pytest.mark.gpu

EPS = 1e-3


def _step(capi, xd, gd, bd, dyd, dtype):
    import torch

    y, m, r = capi.in_fwd(xd, gd, bd, EPS, dtype, True)
    dx, dg, db = capi.in_bwd(dyd, xd, gd, m, r, dtype, True)
    torch.cuda.synchronize()
    return y, m, r, dx, dg, db


def _check(coracle, host, outs, dtype):
    x, gamma, beta, dy = host
    y, m, r, dx, dg, db = (util.to_host(t) for t in outs)
    tol = TOL[dtype]
    y_ref, m_ref, r_ref = coracle.in_fwd(x, gamma, beta, EPS, dtype, True)
    assert_close(y, y_ref, tol["y"], "y")
    assert_close(m, m_ref, tol["stat"], "mean")
    assert_close(r, r_ref, tol["stat"], "inv_std")
    dx_ref, dg_ref, db_ref = coracle.in_bwd(dy, x, gamma, m, r, dtype, True)
    scale = util.dx_scale(dy, np.sqrt(np.mean(gamma.astype(np.float64) ** 2)), r, dtype)
    assert_close(dx, dx_ref, tol["dx"], "dx", scale=scale)
    assert_close(dg, dg_ref, tol["dw"], "dgamma")
    assert_close(db, db_ref, tol["dw"], "dbeta")


def _device(N, C, D, dtype, seed):
    import torch

    x, gamma, beta, dy = util.in_inputs(N, C, D, dtype, True, seed)
    return (x, gamma, beta, dy), (util.to_device(x, dtype), torch.from_numpy(gamma).cuda(),
                                  torch.from_numpy(beta).cuda(), util.to_device(dy, dtype))


# the longest plane of one workgroup has 32768 / 16384 elements (16-bit / float32), of a chunk too;
# C = 8: the fold over the batch in the kernel
@pytest.mark.parametrize("N,C,D,dtype", [
    (1, 1, 32769, "f16"), (2, 8, 32775, "bf16"), (3, 5, 65537, "f16"), (2, 3, 65543, "bf16"),
    (1, 8, 98303, "f16"), (2, 8, 40000, "f16"), (1, 1, 2097151, "bf16"), (1, 2, 2097144, "f16"),
    (2, 8, 16385, "f32"), (1, 3, 32771, "f32"), (9, 1, 50001, "f32"), (1, 1, 1048575, "f32"),
])
def test_planes_of_any_length_over_several_workgroups(coracle, N, C, D, dtype):
    capi = util.Capi(bench=True)
    L = capi.L
    print(f"ragged planes N={N} C={C} D={D} {dtype}", flush=True)
    host, dev = _device(N, C, D, dtype, 60)
    ref = _step(capi, *dev, dtype)
    _check(coracle, host, ref, dtype)
    try:
        for polls in (0, 2):
            assert L.atexn_set_tuning(b"plane_single_polls", polls) == 0
            got = _step(capi, *dev, dtype)
            for name, a, b in zip(("y", "mean", "inv_std", "dx", "dgamma", "dbeta"), got, ref):
                assert bool((a == b).all()), f"{polls} polls: {name} differs"
        # as after a call whose waits ran out: patient waits are cut short
        assert L.atexn_set_tuning(b"plane_single_polls", 500) == 0
        assert L.atexn_bench_mark_exchange_trouble(1) == 0
        for name, a, b in zip(("y", "mean", "inv_std", "dx", "dgamma", "dbeta"), _step(capi, *dev, dtype), ref):
            assert bool((a == b).all()), f"waits cut short: {name} differs"
    finally:
        L.atexn_set_tuning(b"plane_single_polls", 500)
        L.atexn_bench_mark_exchange_trouble(0)


@pytest.mark.parametrize("shift_x,shift_dy", [(1, 0), (3, 3), (0, 5)])
def test_tensors_off_their_alignment(coracle, shift_x, shift_dy):
    capi = util.Capi()
    host, (xd, gd, bd, dyd) = _device(2, 3, 33333, "f16", 61)
    outs = _step(capi, util.misalign(xd, shift_x) if shift_x else xd, gd, bd,
                 util.misalign(dyd, shift_dy) if shift_dy else dyd, "f16")
    _check(coracle, host, outs, "f16")


def test_in_place(coracle):
    import torch

    capi = util.Capi()
    host, (xd, gd, bd, dyd) = _device(2, 3, 40001, "f16", 62)
    x_keep = xd.clone()
    y, m, r = capi.in_fwd(xd, gd, bd, EPS, "f16", True, y=xd)
    dx, dg, db = capi.in_bwd(dyd, x_keep, gd, m, r, "f16", True, dx=dyd)
    torch.cuda.synchronize()
    _check(coracle, host, (y, m, r, dx, dg, db), "f16")


@pytest.mark.parametrize("N,C,D", [(2, 8, 40001), (3, 5, 70003)])
def test_replays_of_a_recorded_launch_take_new_data(N, C, D):
    """Every replay draws its own tag; with the fold over the batch in the kernel (C = 8) and without."""
    import torch

    capi = util.Capi()
    dtype = "f16"
    _, (xd, gd, bd, dyd) = _device(N, C, D, dtype, 63)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        _step(capi, xd, gd, bd, dyd, dtype)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y, m, r = capi.in_fwd(xd, gd, bd, EPS, dtype, True)
        outs = (y, m, r) + tuple(capi.in_bwd(dyd, xd, gd, m, r, dtype, True))
    for replay in range(4):
        xd.copy_(torch.randn(xd.shape, device="cuda").to(xd.dtype) * (replay + 1))
        for t in outs:
            t.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip(outs, _step(capi, xd, gd, bd, dyd, dtype)):
            assert torch.equal(a, b), f"replay {replay}"
