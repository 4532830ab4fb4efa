"""LayerNorm rows spread over the workgroups of an XCD (long_rows_fwd / long_rows_bwd): parity at the
edges of their chunks and routing, the same bits when every wait between workgroups runs out at
once or early (benchmark build), in-place calls, and recorded launches replayed with new data."""
import numpy as np
import pytest

from tests import util
from tests.util import TOL, assert_close

pytestmark = pytest.mark.gpu

EPS = 1e-3
DEFAULT_POLLS = 500


def _device(N, D, dtype, seed):
    import torch

    x, gamma, beta, dy = util.ln_inputs("row_mean", N, D, dtype, seed)
    return (x, gamma, beta, dy), (util.to_device(x, dtype), torch.from_numpy(gamma).cuda(),
                                  torch.from_numpy(beta).cuda(), util.to_device(dy, dtype))


def _step(capi, xd, gd, bd, dyd, dtype):
    import torch

    y, m, r = capi.ln_fwd(xd, gd, bd, EPS, dtype)
    dx, dg, db = capi.ln_bwd(dyd, xd, gd, m, r, dtype)
    torch.cuda.synchronize()
    return y, m, r, dx, dg, db


def _check(coracle, host, outs, dtype):
    x, gamma, beta, dy = host
    y, m, r, dx, dg, db = (util.to_host(t) for t in outs)
    tol = TOL[dtype]
    y_ref, m_ref, r_ref = coracle.ln_fwd(x, gamma, beta, EPS, dtype)
    assert_close(y, y_ref, tol["y"], "y")
    assert_close(m, m_ref, tol["stat"], "mean")
    assert_close(r, r_ref, tol["stat"], "inv_std")
    dx_ref, dg_ref, db_ref = coracle.ln_bwd(dy, x, gamma, m, r, dtype)
    scale = util.dx_scale(dy, np.sqrt(np.mean(gamma.astype(np.float64) ** 2)), r, dtype)
    assert_close(dx, dx_ref, tol["dx"], "dx", scale=scale)
    assert_close(dg, dg_ref, tol["dw"], "dgamma")
    assert_close(db, db_ref, tol["dw"], "dbeta")


# 4096 / 2048 columns: a chunk of one vector per thread (16-bit / float32); forward rows start above
# 32768 / 16384, backward rows above 12288 / 8192 (float32 from three rows per CU: 5632)
@pytest.mark.parametrize("N,D,dtype", [
    (1, 32769, "f16"), (7, 12289, "f16"), (9, 32776, "f16"), (130, 33001, "bf16"), (70, 36864, "bf16"),
    (64, 12296, "bf16"), (3, 262144, "f16"), (1, 100003, "f16"), (300, 20417, "f16"),
    (5, 8193, "f32"), (770, 5635, "f32"), (40, 16385, "f32"), (260, 16388, "f32"), (2, 131075, "f32"), (17, 40000, "f32"),
])
def test_rows_over_several_workgroups(coracle, N, D, dtype):
    capi = util.Capi(bench=True)
    L = capi.L
    print(f"long rows N={N} D={D} {dtype}", flush=True)
    host, dev = _device(N, D, dtype, 50)
    ref = _step(capi, *dev, dtype)
    _check(coracle, host, ref, dtype)
    try:
        for polls in (0, 2, 8):
            assert L.atexn_set_tuning(b"long_rows_polls", polls) == 0
            got = _step(capi, *dev, dtype)
            for name, a, b in zip(("y", "mean", "inv_std", "dx", "dgamma", "dbeta"), got, ref):
                assert bool((a == b).all()), f"{polls} polls: {name} differs"
        # as after a call whose waits ran out: patient waits are cut short
        assert L.atexn_set_tuning(b"long_rows_polls", DEFAULT_POLLS) == 0
        assert L.atexn_bench_mark_exchange_trouble(1) == 0
        for name, a, b in zip(("y", "mean", "inv_std", "dx", "dgamma", "dbeta"), _step(capi, *dev, dtype), ref):
            assert bool((a == b).all()), f"waits cut short: {name} differs"
    finally:
        L.atexn_set_tuning(b"long_rows_polls", DEFAULT_POLLS)
        L.atexn_bench_mark_exchange_trouble(0)


def test_in_place_rows_keep_to_one_workgroup_or_two_passes(coracle):
    import torch

    capi = util.Capi()
    host, (xd, gd, bd, dyd) = _device(20, 40001, "f16", 51)
    x_keep = xd.clone()
    y, m, r = capi.ln_fwd(xd, gd, bd, EPS, "f16", y=xd)
    dx, dg, db = capi.ln_bwd(dyd, x_keep, gd, m, r, "f16", dx=dyd)
    torch.cuda.synchronize()
    _check(coracle, host, (y, m, r, dx, dg, db), "f16")


def test_replays_of_a_recorded_launch_take_new_data():
    """Every replay draws its own tag: what an earlier replay left in the workspace is not taken
    for this one's, and each has the bits of an eager call on the same data."""
    import torch

    capi = util.Capi()
    dtype = "f16"
    _, (xd, gd, bd, dyd) = _device(24, 40008, dtype, 52)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        _step(capi, xd, gd, bd, dyd, dtype)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y, m, r = capi.ln_fwd(xd, gd, bd, EPS, dtype)
        outs = (y, m, r) + tuple(capi.ln_bwd(dyd, xd, gd, m, r, dtype))
    for replay in range(4):
        xd.copy_(torch.randn(xd.shape, device="cuda").to(xd.dtype) * (replay + 1))
        for t in outs:
            t.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip(outs, _step(capi, xd, gd, bd, dyd, dtype)):
            assert torch.equal(a, b), f"replay {replay}"
