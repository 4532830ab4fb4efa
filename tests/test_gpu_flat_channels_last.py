"""The flat channels-last kernels (cl_flat_fwd / cl_flat_bwd), wherever they can run (benchmark build):
parity at channel counts around a period and a workgroup, ragged last pixels, one and many slabs, one and
all XCDs; the same bits when every wait, or some, run out; recorded in a graph; tensors off every alignment."""
import ctypes

import numpy as np
import pytest

from oracle import oracle as O
from tests import util
from tests.util import TOL, assert_close

pytestmark = pytest.mark.gpu

EPS = 1e-3
NAMES = ("y", "mean", "inv_std", "dx", "dgamma", "dbeta")


@pytest.fixture
def flat():
    capi = util.Capi(bench=True)
    assert capi.L.atexn_set_tuning(b"cl_flat", 2) == 0
    yield capi
    capi.L.atexn_set_tuning(b"cl_flat", 1)
    capi.L.atexn_set_tuning(b"cl_flat_polls", 300)
    capi.L.atexn_bench_mark_exchange_trouble(0)


def _describe(capi, N, C, D, dtype):
    text = ctypes.create_string_buffer(512)
    assert capi.L.atexn_bench_describe_bwd(1, O.DTYPE_CODE[dtype], 1, N, C, D, text, 512) > 0
    return text.value.decode()


def _device(N, C, D, dtype, seed):
    import torch

    host = util.in_inputs(N, C, D, dtype, False, seed)
    return host, (util.to_device(host[0], dtype), torch.from_numpy(host[1]).cuda(), torch.from_numpy(host[2]).cuda(),
                  util.to_device(host[3], dtype))


def _step(capi, x, gamma, beta, dy, dtype):
    y, m, r = capi.in_fwd(x, gamma, beta, EPS, dtype, False)
    return (y, m, r, *capi.in_bwd(dy, x, gamma, m, r, dtype, False))


def _check(coracle, host, outs, dtype):
    x, gamma, beta, dy = host
    y, m, r, dx, dg, db = (util.to_host(t) for t in outs)
    tol = TOL[dtype]
    y_ref, m_ref, r_ref = coracle.in_fwd(x, gamma, beta, EPS, dtype, False)
    assert_close(y, y_ref, tol["y"], "y")
    assert_close(m, m_ref, tol["stat"], "mean")
    assert_close(r, r_ref, tol["stat"], "inv_std")
    dx_ref, dg_ref, db_ref = coracle.in_bwd(dy, x, gamma, m, r, dtype, False)
    scale = util.dx_scale(dy, np.sqrt(np.mean(gamma.astype(np.float64) ** 2)), r, dtype)
    assert_close(dx, dx_ref, tol["dx"], "dx", scale=scale)
    assert_close(dg, dg_ref, tol["dw"], "dgamma")
    assert_close(db, db_ref, tol["dw"], "dbeta")


def _same(got, want, what):
    for name, a, b in zip(NAMES, got, want):
        assert bool((a == b).all()), f"{what}: {name} differs"


# N, C, D, dtype; C = 9, 17: periods of 8 pixels; 255 / 257: on 256 and 512 threads; 1024 halves and 511
# floats: one or two periods to a workgroup; D off the period; 1, 2, 8 to 64 and more than 64 slabs per instance
@pytest.mark.parametrize("N,C,D,dtype", [
    (3, 9, 7, "f16"), (1, 17, 1003, "bf16"), (5, 33, 2048, "f16"), (9, 17, 4097, "f16"), (8, 24, 3216, "bf16"),
    (2, 255, 777, "f16"), (2, 257, 777, "f16"), (3, 1024, 40, "f16"), (2, 511, 333, "f32"), (13, 66, 1500, "f32"),
    (1, 85, 60001, "bf16"), (16, 85, 3328, "f16"), (2, 10, 100001, "f32"), (17, 64, 2500, "f16"),
])
def test_instances_as_flat_arrays(flat, coracle, N, C, D, dtype):
    import torch

    what = _describe(flat, N, C, D, dtype)
    print(f"flat channels-last N={N} C={C} D={D} {dtype}: {what}", flush=True)
    assert what.startswith("cl_flat_bwd")
    host, dev = _device(N, C, D, dtype, 120)
    ref = _step(flat, *dev, dtype)
    _check(coracle, host, ref, dtype)
    for polls in (0, 1, 4):  # all workgroups help themselves, or some do
        assert flat.L.atexn_set_tuning(b"cl_flat_polls", polls) == 0
        _same(_step(flat, *dev, dtype), ref, f"{polls} polls")
    assert flat.L.atexn_set_tuning(b"cl_flat_polls", 300) == 0
    assert flat.L.atexn_bench_mark_exchange_trouble(1) == 0  # patient waits are cut short
    _same(_step(flat, *dev, dtype), ref, "waits cut short")
    x, gamma, beta, dy = dev
    moved = _step(flat, util.misalign(x), util.misalign(gamma), util.misalign(beta), util.misalign(dy), dtype)
    _same(moved, ref, "tensors off alignment")
    torch.cuda.synchronize()


@pytest.mark.parametrize("N,C,D,dtype", [(24, 57, 9384, "f16"), (1, 17, 200000, "bf16")])
def test_flat_kernels_in_a_graph(flat, coracle, N, C, D, dtype):
    """Recorded launches take their tag on the device: replays, with eager calls between them, have the
    eager call's bits."""
    import torch

    _, dev = _device(N, C, D, dtype, 121)
    ref = _step(flat, *dev, dtype)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = _step(flat, *dev, dtype)
    for i in range(4):
        for t in out:
            t.zero_()
        graph.replay()
        torch.cuda.synchronize()
        _same(out, ref, f"replay {i}")
        _same(_step(flat, *dev, dtype), ref, "eager between replays")


def test_drawn_classes_take_the_flat_kernels():
    """The product's rule: ragged pixels of some megabytes, and not in place."""
    capi = util.Capi(bench=True)
    assert _describe(capi, 24, 57, 5000, "f16").startswith("cl_flat_bwd")
    assert not _describe(capi, 24, 57, 800, "f16").startswith("cl_flat_bwd")
    assert not _describe(capi, 8, 64, 16384, "f16").startswith("cl_flat_bwd")


def test_flat_shape_in_place_takes_two_stages(coracle):
    import torch

    capi = util.Capi()
    N, C, D, dtype = 24, 57, 9384, "f16"
    host, (x, gamma, beta, dy) = _device(N, C, D, dtype, 122)
    y_ref, m_ref, r_ref = capi.in_fwd(x, gamma, beta, EPS, dtype, False)
    xi = x.clone()
    y, m, r = capi.in_fwd(xi, gamma, beta, EPS, dtype, False, y=xi)
    dx, dg, db = capi.in_bwd(dy, x, gamma, m, r, dtype, False, dx=dy)
    torch.cuda.synchronize()
    _check(coracle, host, (y, m, r, dx, dg, db), dtype)
