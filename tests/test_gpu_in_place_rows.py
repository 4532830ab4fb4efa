"""LayerNorm rows whose y == x (dx == dy) calls, and whose calls in a process with ATEXN_NO_EXCHANGE, take
other kernels than the rest: the backward for rows of one workgroup (rows_bwd_resident with four vectors
per lane, rows_bwd_lds) and the 2-D tiles.  Here they run with inputs and outputs apart, through the
benchmark build with long_rows off, at the edges of their ranges and in the roles that the one-launch
kernels have taken over from them elsewhere in these tests."""
import ctypes
import os
import subprocess
import sys

import pytest

from tests import test_gpu_conditioning, test_gpu_graph_capture, test_gpu_nonfinite, util
from tests.test_gpu_layer_norm import run_case

pytestmark = pytest.mark.gpu


@pytest.fixture
def capi(monkeypatch):
    bench = util.Capi(bench=True)
    assert bench.L.atexn_set_tuning(b"long_rows", 0) == 0
    monkeypatch.setattr(util, "Capi", lambda bench_=False, **kw: bench)
    yield bench
    assert bench.L.atexn_set_tuning(b"long_rows", 1) == 0


def _describe(capi, N, D, dtype):
    from oracle import oracle as O

    text = ctypes.create_string_buffer(512)
    assert capi.L.atexn_bench_describe_bwd(0, O.DTYPE_CODE[dtype], 0, N, 1, D, text, 512) > 0
    return text.value.decode()


@pytest.mark.parametrize("kernel,N,D,dtype", [
    ("rows_bwd_resident", 300, 16384, "f16"), ("rows_bwd_resident", 65, 12289, "bf16"), ("rows_bwd_resident", 770, 8192, "f32"),
    ("rows_bwd_resident", 770, 5635, "f32"),
    ("rows_bwd_lds", 600, 18432, "f16"), ("rows_bwd_lds", 257, 17001, "bf16"), ("rows_bwd_lds", 1, 20416, "f16"),
    ("rows_bwd_lds", 300, 9000, "f32"), ("rows_bwd_lds", 40, 16384, "f32"), ("rows_bwd_lds", 7, 8193, "f32"),
    ("tile_bwd_sums", 300, 20417, "f16"), ("tile_bwd_sums", 6, 70001, "f16"), ("tile_bwd_sums", 1, 100003, "bf16"),
    ("tile_bwd_sums", 40, 16385, "f32"), ("tile_bwd_sums", 130, 33001, "f32"), ("tile_bwd_sums", 3, 262147, "f32"),
])
def test_parity(capi, coracle, kernel, N, D, dtype):
    assert _describe(capi, N, D, dtype).startswith(kernel)
    run_case(capi, coracle, "row_mean", N, D, dtype, 70)


@pytest.mark.parametrize("N,D,row,col", [(5, 70001, 2, 70000), (5, 70001, 4, 8191), (9, 18433, 8, 18432)])
def test_a_non_finite_row_stays_alone(capi, N, D, row, col):
    test_gpu_nonfinite.test_layer_norm_row_isolation(N, D, row, col, float("nan"))


def test_outlier_samples_in_tiles(capi, coracle):
    test_gpu_conditioning.test_outlier_samples(coracle, "LayerNorm rows over several workgroups", 1000.0)


@pytest.mark.parametrize("case", ["ln_tiles", "ln_accumulators_in_lds"])
def test_replays_match_eager_calls(capi, case):
    test_gpu_graph_capture._replay_matches_eager(capi, case)


_DIGEST_SCRIPT = r"""
import hashlib, sys
import torch
sys.path.insert(0, sys.argv[1])
from tests import util
capi = util.Capi(bench=sys.argv[2] == "bench")
if sys.argv[2] == "bench":
    for name in (b"long_rows", b"plane_single"):
        assert capi.L.atexn_set_tuning(name, 0) == 0
h = hashlib.sha256()
for kind, shape, W in (("ln", (300, 18433), 18433), ("ln", (6, 70001), 70001), ("cf", (2, 3, 40001), 3), ("cf", (8, 64, 36865), 64)):
    gen = torch.Generator(device="cuda").manual_seed(99 + W)
    x = (torch.randn(shape, device="cuda", generator=gen) + 0.5).half()
    dy = torch.randn(shape, device="cuda", generator=gen).half()
    gamma = torch.rand(W, device="cuda", generator=gen) + 0.5
    beta = torch.randn(W, device="cuda", generator=gen)
    if kind == "ln":
        y, m, r = capi.ln_fwd(x, gamma, beta, 1e-3, "f16")
        dx, dg, db = capi.ln_bwd(dy, x, gamma, m, r, "f16")
    else:
        y, m, r = capi.in_fwd(x, gamma, beta, 1e-3, "f16", True)
        dx, dg, db = capi.in_bwd(dy, x, gamma, m, r, "f16", True)
    torch.cuda.synchronize()
    for t in (y, m, r, dx, dg, db):
        h.update(t.contiguous().view(torch.uint8).cpu().numpy().tobytes())
    print("done", kind, shape, flush=True)
print("DIGEST", h.hexdigest())
"""


def test_no_exchange_keeps_long_rows_and_ragged_planes_on_them():
    """ATEXN_NO_EXCHANGE=1 and the product library against the benchmark build with the one-launch kernels
    switched off, each in a child process: the same bits."""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

    def digest(flavour, value):
        out = subprocess.run([sys.executable, "-c", _DIGEST_SCRIPT, root, flavour], env=dict(os.environ, ATEXN_NO_EXCHANGE=value),
                             capture_output=True, text=True, timeout=300)
        assert out.returncode == 0, out.stderr[-2000:]
        return [line for line in out.stdout.splitlines() if line.startswith("DIGEST ")]

    off_by_env, off_by_switch = digest("product", "1"), digest("bench", "0")
    assert len(off_by_env) == 1 and off_by_env == off_by_switch
    assert off_by_env != digest("product", "0")  # (the one-launch kernels add in another order)


def test_in_place_calls_take_the_same_kernels():
    """... as the switch: the bits of dx over dy and of y over x are those with long_rows off."""
    import torch

    product, bench = util.Capi(), util.Capi(bench=True)
    x, gamma, beta, dy = util.ln_inputs("row_mean", 40, 40001, "f16", 71)
    xd, dyd, gd, bd = util.to_device(x, "f16"), util.to_device(dy, "f16"), torch.from_numpy(gamma).cuda(), torch.from_numpy(beta).cuda()
    assert bench.L.atexn_set_tuning(b"long_rows", 0) == 0
    try:
        y, m, r = bench.ln_fwd(xd, gd, bd, 1e-3, "f16")
        apart = (y, m, r) + tuple(bench.ln_bwd(dyd, xd, gd, m, r, "f16"))
        torch.cuda.synchronize()
    finally:
        assert bench.L.atexn_set_tuning(b"long_rows", 1) == 0
    x2, dy2 = xd.clone(), dyd.clone()
    dx, dg, db = product.ln_bwd(dy2, xd, gd, m, r, "f16", dx=dy2)
    y2, m2, r2 = product.ln_fwd(x2, gd, bd, 1e-3, "f16", y=x2)
    torch.cuda.synchronize()
    for name, a, b in zip(("y", "mean", "inv_std", "dx", "dgamma", "dbeta"), (y2, m2, r2, dx, dg, db), apart):
        assert torch.equal(a, b), name
