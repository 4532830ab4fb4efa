"""LayerNorm backward of few rows in one launch (rows_bwd_pair): parity at the edges of a strip, a wave, a
workgroup and a batch of rows, tensors off every alignment, and in place on the row kernels."""
import ctypes

import numpy as np
import pytest

from oracle import oracle as O
from tests import util
from tests.util import TOL, assert_close

pytestmark = pytest.mark.gpu

EPS = 1e-3


def _describe(capi, N, D, dtype):
    text = ctypes.create_string_buffer(512)
    assert capi.L.atexn_bench_describe_bwd(0, O.DTYPE_CODE[dtype], 0, N, 1, D, text, 512) > 0
    return text.value.decode()


# strips of 4 and 8 vectors and what is left of one; rows of 1 to 2048 vectors on a wave (up to 256) and on a
# workgroup; 1, 8, 9 rows, around 64 / 128 rows at once and around a batch of 8 steps
@pytest.mark.parametrize("N,D,dtype", [
    (1, 8, "f16"), (3, 4, "f32"), (9, 9, "bf16"), (8, 33, "f16"), (7, 512, "f16"), (129, 513, "bf16"), (64, 1025, "f32"),
    (127, 2048, "f16"), (512, 2049, "f16"), (1024, 250, "bf16"), (65, 4096, "f16"), (513, 4097, "bf16"), (33, 4104, "f16"),
    (10, 8191, "f16"), (768, 8200, "f16"), (5, 16384, "bf16"), (31, 8189, "f32"), (2, 8192, "f32"),
])
def test_few_rows_in_one_launch(coracle, N, D, dtype):
    import torch

    capi = util.Capi(bench=True)
    what = _describe(capi, N, D, dtype)
    print(f"pair rows N={N} D={D} {dtype}: {what}", flush=True)
    assert what.startswith("rows_bwd_pair")
    x, gamma, beta, dy = util.ln_inputs("scaled_rows", N, D, dtype, 140)
    xd, dyd, gd = util.to_device(x, dtype), util.to_device(dy, dtype), torch.from_numpy(gamma).cuda()
    _, m, r = capi.ln_fwd(xd, gd, torch.from_numpy(beta).cuda(), EPS, dtype)
    dx_ref, dg_ref, db_ref = coracle.ln_bwd(dy, x, gamma, util.to_host(m), util.to_host(r), dtype)
    scale = util.dx_scale(dy, np.sqrt(np.mean(gamma.astype(np.float64) ** 2)), util.to_host(r), dtype)
    tol = TOL[dtype]

    def check(outs):
        dx, dg, db = (util.to_host(t) for t in outs)
        assert_close(dx, dx_ref, tol["dx"], "dx", scale=scale)
        assert_close(dg, dg_ref, tol["dw"], "dgamma")
        assert_close(db, db_ref, tol["dw"], "dbeta")

    first = capi.ln_bwd(dyd, xd, gd, m, r, dtype)
    check(first)
    moved = capi.ln_bwd(util.misalign(dyd), util.misalign(xd), util.misalign(gd), util.misalign(m), util.misalign(r), dtype)
    for a, b in zip(moved, first):
        assert bool((a == b).all())
    check(capi.ln_bwd(dyd, xd, gd, m, r, dtype, dx=dyd))  # in place: the row kernels


@pytest.mark.parametrize("N,D,dtype", [(32, 1024, "f16"), (512, 4096, "bf16"), (200, 2051, "f32")])
def test_gradients_over_the_weights_keep_the_row_kernels(N, D, dtype):
    """dgamma written over gamma (dbeta over gamma, or into its second half) or over x or dy: the bits of the row
    kernels, which write them when everything is read."""
    import torch

    capi = util.Capi(bench=True)
    L, code = capi.L, O.DTYPE_CODE[dtype]
    x, gamma, beta, dy = util.ln_inputs("plain", N, D, dtype, 141)
    xd, dyd, gd = util.to_device(x, dtype), util.to_device(dy, dtype), torch.from_numpy(gamma).cuda()
    _, m, r = capi.ln_fwd(xd, gd, torch.from_numpy(beta).cuda(), EPS, dtype)
    need = L.atexn_layer_norm_bwd_workspace_bytes(code, N, D)
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")

    def run(place):
        buf = torch.zeros(3 * D, device="cuda")
        buf[:D] = gd
        dx = torch.empty_like(xd)
        dg, db = (buf[o:o + D] for o in place)
        assert L.atexn_layer_norm_bwd(code, dyd.data_ptr(), xd.data_ptr(), buf.data_ptr(), m.data_ptr(), r.data_ptr(), N, D,
                                      dx.data_ptr(), dg.data_ptr(), db.data_ptr(), ws.data_ptr(), need,
                                      torch.cuda.current_stream().cuda_stream) == 0
        torch.cuda.synchronize()
        return dx, dg.clone(), db.clone()

    try:
        assert L.atexn_set_tuning(b"pair_rows", 0) == 0
        want = run((D, 2 * D))
    finally:
        assert L.atexn_set_tuning(b"pair_rows", 1) == 0
    print(f"dgamma / dbeta over gamma N={N} D={D} {dtype}", flush=True)
    assert not all(bool((a == b).all()) for a, b in zip(run((D, 2 * D)), want))  # (rows_bwd_pair sums differently)
    for place in ((0, D), (D, 0), (D // 2, 2 * D)):
        for name, a, b in zip(("dx", "dgamma", "dbeta"), run(place), want):
            assert bool((a == b).all()), f"{place}: {name}"
    # ... and over x and dy
    half = 2 * D if dtype != "f32" else D  # elements that D floats cover
    for over_x, over_dy in ((True, False), (False, True), (True, True)):
        ops = {True: xd.clone(), False: dyd.clone()}
        out = [ops[k].view(-1)[:half].view(torch.float32) if over else torch.empty(D, device="cuda")
               for k, over in ((True, over_x), (False, over_dy))]
        dx = torch.empty_like(xd)
        assert L.atexn_layer_norm_bwd(code, ops[False].data_ptr(), ops[True].data_ptr(), gd.data_ptr(), m.data_ptr(), r.data_ptr(),
                                      N, D, dx.data_ptr(), out[0].data_ptr(), out[1].data_ptr(), ws.data_ptr(), need,
                                      torch.cuda.current_stream().cuda_stream) == 0
        torch.cuda.synchronize()
        for name, a, b in zip(("dx", "dgamma", "dbeta"), (dx, *out), want):
            assert bool((a == b).all()), f"over x {over_x}, over dy {over_dy}: {name}"


def test_more_rows_stay_on_the_row_kernels():
    capi = util.Capi(bench=True)
    for N, D, dtype in ((1025, 64, "f16"), (513, 1024, "f16"), (769, 8192, "f16"), (513, 8192, "f32"), (8, 16392, "f16")):
        assert not _describe(capi, N, D, dtype).startswith("rows_bwd_pair"), (N, D, dtype)
