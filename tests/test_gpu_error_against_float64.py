"""Errors of float32 sums against float64 (2-norm) where a kernel chooses how many additions follow one
another.  Sums of random terms, each addition rounded to nearest: an addition's relative error is
0.425 * 2^-24 rms (half a unit in the last place, uniform, over log-uniform mantissas), and n of them
in a row leave 0.425 * 2^-24 * sqrt(n / 2) of the sum."""
import re

import pytest

from tests import util

pytestmark = pytest.mark.gpu

EPS = 1e-3
ROUNDING = 0.425 * 2.0 ** -24


def _rel(a, ref):
    return float((a.double() - ref).norm() / ref.norm())


def _in_slices(rows, width):
    step = max(1, (1 << 25) // width)
    return [slice(i, min(rows, i + step)) for i in range(0, rows, step)]


@pytest.mark.parametrize("N,D,dtype", [(6000, 14000, "f32"), (20000, 9001, "f32"), (6000, 40000, "f16"), (6000, 33001, "bf16")])
def test_weight_gradients_of_many_rows_per_workgroup(N, D, dtype):
    """long_rows_bwd: a group of workgroups adds up hundreds of rows per column.  In two levels of about
    sqrt(rows) each the error is that of 2 sqrt(rows) additions (and 2 rows that are in the first chain
    before it counts), not of `rows`; the roundings of a term itself and of the final sum come on top
    as 4 more.  The factor 1.5 is the model's margin; one level exceeds it at each of these sizes."""
    import ctypes

    import torch

    from oracle import oracle as O

    capi = util.Capi(bench=True)
    text = ctypes.create_string_buffer(512)
    assert capi.L.atexn_bench_describe_bwd(0, O.DTYPE_CODE[dtype], 0, N, 1, D, text, 512) > 0
    m = re.search(rb"long_rows_bwd \(.* (\d+) groups", text.value)
    assert m, text.value
    rows = N / int(m.group(1))
    bound = 1.5 * ROUNDING * (((2 * rows ** 0.5 + 2) / 2 + 4) ** 0.5)
    assert bound < ROUNDING * ((rows / 2 + 4) ** 0.5)  # one level of additions would show
    g = torch.Generator(device="cuda").manual_seed(11)
    x = torch.empty((N, D), device="cuda", dtype=util.torch_dtype(dtype))
    dy = torch.empty_like(x)
    gamma = torch.rand(D, device="cuda", generator=g) + 0.5
    mean = torch.rand(N, device="cuda", generator=g) - 0.5
    rstd = torch.rand(N, device="cuda", generator=g) + 0.5
    dg_ref = torch.zeros(D, device="cuda", dtype=torch.float64)
    db_ref = torch.zeros_like(dg_ref)
    for s in _in_slices(N, D):
        x[s] = torch.randn(x[s].shape, device="cuda", generator=g).to(x.dtype)
        dy[s] = torch.randn(x[s].shape, device="cuda", generator=g).to(x.dtype)
        d = dy[s].double()
        db_ref += d.sum(0)
        dg_ref += (d * (x[s].double() - mean[s].double()[:, None]) * rstd[s].double()[:, None]).sum(0)
        del d
    _, dg, db = capi.ln_bwd(dy, x, gamma, mean, rstd, dtype)
    torch.cuda.synchronize()
    errors = _rel(dg, dg_ref), _rel(db, db_ref)
    print(f"LN bwd [{N}, {D}] {dtype}: {rows:.0f} rows per group, dgamma {errors[0]:.3e} dbeta {errors[1]:.3e} bound {bound:.3e}", flush=True)
    assert max(errors) <= bound


@pytest.mark.parametrize("N,C,D,dtype", [(4, 64, 50001, "f32"), (2, 64, 157685, "f32"), (1, 300, 100003, "f16"), (5, 33, 110001, "bf16"),
                                         (2, 32, 1500000, "f16"), (3, 64, 16388, "f32")])
def test_means_of_planes_over_several_workgroups(N, C, D, dtype):
    """Planes of a length that no power of two divides into (plane_fwd_ragged, and plane_fwd_single where
    a thread holds fewer vectors than it could).  From a thread's mean on there are 22 roundings on the
    way of every element: a product, six additions and a division in the wave, a product, three
    additions and a division in the workgroup, a product, six additions and a product with 1 / D (itself
    rounded) over the chunks.  Unbiased, as many leave sqrt(22) of one.  (That those of a wave or of a
    chunk average out over 8 waves or S chunks is the bound's margin.)"""
    import torch

    bound = ROUNDING * 22 ** 0.5
    capi = util.Capi()
    g = torch.Generator(device="cuda").manual_seed(12)
    x = torch.empty((N * C, D), device="cuda", dtype=util.torch_dtype(dtype))
    ref = torch.empty(N * C, device="cuda", dtype=torch.float64)
    for s in _in_slices(N * C, D):
        offset = torch.rand((x[s].shape[0], 1), device="cuda", generator=g) * 4 - 2
        x[s] = (torch.randn(x[s].shape, device="cuda", generator=g) + offset).to(x.dtype)
        ref[s] = x[s].double().mean(1)
    one, zero = torch.ones(C, device="cuda"), torch.zeros(C, device="cuda")
    _, mean, _ = capi.in_fwd(x.view(N, C, D), one, zero, EPS, dtype, True)
    torch.cuda.synchronize()
    error = _rel(mean.view(-1), ref)
    print(f"IN fwd channel-first [{N}, {C}, {D}] {dtype}: mean {error:.3e} bound {bound:.3e}", flush=True)
    assert error <= bound
