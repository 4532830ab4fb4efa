"""The channels-last kernels that hold an instance's slabs (cl_hold_fwd / cl_hold_bwd), wherever they can run
(benchmark build): parity over their kinds (registers alone, LDS too, vectors read twice), with ragged last
pixels; the same bits when every wait, or some, run out; recorded in a graph; tensors off every alignment."""
import pytest

from tests import util
from tests.test_gpu_flat_channels_last import _check, _describe, _device, _same, _step

pytestmark = pytest.mark.gpu


@pytest.fixture
def hold():
    capi = util.Capi(bench=True)
    assert capi.L.atexn_set_tuning(b"cl_hold", 2) == 0
    yield capi
    capi.L.atexn_set_tuning(b"cl_hold", 1)
    capi.L.atexn_set_tuning(b"cl_flat_polls", 300)
    capi.L.atexn_bench_mark_exchange_trouble(0)


# N, C, D, dtype, vectors of a thread that the backward reads twice.  One slab per CU or two; every kind of
# either direction; one instance and two on the chip at once, four with a second round; C off and on 16 bytes
@pytest.mark.parametrize("N,C,D,dtype,twice", [
    (1, 17, 1000003, "f16", 0), (24, 57, 9384, "f16", 0), (3, 40, 260011, "bf16", 0), (1, 300, 90011, "f16", 0),
    (2, 32, 1000000, "f16", 6), (1, 33, 1200017, "f32", 54), (4, 9, 700001, "f32", 0), (1, 512, 120001, "bf16", 30),
])
def test_instances_held_by_the_chip(hold, coracle, N, C, D, dtype, twice):
    import torch

    what = _describe(hold, N, C, D, dtype)
    print(f"hold channels-last N={N} C={C} D={D} {dtype}: {what}", flush=True)
    assert what.startswith("cl_hold_bwd") and f", {twice} read twice" in what
    host, dev = _device(N, C, D, dtype, 130)
    ref = _step(hold, *dev, dtype)
    _check(coracle, host, ref, dtype)
    for polls in (0, 2):  # all workgroups help themselves, or some do
        assert hold.L.atexn_set_tuning(b"cl_flat_polls", polls) == 0
        _same(_step(hold, *dev, dtype), ref, f"{polls} polls")
    assert hold.L.atexn_set_tuning(b"cl_flat_polls", 300) == 0
    assert hold.L.atexn_bench_mark_exchange_trouble(1) == 0  # patient waits are cut short
    _same(_step(hold, *dev, dtype), ref, "waits cut short")
    x, gamma, beta, dy = dev
    moved = _step(hold, util.misalign(x), util.misalign(gamma), util.misalign(beta), util.misalign(dy), dtype)
    _same(moved, ref, "tensors off alignment")
    torch.cuda.synchronize()


def test_hold_kernels_in_a_graph(hold):
    import torch

    N, C, D, dtype = 2, 17, 700003, "f16"
    _, dev = _device(N, C, D, dtype, 131)
    ref = _step(hold, *dev, dtype)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = _step(hold, *dev, dtype)
    for i in range(3):
        for t in out:
            t.zero_()
        graph.replay()
        torch.cuda.synchronize()
        _same(out, ref, f"replay {i}")
        _same(_step(hold, *dev, dtype), ref, "eager between replays")


def test_large_instances_are_held():
    """The product's rule, and that a call in place takes the two stages."""
    capi = util.Capi(bench=True)
    for shape in ((2, 32, 2097152, "f16"), (1, 48, 884736, "f32"), (7, 43, 83628, "bf16")):
        assert _describe(capi, *shape).startswith("cl_hold_bwd")
        assert "when dx == dy" in _describe(capi, *shape)
    for shape in ((8, 64, 16384, "f16"), (1, 32, 131072, "f16"), (64, 64, 16384, "bf16")):
        assert not _describe(capi, *shape).startswith("cl_hold_bwd")
