"""The kernels whose workgroups exchange results, beside a kernel that holds whole CUs.

A bounded busy kernel of the benchmark build (atexn_bench_occupy: 1024 threads and nearly all of
a CU's LDS per workgroup, gone after 20 ms at the latest) takes 192 of the 256 CUs on a second
stream; the InstanceNorm calls that run meanwhile find fewer places on an XCD than an instance has
slabs (a plane has chunks), so their waits run out for real: workgroups give up, claim and compute
what is missing, record the vain wait, and later waits are cut short.  Whatever the timing, the
outputs must have the bits of a run on the GPU alone."""
import os

import numpy as np
import pytest

from tests import util

pytestmark = pytest.mark.gpu

EPS = 1e-3
# random shapes beside the occupier; a longer sweep: ATEXN_SHARED_SEEDS=1000 python -m pytest tests/test_gpu_shared_gpu.py
N_SEEDS = int(os.environ.get("ATEXN_SHARED_SEEDS", "32"))


def _bits(t):
    import torch

    return t.view(torch.uint8)


@pytest.mark.parametrize("N,C,S,cf", [(8, 64, 16384, False), (16, 64, 16384, False), (2, 16, 2097152, True),
                                      (4, 32, 262144, True)])
def test_results_do_not_depend_on_who_else_runs(N, C, S, cf):
    import torch

    capi = util.Capi(bench=True)
    L = capi.L
    shape = (N, C, S) if cf else (N, S, C)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(77)
    x = torch.randn(shape, device="cuda", generator=gen).half()
    dy = torch.randn(shape, device="cuda", generator=gen).half()
    gamma = torch.rand(C, device="cuda", generator=gen) + 0.5
    beta = torch.randn(C, device="cuda", generator=gen) * 0.1
    side = torch.cuda.Stream()

    def run():
        y, m, r = capi.in_fwd(x, gamma, beta, EPS, "f16", cf)
        dx, dg, db = capi.in_bwd(dy, x, gamma, m, r, "f16", cf)
        return y, m, r, dx, dg, db

    alone = run()
    torch.cuda.synchronize()
    names = ("y", "mean", "inv_std", "dx", "dgamma", "dbeta")
    assert L.atexn_bench_mark_exchange_trouble(0) == 0
    recorded = 0
    try:
        for rep in range(4):
            torch.cuda.synchronize()
            assert L.atexn_bench_occupy(192, 20.0, side.cuda_stream) == 0
            torch.cuda._sleep(400000)  # the occupier gets its CUs first
            shared = run()
            torch.cuda.synchronize()
            for n_, a, b in zip(names, alone, shared):
                assert torch.equal(_bits(a), _bits(b)), f"run {rep} beside the occupier differs in {n_}"
            age = L.atexn_bench_exchange_trouble_age()
            recorded += 0 <= age < 64
    finally:
        torch.cuda.synchronize()
        L.atexn_bench_mark_exchange_trouble(0)
    # (how often a wait really ran out depends on where the occupier's workgroups landed: reported,
    # not required)
    print(f"IN N={N} C={C} spatial={S} {'channel-first' if cf else 'channels-last'}: "
          f"{recorded} of 4 runs beside the occupier recorded a wait that ran out", flush=True)


@pytest.mark.parametrize("kind,shape,dtype", [("ln", (300, 40001), "f16"), ("ln", (30, 200000), "bf16"), ("ln", (20, 60001), "f32"),
                                              ("cf", (2, 8, 300001), "f16"), ("cf", (1, 8, 1500001), "f16"), ("cf", (2, 3, 700001), "f32")])
def test_long_rows_and_ragged_planes_beside_the_occupier(kind, shape, dtype):
    """LayerNorm rows over several workgroups, one row after another, and planes of any length: on fewer
    workgroups than an XCD still has places for, and on more, where waits run out."""
    import torch

    capi = util.Capi(bench=True)
    L = capi.L
    gen = torch.Generator(device="cuda").manual_seed(78)
    x = torch.randn(shape, device="cuda", generator=gen).to(util.torch_dtype(dtype))
    dy = torch.randn(shape, device="cuda", generator=gen).to(util.torch_dtype(dtype))
    width = shape[1]
    gamma = torch.rand(width, device="cuda", generator=gen) + 0.5
    beta = torch.randn(width, device="cuda", generator=gen) * 0.1
    side = torch.cuda.Stream()
    print(kind, shape, dtype, flush=True)

    def run():
        if kind == "ln":
            y, m, r = capi.ln_fwd(x, gamma, beta, EPS, dtype)
            return (y, m, r) + tuple(capi.ln_bwd(dy, x, gamma, m, r, dtype))
        y, m, r = capi.in_fwd(x, gamma, beta, EPS, dtype, True)
        return (y, m, r) + tuple(capi.in_bwd(dy, x, gamma, m, r, dtype, True))

    assert L.atexn_bench_mark_exchange_trouble(0) == 0
    alone = run()
    recorded = 0
    try:
        for wgs in (192, 128):
            for rep in range(2):
                torch.cuda.synchronize()
                assert L.atexn_bench_occupy(wgs, 20.0, side.cuda_stream) == 0
                torch.cuda._sleep(400000)  # the occupier gets its CUs first
                shared = run()
                torch.cuda.synchronize()
                for n_, a, b in zip(("y", "mean", "inv_std", "dx", "dgamma", "dbeta"), alone, shared):
                    assert torch.equal(_bits(a), _bits(b)), f"beside {wgs} occupied CUs, run {rep}: {n_} differs"
                age = L.atexn_bench_exchange_trouble_age()
                recorded += 0 <= age < 64
    finally:
        torch.cuda.synchronize()
        L.atexn_bench_mark_exchange_trouble(0)
    print(f"{recorded} of 4 runs beside the occupier recorded a wait that ran out", flush=True)


@pytest.mark.parametrize("seed", range(N_SEEDS))
def test_random_shapes_beside_the_occupier(seed):
    """Shapes of every kernel family that exchanges results (and a few that do not), in the three
    dtypes and both layouts: beside an occupier of 192 and of 128 CUs, the bits of a run alone."""
    import torch

    capi = util.Capi(bench=True)
    L = capi.L
    rng = np.random.Generator(np.random.PCG64(9000 + seed))
    cf = bool(rng.integers(0, 2))
    dtype = ["f16", "bf16", "f32"][int(rng.integers(0, 3))]
    if cf:
        N = int(rng.integers(1, 9))
        C = int(rng.choice([1, 3, 8, 16, 24, 32, 64]))
        S = int(rng.choice([40000, 65536, 100000, 131072, 262144, 524288, 1048576, 300008]))
        if N * C * S > 40_000_000:
            S = max(40000, 40_000_000 // (N * C) // 8 * 8)
    else:
        N = int(rng.integers(1, 40))
        C = int(rng.choice([8, 16, 24, 32, 48, 64, 96, 128, 256]))
        S = int(rng.choice([1024, 2000, 4096, 5000, 8192, 16384, 20000]))
        if N * C * S > 40_000_000:
            N = max(1, 40_000_000 // (C * S))
    shape = (N, C, S) if cf else (N, S, C)
    tdt = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}[dtype]
    gen = torch.Generator(device="cuda")
    gen.manual_seed(1000 + seed)
    x = torch.randn(shape, device="cuda", generator=gen).to(tdt)
    dy = torch.randn(shape, device="cuda", generator=gen).to(tdt)
    gamma = torch.rand(C, device="cuda", generator=gen) + 0.5
    beta = torch.randn(C, device="cuda", generator=gen) * 0.1
    side = torch.cuda.Stream()
    print(f"IN {shape} {dtype} {'channel-first' if cf else 'channels-last'}", flush=True)

    def run():
        y, m, r = capi.in_fwd(x, gamma, beta, EPS, dtype, cf)
        dx, dg, db = capi.in_bwd(dy, x, gamma, m, r, dtype, cf)
        torch.cuda.synchronize()
        return y, m, r, dx, dg, db

    assert L.atexn_bench_mark_exchange_trouble(0) == 0
    alone = run()
    try:
        for wgs in (192, 128):
            for rep in range(2):
                torch.cuda.synchronize()
                assert L.atexn_bench_occupy(wgs, 6.0, side.cuda_stream) == 0
                torch.cuda._sleep(300000)
                shared = run()
                for n_, a, b in zip(("y", "mean", "inv_std", "dx", "dgamma", "dbeta"), alone, shared):
                    assert torch.equal(_bits(a), _bits(b)), f"beside {wgs} occupied CUs, run {rep}: {n_} differs"
    finally:
        torch.cuda.synchronize()
        L.atexn_bench_mark_exchange_trouble(0)


def _median_us(call, before, reps=7):
    """Median duration of single calls behind a busy stretch of the stream, the first left out."""
    import torch

    times = []
    for _ in range(reps):
        torch.cuda.synchronize()
        before()
        torch.cuda._sleep(400000)
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record()
        call()
        e1.record()
        torch.cuda.synchronize()
        times.append(e0.elapsed_time(e1) * 1e3)
    return float(np.median(times[1:]))


def _stream_beside(L):
    """A stream whose work runs beside the current stream's (streams share a few hardware queues)."""
    import torch

    word = torch.zeros(1, device="cuda")
    for _ in range(16):
        side = torch.cuda.Stream()
        torch.cuda.synchronize()
        assert L.atexn_bench_occupy(1, 5.0, side.cuda_stream) == 0
        over, here = torch.cuda.Event(), torch.cuda.Event()
        over.record(side)
        word.add_(1.0)
        here.record()
        here.synchronize()
        beside = not over.query()
        torch.cuda.synchronize()
        if beside:
            return side
    raise AssertionError("no stream runs beside the current one")


def _channels_last_calls(capi, N, S, C, dtype):
    import torch

    gen = torch.Generator(device="cuda").manual_seed(79)
    x, dy = (torch.randn((N, S, C), device="cuda", generator=gen).to(util.torch_dtype(dtype)) for _ in range(2))
    gamma = torch.rand(C, device="cuda", generator=gen) + 0.5
    beta = torch.randn(C, device="cuda", generator=gen) * 0.1
    _, m, r = capi.in_fwd(x, gamma, beta, EPS, dtype, False)
    return (lambda: capi.in_fwd(x, gamma, beta, EPS, dtype, False),
            lambda: capi.in_bwd(dy, x, gamma, m, r, dtype, False))


# held instances one and two at a time, flat ones on one XCD each and over all of them
HELD_AND_FLAT = [(2, 2097152, 32, "f16"), (8, 524288, 32, "f16"), (1, 385517, 144, "f32"), (36, 36288, 29, "bf16"),
                 (1, 598464, 17, "f16")]


@pytest.mark.parametrize("N,S,C,dtype", HELD_AND_FLAT)
def test_held_and_flat_instances_beside_the_occupier(N, S, C, dtype):
    """One CU taken is enough for held instances never to be on the chip together.  The bits of a run alone; and
    the workgroups that are there share out what is missing in at most three times the duration of the slab
    kernels, which need no company (each walking through an instance's slabs on its own: 5 to 10 times)."""
    import torch

    capi = util.Capi(bench=True)
    L = capi.L
    calls = _channels_last_calls(capi, N, S, C, dtype)
    side = _stream_beside(L)
    alone = [call() for call in calls]
    torch.cuda.synchronize()
    switches = (b"cl_hold", b"cl_flat", b"cl_single")
    try:
        assert L.atexn_bench_mark_exchange_trouble(0) == 0
        for wgs in (1, 192):
            def occupy():
                assert L.atexn_bench_occupy(wgs, 8.0, side.cuda_stream) == 0

            for what, call, want in zip(("forward", "backward"), calls, alone):
                for _ in range(2):
                    torch.cuda.synchronize()
                    occupy()
                    torch.cuda._sleep(400000)  # the occupier gets its CUs first
                    got = call()
                    torch.cuda.synchronize()
                    for a, b in zip(got, want):
                        assert torch.equal(_bits(a), _bits(b)), f"{what} beside {wgs} occupied CUs differs"
                shared = _median_us(call, occupy)
                for s in switches:
                    assert L.atexn_set_tuning(s, 0) == 0
                slabs = _median_us(call, occupy)
                for s in switches:
                    assert L.atexn_set_tuning(s, 1) == 0
                print(f"{what} [{N}, {S}, {C}] {dtype} beside {wgs}: {shared:.1f} us, slab kernels {slabs:.1f} us", flush=True)
                assert shared < 3.0 * slabs + 20.0, f"{what} beside {wgs} occupied CUs"
    finally:
        torch.cuda.synchronize()
        for s in switches:
            L.atexn_set_tuning(s, 1)
        L.atexn_bench_mark_exchange_trouble(0)


@pytest.mark.parametrize("N,S,C,dtype", HELD_AND_FLAT)
def test_waits_cut_short_find_peers_that_are_running(N, S, C, dtype):
    """After a wait that ran out, on a GPU that is free again: slabs of hundreds of KB end microseconds apart,
    and a wait cut short still lasts that long (or every workgroup redoes its peers' work: 4 to 6 times the
    duration, where 1.4 is allowed)."""
    capi = util.Capi(bench=True)
    calls = _channels_last_calls(capi, N, S, C, dtype)
    try:
        for what, call in zip(("forward", "backward"), calls):
            patient = _median_us(call, lambda: capi.L.atexn_bench_mark_exchange_trouble(0))
            short = _median_us(call, lambda: capi.L.atexn_bench_mark_exchange_trouble(1))
            print(f"{what} [{N}, {S}, {C}] {dtype}: patient {patient:.1f} us, cut short {short:.1f} us", flush=True)
            assert short < 1.4 * patient + 5.0, what
    finally:
        capi.L.atexn_bench_mark_exchange_trouble(0)


@pytest.mark.parametrize("N,S,C,dtype", [(2, 2097152, 32, "f16"), (3, 703459, 23, "bf16")])
def test_held_calls_on_two_streams(N, S, C, dtype):
    """Two calls at a time, each of which wants the whole chip: their instances take CUs from each other between
    two instances of a call.  The bits of calls one after another."""
    import torch

    capi = util.Capi(bench=True)
    calls = _channels_last_calls(capi, N, S, C, dtype)
    side = _stream_beside(capi.L)
    alone = [call() for call in calls]
    torch.cuda.synchronize()
    main = torch.cuda.current_stream()
    e = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
    for first, second in ((0, 0), (0, 1), (1, 1)):
        got = []
        torch.cuda.synchronize()
        torch.cuda._sleep(400000)
        e[0].record()
        side.wait_stream(main)
        for _ in range(4):
            got.append((first, calls[first]()))
            with torch.cuda.stream(side):
                got.append((second, calls[second]()))
        main.wait_stream(side)
        e[1].record()
        torch.cuda.synchronize()
        print(f"[{N}, {S}, {C}] {dtype}: eight calls on two streams {e[0].elapsed_time(e[1]) * 1e3:.0f} us", flush=True)
        for which, out in got:
            for a, b in zip(out, alone[which]):
                assert torch.equal(_bits(a), _bits(b))
        del got
    capi.L.atexn_bench_mark_exchange_trouble(0)


@pytest.mark.parametrize("N,S,C,dtype", [(2, 2097152, 32, "f32"), (1, 1 << 24, 64, "bf16")])
def test_patience_grows_with_the_slabs(N, S, C, dtype):
    """Instances of 268 MB and 2 GB on a free GPU: nobody runs out of a wait, cut short or not, whose slab is merely
    large (a fifth more time where some did; a tenth is allowed)."""
    capi = util.Capi(bench=True)
    L = capi.L
    calls = _channels_last_calls(capi, N, S, C, dtype)
    try:
        for what, call in zip(("forward", "backward"), calls):
            assert L.atexn_set_tuning(b"cl_flat_polls", 10000) == 0
            endless = _median_us(call, lambda: L.atexn_bench_mark_exchange_trouble(0))
            assert L.atexn_set_tuning(b"cl_flat_polls", 300) == 0
            patient = _median_us(call, lambda: L.atexn_bench_mark_exchange_trouble(0))
            short = _median_us(call, lambda: L.atexn_bench_mark_exchange_trouble(1))
            print(f"{what} [{N}, {S}, {C}] {dtype}: {endless:.1f} us, patient {patient:.1f}, cut short {short:.1f}", flush=True)
            assert max(patient, short) < 1.1 * endless, what
    finally:
        L.atexn_set_tuning(b"cl_flat_polls", 300)
        L.atexn_bench_mark_exchange_trouble(0)


def test_the_occupier_leaves_in_time():
    import time

    import torch

    capi = util.Capi(bench=True)
    L = capi.L
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    assert L.atexn_bench_occupy(256, 5.0, torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    took = time.perf_counter() - t0
    assert took < 0.5, f"a 5 ms occupier took {took * 1e3:.1f} ms"
    assert L.atexn_bench_occupy(0, 5.0, None) != 0 and L.atexn_bench_occupy(8, 1000.0, None) != 0
