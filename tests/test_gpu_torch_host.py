"""The op and layer calls that go through csrc/torch_host.cc against the same calls through ctypes and
the Python autograd functions (the way of everything that is not a plain GPU tensor): same bits, same
errors, and gradients that arrive in every form autograd hands them out."""
import pytest

from tests import util  # noqa: F401

pytestmark = pytest.mark.gpu


class _NeverPlain:
    """Stands in for the extension: declines every call."""

    def __getattr__(self, name):
        return lambda *a: None


def _inputs(kind, dtype, grad=False):
    import torch

    g = torch.Generator(device="cuda").manual_seed(7)
    shape, width = {"ln": ((6, 5, 96), 96), "cl": ((3, 7, 9, 24), 24), "cf": ((3, 8, 9, 11), 8)}[kind]
    x = torch.randn(shape, device="cuda", generator=g).to(dtype)
    gamma = torch.rand(width, device="cuda", generator=g) + 0.5
    beta = torch.randn(width, device="cuda", generator=g)
    dy = torch.randn(shape, device="cuda", generator=g).to(dtype)
    for t in (x, gamma, beta):
        t.requires_grad_(grad)
    return x, gamma, beta, dy


def _ops(kind):
    from atex_amd import nv_norms as n

    if kind == "ln":
        return (lambda x, g, b: n.fused_layer_norm_op(x, g, b, axis=[-1]),
                lambda dy, x, g, m, r: n.fused_layer_norm_grad_op(dy, x, g, m, r, axis=-1),
                lambda x, g, b: n.fused_layer_norm(x, g, b, axis=(2,)))
    fmt = "N...C" if kind == "cl" else "NC..."
    return (lambda x, g, b: n.fused_instance_norm_op(x, g, b, data_format=fmt),
            lambda dy, x, g, m, r: n.fused_instance_norm_grad_op(dy, x, g, m, r, data_format=fmt),
            lambda x, g, b: n.fused_instance_norm(x, g, b, data_format=fmt))


@pytest.mark.parametrize("kind", ["ln", "cl", "cf"])
@pytest.mark.parametrize("dtype", ["float32", "float16", "bfloat16"])
def test_same_bits_as_through_ctypes(kind, dtype, monkeypatch):
    import torch

    from atex_amd.nv_norms import _capi

    fwd, bwd, diff = _ops(kind)
    x, gamma, beta, dy = _inputs(kind, getattr(torch, dtype), grad=True)

    def everything():
        y, m, r = fwd(x, gamma, beta)
        outs = [y, m, r, *bwd(dy, x, gamma, m, r)]
        assert not any(t.requires_grad for t in outs)
        y2, m2, r2 = diff(x, gamma, beta)
        assert y2.requires_grad and not m2.requires_grad and not r2.requires_grad
        outs += [y2.detach(), m2, r2]
        outs += torch.autograd.grad(y2, [x, gamma, beta], dy, retain_graph=True)
        # not contiguous, twice over a kept graph, and for one input alone
        outs += torch.autograd.grad(y2, [x, gamma, beta], dy.transpose(0, 1).contiguous().transpose(0, 1), retain_graph=True)
        outs += torch.autograd.grad(y2, [gamma], dy)
        with torch.no_grad():
            outs.append(diff(x, gamma, beta)[0])
        assert not outs[-1].requires_grad
        return outs

    assert _capi.torch_host().__file__.endswith("_torch_host.so")
    host = everything()
    monkeypatch.setattr(_capi, "_host", _NeverPlain())
    for i, (a, b) in enumerate(zip(host, everything())):
        assert a.dtype == b.dtype and torch.equal(a, b), f"output {i}"


def test_same_errors_as_through_ctypes(monkeypatch):
    import torch

    from atex_amd import nv_norms as n
    from atex_amd.nv_norms import _capi

    x, gamma, beta, dy = _inputs("ln", torch.float16)
    bad = [
        lambda: n.fused_layer_norm_op(x, gamma[:5].contiguous(), beta),
        lambda: n.fused_layer_norm_op(x, gamma.half(), beta),
        lambda: n.fused_layer_norm_op(x.transpose(0, 1), gamma, beta),
        lambda: n.fused_layer_norm_op(x.double(), gamma, beta),
        lambda: n.fused_layer_norm_op(x, gamma, beta, axis=(0,)),
        lambda: n.fused_layer_norm_op(x, gamma, beta, axis="NC"),
        lambda: n.fused_layer_norm_op(x, gamma.cpu(), beta),
        lambda: n.fused_layer_norm(x, gamma, beta, axis=2),
        lambda: n.fused_layer_norm_grad_op(dy.float(), x, gamma, beta, beta),
        lambda: n.fused_instance_norm_op(x, gamma, beta, data_format="NHWC"),
        lambda: n.fused_instance_norm_op(x.reshape(6, 5, 8, 12), gamma, beta, data_format=(1, 2)),
        lambda: n.fused_instance_norm_op(x.reshape(6, 5, 8, 12), gamma, beta),
    ]

    def errors():
        got = []
        for f in bad:
            with pytest.raises(Exception) as e:
                f()
            got.append((type(e.value), str(e.value)))
        return got

    host = errors()
    monkeypatch.setattr(_capi, "_host", _NeverPlain())
    assert host == errors()


def test_modified_inputs_and_freed_graphs_are_noticed():
    import torch

    from atex_amd import nv_norms as n

    x, gamma, beta, dy = _inputs("cf", torch.float32, grad=True)
    z = x * 1.0
    y, _, _ = n.fused_instance_norm(z, gamma, beta, data_format="NC...")
    with torch.no_grad():
        z.add_(1.0)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        y.backward(dy)
    y, _, _ = n.fused_instance_norm(x, gamma, beta, data_format="NC...")
    y.backward(dy)
    with pytest.raises(RuntimeError, match="second time"):
        y.backward(dy)


@pytest.mark.parametrize("kind", ["ln", "cl"])
def test_tracers_modes_and_transforms_see_the_call(kind):
    """They never see what the extension does, so it leaves these calls to Python: a traced layer
    stays a function of its input."""
    import torch
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode

    from atex_amd import nv_norms as n

    x, gamma, beta, dy = _inputs(kind, torch.float32)
    layer = n.LayerNormalization(axis=-1) if kind == "ln" else n.InstanceNormalization(axis=-1)
    layer.build(x.shape, device="cuda")
    traced = torch.jit.trace(layer, (x,), check_trace=False)
    assert torch.equal(traced(dy), layer(dy)) and torch.equal(traced(x), layer(x))

    class Seen(TorchDispatchMode):
        calls = 0

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.calls += 1
            return func(*args, **(kwargs or {}))

    fwd, _, diff = _ops(kind)
    with Seen() as seen:
        fwd(x, gamma, beta)
    assert seen.calls > 0

    class Functions(TorchFunctionMode):
        calls = 0

        def __torch_function__(self, func, types, args=(), kwargs=None):
            self.calls += func in (torch.empty, torch.empty_like)
            return func(*args, **(kwargs or {}))

    for call in (fwd, diff):
        with Functions() as seen, torch.device("cuda"):
            call(x, gamma, beta)
        assert seen.calls > 0
    with pytest.raises(RuntimeError, match="setup_context"):
        torch.vmap(lambda a: a + diff(x, gamma, beta)[0].sum())(dy)


@pytest.mark.parametrize("kind", ["ln", "cl", "cf"])
def test_compiled_autograd_takes_the_gradient(kind):
    import torch
    from torch._dynamo import compiled_autograd

    x, gamma, beta, dy = _inputs(kind, torch.float32, grad=True)
    diff = _ops(kind)[2]

    def grads():
        y = diff(x * 2.0, gamma, beta)[0]
        return torch.autograd.grad(y * 3.0, [x, gamma, beta], dy)

    eager = grads()
    with compiled_autograd._enable(lambda graph: torch.compile(graph, backend="eager")):
        compiled = grads()
    for i, (a, b) in enumerate(zip(eager, compiled)):
        assert torch.equal(a, b), f"gradient {i}"


@pytest.mark.parametrize("kind", ["ln", "cf"])
def test_errors_of_the_backward_are_those_of_the_op(kind, monkeypatch):
    """Saved-tensor hooks may hand the backward anything; what the op refuses raises the op's error."""
    import torch

    from atex_amd.nv_norms import InvalidArgumentError, _capi

    x, gamma, beta, dy = _inputs(kind, torch.float32, grad=True)
    diff = _ops(kind)[2]
    swaps = [lambda t: t.transpose(0, 1).contiguous().transpose(0, 1), lambda t: t.double(), lambda t: t.cpu(),
             lambda t: t[:1].contiguous()]

    def errors():
        got = []
        for swap in swaps:
            with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: swap(t) if t.shape == x.shape else t):
                y = diff(x, gamma, beta)[0]
            with pytest.raises(Exception) as e:
                torch.autograd.grad(y, [x, gamma, beta], dy)
            got.append((type(e.value), str(e.value)))
        return got

    here = errors()
    assert all(t is InvalidArgumentError for t, _ in here), here
    monkeypatch.setattr(_capi, "_host", _NeverPlain())
    assert here == errors()


def test_a_default_device_is_not_in_the_way(monkeypatch):
    """... though it is a torch-function mode: the extension takes the call."""
    import torch

    from atex_amd.nv_norms import ops

    x, gamma, beta, _ = _inputs("ln", torch.float16)
    fwd, _, _ = _ops("ln")
    plain = fwd(x, gamma, beta)
    monkeypatch.setattr(ops, "_desc", None)  # what the way through Python starts with
    with torch.device("cuda"):
        got = fwd(x, gamma, beta)
    for a, b in zip(got, plain):
        assert torch.equal(a, b)


@pytest.mark.parametrize("kind", ["ln", "cl"])
def test_a_profiler_sees_the_call(kind, monkeypatch):
    """By the name, the inputs and the link from the backward that the Python autograd function has."""
    import torch

    from atex_amd.nv_norms import _capi

    x, gamma, beta, dy = _inputs(kind, torch.float32, grad=True)
    diff = _ops(kind)[2]
    name = "_FusedLayerNormFn" if kind == "ln" else "_FusedInstanceNormFn"

    def seen():
        with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU], record_shapes=True) as p:
            y = diff(x, gamma, beta)[0]
            torch.autograd.grad(y, [x, gamma, beta], dy)
        calls = [e for e in p.events() if e.name == name]
        backward = [e for e in p.events() if "evaluate_function" in e.name and e.sequence_nr == calls[0].sequence_nr]
        return [e.input_shapes[:3] for e in calls], len(backward)

    here = seen()
    assert len(here[0]) == 1 and here[1] == 1, here
    monkeypatch.setattr(_capi, "_host", _NeverPlain())
    assert here == seen()


@pytest.mark.parametrize("kind", ["ln", "cl", "cf"])
def test_side_streams_and_threads(kind):
    """The current stream of the calling thread, for the outputs and the scratch memory too: what the
    allocator hands out again is not written by a call that is still running on another stream."""
    import threading

    import torch

    _, _, diff = _ops(kind)
    inputs = [[t.detach().clone().requires_grad_(i < 3) for i, t in enumerate(_inputs(kind, torch.float16))] for _ in range(3)]
    for i, (x, _, _, dy) in enumerate(inputs):
        with torch.no_grad():
            x.add_(i)
            dy.mul_(i + 1)

    def step(x, gamma, beta, dy):
        y = diff(x * 2.0, gamma, beta)[0]
        return [y.detach(), *torch.autograd.grad(y, [x, gamma, beta], dy)]

    want = [step(*i) for i in inputs]
    torch.cuda.synchronize()
    got = [None] * 3

    def work(i):
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            for _ in range(20):
                got[i] = step(*inputs[i])
        stream.synchronize()

    threads = [threading.Thread(target=work, args=(i,)) for i in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for a, b in zip(want, got):
        for p, q in zip(a, b):
            assert torch.equal(p, q)


@pytest.mark.parametrize("kind", ["ln", "cf"])
def test_captured_steps(kind):
    import torch

    x, gamma, beta, dy = _inputs(kind, torch.float16, grad=True)
    diff = _ops(kind)[2]

    def step():
        y = diff(x, gamma, beta)[0]
        return [y, *torch.autograd.grad(y, [x, gamma, beta], dy)]

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outs = step()
    for replay in range(3):
        with torch.no_grad():
            x.mul_(1.5).add_(0.25)
        want = [t.detach().clone() for t in step()]
        for t in outs:
            t.detach().fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip(outs, want):
            assert torch.equal(a.detach(), b), f"replay {replay}"


def test_saved_tensor_hooks_and_checkpoints():
    import torch
    from torch.utils.checkpoint import checkpoint

    x, gamma, beta, dy = _inputs("ln", torch.float32, grad=True)
    diff = _ops("ln")[2]
    want = torch.autograd.grad(diff(x, gamma, beta)[0], [x, gamma, beta], dy)
    packed = []

    def pack(t):
        packed.append(t.shape)
        return t.cpu()

    with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t.cuda()):
        y = diff(x, gamma, beta)[0]
    assert sorted(packed) == sorted([x.shape, gamma.shape, torch.Size([30]), torch.Size([30])])
    for a, b in zip(want, torch.autograd.grad(y, [x, gamma, beta], dy)):
        assert torch.equal(a, b)
    y = checkpoint(lambda t: diff(t, gamma, beta)[0], x, use_reentrant=False)
    for a, b in zip(want, torch.autograd.grad(y, [x, gamma, beta], dy)):
        assert torch.equal(a, b)


def test_inference_mode_and_forward_mode(monkeypatch):
    import torch
    from torch.autograd import forward_ad

    from atex_amd.nv_norms import _capi

    x, gamma, beta, dy = _inputs("cl", torch.float32)
    diff = _ops("cl")[2]
    want = diff(x, gamma, beta)[0]
    with torch.inference_mode():
        y = diff(x, gamma, beta)[0]
        assert y.is_inference() and torch.equal(y, want)

    def refusal():  # no forward-mode formula: refused, not silently without a tangent
        with forward_ad.dual_level(), pytest.raises(Exception) as e:
            diff(forward_ad.make_dual(x, dy), gamma, beta)
        return type(e.value), str(e.value)

    here = refusal()
    monkeypatch.setattr(_capi, "_host", _NeverPlain())
    assert here == refusal()


@pytest.mark.parametrize("kind", ["ln", "cf"])
def test_a_compiled_model_breaks_its_graph_at_the_call(kind):
    import torch

    from atex_amd import nv_norms as n

    x, _, _, dy = _inputs(kind, torch.float32, grad=True)
    layer = n.LayerNormalization(axis=-1) if kind == "ln" else n.InstanceNormalization(axis=1)
    layer.build(x.shape, device="cuda")
    model = torch.nn.Sequential(torch.nn.ReLU(), layer, torch.nn.ReLU())

    def step(f):
        y = f(x)
        return [y.detach(), *torch.autograd.grad(y, [x, layer.gamma, layer.beta], dy)]

    for a, b in zip(step(model), step(torch.compile(model, backend="eager"))):
        assert torch.equal(a, b)


def test_anomaly_mode_and_node_hooks():
    import torch

    x, gamma, beta, dy = _inputs("ln", torch.float32, grad=True)
    diff = _ops("ln")[2]
    seen = []
    with torch.autograd.detect_anomaly(check_nan=True):
        y = diff(x, gamma, beta)[0]
        y.grad_fn.register_hook(lambda into, out: seen.append(len(into)))
        want = torch.autograd.grad(y, [x, gamma, beta], dy, retain_graph=True)
        bad = dy.clone()
        bad.view(-1)[0] = float("nan")
        with pytest.raises(RuntimeError, match="FusedLayerNormBackward.* returned nan"):
            torch.autograd.grad(y, [x, gamma, beta], bad)
    assert seen[0] == 3
    for a, b in zip(want, torch.autograd.grad(diff(x, gamma, beta)[0], [x, gamma, beta], dy)):
        assert torch.equal(a, b)
