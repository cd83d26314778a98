"""The operators' compiled host side (csrc/host/host_ops.cpp) against their Python classes, which run the same kernels."""
import contextlib
import threading

import pytest
import torch

import vision_rwkv_amd as ops
from vision_rwkv_amd import _lib
from vision_rwkv_amd.ops import _WKVDivided

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _inputs(kind, dtype, B=3, T=21, C=128, grad=True):
    g = torch.Generator().manual_seed(7)
    t = lambda *s: torch.randn(*s, generator=g).to(DEV, dtype)
    if kind == "wkv6":
        xs = [t(B, T, C), t(B, T, C), t(B, T, C), t(B, T, C), t(C // 64, 64).float()]
        native = lambda *a: ops.RUN_CUDA_RWKV6(B, T, C, C // 64, *a)
        python = lambda *a: ops.WKV_6.apply(B, T, C, C // 64, *a)
    else:
        xs = [t(C), t(C), t(B, T, C), t(B, T, C)]
        native = ops.RUN_CUDA if kind == "wkv" else lambda w, u, k, v: ops.ops.wkv_divided(w, u, T, k, v)
        python = ops.WKV.apply if kind == "wkv" else lambda w, u, k, v: _WKVDivided.apply(w, u, T, k, v)
    return [x.requires_grad_(grad) for x in xs], native, python


@pytest.mark.parametrize("kind", ["wkv", "divided", "wkv6"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("grad", [True, False])
def test_the_compiled_call_is_the_python_class(kind, dtype, grad):
    xs, native, python = _inputs(kind, dtype, grad=grad)
    got, want = native(*xs), python(*xs)
    assert torch.equal(got, want) and got.dtype == want.dtype and (got.grad_fn is not None) == (want.grad_fn is not None) == grad
    with torch.no_grad():
        assert native(*xs).grad_fn is None
    with torch.inference_mode():
        assert native(*xs).is_inference()
    if grad:
        assert "Backward" not in type(got.grad_fn).__name__                       # the compiled node
        gy = torch.randn(got.shape, device=DEV).to(got.dtype)
        a, b = torch.autograd.grad(got, xs, gy, retain_graph=True), torch.autograd.grad(want, xs, gy, retain_graph=True)
        assert all(torch.equal(p, q) and p.dtype == q.dtype and p.shape == q.shape for p, q in zip(a, b))
        some = torch.autograd.grad(got, xs[2], gy, retain_graph=True, create_graph=True)[0]
        assert torch.equal(some, a[2]) and not some.requires_grad                 # no second derivative, as before
        # an unrecorded input's gradient is dropped; the others are the same
        part = [x.detach().requires_grad_(i == 1) for i, x in enumerate(xs)]
        assert torch.equal(torch.autograd.grad(native(*part), part[1], gy)[0], a[1])


@pytest.mark.parametrize("kind", ["wkv", "divided", "wkv6"])
def test_what_autograd_promises_holds(kind):
    xs, native, python = _inputs(kind, torch.bfloat16)
    gy = torch.randn(3, 21, 128, device=DEV).to(native(*xs).dtype)
    want = torch.autograd.grad(python(*xs), xs, gy)
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t) or t.cpu(), lambda t: t.to(DEV)):
        y = native(*xs)
    assert len(packed) == len(xs)
    assert all(torch.equal(p, q) for p, q in zip(torch.autograd.grad(y, xs, gy), want))
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: t.cpu()):
        y = native(*xs)
    with pytest.raises(RuntimeError, match="one device"):
        torch.autograd.grad(y, xs, gy)
    y = native(*xs)
    with torch.no_grad():
        xs[3].mul_(1)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        torch.autograd.grad(y, xs, gy)
    y = native(*xs)
    torch.autograd.grad(y, xs, gy)
    with pytest.raises(RuntimeError, match="second time"):
        torch.autograd.grad(y, xs, gy)
    y = native(*xs)
    with pytest.raises(RuntimeError):                                             # a cotangent without memory of its own
        torch.vmap(lambda g: torch.autograd.grad(y, xs[2], g, retain_graph=True)[0])(torch.stack([gy, gy]))
    wide = gy.new_zeros(()).expand(gy.shape)
    with pytest.raises(AssertionError) if kind == "wkv6" else contextlib.nullcontext():
        torch.autograd.grad(y, xs, wide)


@pytest.mark.parametrize("kind", ["wkv", "wkv6"])
def test_other_calls_are_left_to_the_python_class(kind):
    xs, native, python = _inputs(kind, torch.float32)
    host = _lib.host()
    call = (lambda *a: host.wkv(*a, 1.0)) if kind == "wkv" else (lambda *a: host.wkv6(3, 21, 128, 2, *a, False))
    assert call(*xs) is not None
    swap = lambda i, t: [t if j == i else x for j, x in enumerate(xs)]
    for other in (xs[2].transpose(0, 1).contiguous().transpose(0, 1), xs[2].cpu(), xs[2].double(), xs[2][:, :5].contiguous(), xs[2].half(),
                  xs[2].detach().as_subclass(type("Sub", (torch.Tensor,), {}))):
        assert call(*swap(2, other)) is None
    assert call(*swap(1, None)) is None
    empty = [x[:0] if x.dim() == 3 else x for x in xs]
    assert call(*empty) is None
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(xs[2].detach(), torch.ones_like(xs[2]))
        assert call(*swap(2, dual)) is None
    class Seen(torch.overrides.TorchFunctionMode):
        def __torch_function__(self, f, types, args=(), kwargs=None):
            return f(*args, **(kwargs or {}))
    with Seen():
        assert call(*xs) is None
    with pytest.raises(Exception):
        torch.func.vmap(native, in_dims=tuple(0 if i == 2 else None for i in range(len(xs))))(*swap(2, torch.stack([xs[2]] * 2)))


@pytest.mark.parametrize("kind", ["wkv", "wkv6"])
def test_threads_and_streams_each_get_their_own_results(kind):
    want = {}
    def work(i):
        xs, native, _ = _inputs(kind, torch.bfloat16, B=2 + i)
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.default_stream())
        with torch.cuda.stream(stream):
            for _ in range(5):
                y = native(*xs)
                grads = torch.autograd.grad(y, xs, torch.ones_like(y))
        stream.synchronize()
        want[i] = (xs, y, grads)
    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    [t.start() for t in threads], [t.join() for t in threads]
    assert len(want) == 4
    for i, (xs, y, grads) in want.items():
        ref = _inputs(kind, torch.bfloat16, B=2 + i)[2](*xs)
        assert torch.equal(y, ref) and all(torch.equal(a, b) for a, b in zip(grads, torch.autograd.grad(ref, xs, torch.ones_like(ref))))


def test_recorded_into_a_graph_forward_and_backward():
    xs, native, python = _inputs("wkv", torch.bfloat16)
    gy = torch.randn(3, 21, 128, device=DEV).bfloat16()
    run = lambda f: (lambda y: (y, *torch.autograd.grad(y, xs, gy)))(f(*xs))
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        run(native)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outs = run(native)
    for i in range(3):
        with torch.no_grad():
            for x in xs:
                x.copy_(torch.randn(x.shape, device=DEV))
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(outs, run(python)))


@pytest.mark.parametrize("kind", ["wkv", "divided", "wkv6"])
def test_the_operators_without_the_compiled_module(kind, monkeypatch):
    xs, native, _ = _inputs(kind, torch.bfloat16)
    run = lambda: (lambda y: (y, *torch.autograd.grad(y, xs, torch.ones_like(y))))(native(*xs))
    want = run()
    monkeypatch.setattr(_lib, "_host", _lib._NoHost)
    got = run()
    assert type(got[0].grad_fn).__name__ == {"wkv": "WKV", "divided": "_WKVDivided", "wkv6": "WKV_6"}[kind] + "Backward" and all(torch.equal(a, b) for a, b in zip(got, want))


def test_a_block_without_the_compiled_module(monkeypatch):
    net = ops.VRWKV(img_size=32, patch_size=16, embed_dims=64, depth=1).to(DEV, torch.bfloat16).eval()
    x = torch.randn(2, 3, 32, 32, generator=torch.Generator().manual_seed(3)).to(DEV, torch.bfloat16)
    with torch.no_grad():
        want = net(x).float()
        monkeypatch.setattr(_lib, "_host", _lib._NoHost)
        got = net(x).float()
    assert (got - want).norm() <= 2 ** -6 * want.norm()      # a few roundings to 8 bits that the native call leaves out
