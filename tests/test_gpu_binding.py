"""The torch binding (csrc/torch_binding.cpp) against the Python autograd functions: the same results for
the calls it takes, and None for those it must leave to the Python path."""

from __future__ import annotations

import contextlib
import itertools

import pytest
import torch

from rfdetr_jax_amd import (
    MSDeformAttn,
    _native,
    bilinear_grid_sample,
    grouped_attention,
    ms_deform_attn_core_rows,
    ms_deform_attn_fused,
    point_sample,
    scaled_dot_product_attention,
    value_proj_rows,
)

pytestmark = pytest.mark.gpu

SHAPES = ((6, 5), (3, 4))
POSITIONS = 42


def _draw(*shape, dtype=torch.float32):
    return torch.randn(*shape, device="cuda").to(dtype)


def _call(op, dtype):
    """(function of its tensors, tensors) of one small call."""
    torch.manual_seed(3)
    b, q, h, d, p = 2, 7, 2, 8, 2
    levels = len(SHAPES)
    if op == "core":
        attn = torch.softmax(_draw(b, q, h, levels * p), -1)
        return (lambda v, l, a: ms_deform_attn_core_rows(v, SHAPES, l, a)), [_draw(b * h, POSITIONS, d, dtype=dtype), torch.rand(b, q, h, levels, p, 2, device="cuda"), attn]
    if op == "sampler":
        attn = torch.softmax(_draw(b, q, h, levels * p), -1)
        return (lambda v, l, a: ms_deform_attn_core_rows(v, [list(s) for s in SHAPES], l, a, "gather")), [_draw(b * h, POSITIONS, d, dtype=dtype), torch.rand(b, q, h, levels, p, 2, device="cuda"), attn]
    if op == "fused":
        return (lambda v, r, o, l: ms_deform_attn_fused(v, SHAPES, r, o, l)), [_draw(b * h, POSITIONS, d, dtype=dtype), torch.rand(b, q, levels, 4, device="cuda"), _draw(b, q, h, levels, p, 2), _draw(b, q, h, levels * p)]
    if op == "value_proj":
        mask = torch.rand(b, POSITIONS, device="cuda") < 0.3
        return (lambda x, w, c: value_proj_rows(x, w, c, h, mask)), [_draw(b, POSITIONS, 16, dtype=dtype), _draw(h * d, 16), _draw(h * d)]
    if op == "value_proj_plain":
        return (lambda x, w: value_proj_rows(x, w, None, h)), [_draw(b, POSITIONS, 16, dtype=dtype), _draw(h * d, 16)]
    if op == "grid":
        return (lambda x, g: bilinear_grid_sample(x, g)), [_draw(b, 3, 9, 7, dtype=dtype), 2 * torch.rand(b, 4, 5, 2, device="cuda") - 1]
    if op == "points":
        return (lambda x, c: point_sample(x, c)), [_draw(b, 3, 9, 7, dtype=dtype), torch.rand(b, 11, 2, device="cuda")]
    if op == "rows":
        qk = _draw(b, 2 * 33, 2 * 64, dtype=dtype)
        return (lambda q, k, v: grouped_attention(q, k, v, 2, 2)), [qk[..., :64], qk[..., 64:], _draw(b, 66, 64, dtype=dtype)]
    return (lambda q, k, v: scaled_dot_product_attention(q, k, v)), [_draw(b, h, 33, 32, dtype=dtype) for _ in range(3)]


OPS = ["core", "sampler", "fused", "value_proj", "value_proj_plain", "grid", "points", "rows", "heads"]
NAMES = {"core": "Core", "sampler": "Core", "fused": "Fused", "value_proj": "ValueProj", "value_proj_plain": "ValueProj", "grid": "GridSample",
         "points": "GridSample", "rows": "Attention", "heads": "Attention"}


class _Off:
    """A binding that leaves every call to the Python path."""

    core = fused = value_proj = grid_sample = attention = staticmethod(lambda *a: None)


@pytest.fixture
def python_path(monkeypatch):
    @contextlib.contextmanager
    def off():
        with monkeypatch.context() as m:
            m.setattr(_native, "binding", lambda: _Off)
            yield

    return off


def _is_binding(out, op):
    node = out.grad_fn
    while node is not None and NAMES[op] not in node.name():  # through the reshape of a point grid
        node = node.next_functions[0][0] if node.next_functions else None
    return node is not None and "CppNode" in node.name()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("op", OPS)
def test_binding_matches_python_path(op, dtype, python_path):
    """Every subset of tensors that need a gradient, a strided cotangent, and a side stream. Values are
    bit for bit the same except where LDS atomics sum (gradients of value and feature maps)."""
    fn, tensors = _call(op, dtype)
    for wanted in itertools.product([False, True], repeat=len(tensors)):
        results = []
        for python in (False, True):
            with python_path() if python else contextlib.nullcontext():
                ins = [t.detach().requires_grad_(w) for t, w in zip(tensors, wanted)]
                side = torch.cuda.Stream()
                side.wait_stream(torch.cuda.current_stream())
                with torch.cuda.stream(side):
                    out = fn(*ins)
                    grads = []
                    if any(wanted):
                        assert _is_binding(out, op) != python
                        torch.manual_seed(5)
                        g = _draw(*out.shape[:-1], 2 * out.shape[-1])[..., ::2]
                        grads = torch.autograd.grad(out, [t for t in ins if t.requires_grad], g.to(out.dtype))
                torch.cuda.current_stream().wait_stream(side)
                torch.cuda.synchronize()
                results.append((out, *grads))
        for a, b in zip(*results, strict=True):
            assert a.shape == b.shape and a.dtype == b.dtype and a.stride() == b.stride()
            torch.testing.assert_close(a, b, rtol=2.0 ** -7 if a.dtype == torch.bfloat16 else 1e-6, atol=1e-6)


@pytest.mark.parametrize("op", OPS)
def test_binding_leaves_to_python(op, python_path):
    """What the binding does not take runs, or fails, exactly as without it: other types and layouts,
    CPU tensors, subclasses, functorch transforms, forward-mode tangents and modes."""
    fn, tensors = _call(op, torch.float32)

    class Sub(torch.Tensor):
        pass

    class Mode(torch.utils._python_dispatch.TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    def forward_mode():
        import torch.autograd.forward_ad as ad

        with ad.dual_level():
            fn(ad.make_dual(tensors[0], torch.ones_like(tensors[0])), *tensors[1:])

    def mode():
        with Mode():
            return fn(*[t.detach().requires_grad_() for t in tensors])

    def last(t):
        return fn(*tensors[:-1], t)

    cases = {
        "double": lambda: fn(tensors[0].double(), *tensors[1:]),
        "half": lambda: last(tensors[-1].half()),
        "strided": lambda: last(torch.stack([tensors[-1], tensors[-1]], -1)[..., 0]),
        "cpu": lambda: fn(tensors[0].cpu(), *tensors[1:]),
        "shape": lambda: last(tensors[-1][:, :-1] if tensors[-1].dim() > 1 else tensors[-1][:-1]),
        "dims": lambda: fn(tensors[0][None], *tensors[1:]),
        "subclass": lambda: fn(tensors[0].as_subclass(Sub), *tensors[1:]),
        "grad": lambda: torch.func.grad(lambda t: fn(t, *tensors[1:]).sum())(tensors[0]),
        "vmap": lambda: torch.func.vmap(lambda t: fn(t, *tensors[1:]))(tensors[0][None]),
        "forward_mode": forward_mode,
        "mode": mode,
        "none": lambda: last(None),
    }
    for name, case in cases.items():
        seen = []
        for python in (False, True):
            with python_path() if python else contextlib.nullcontext():
                try:
                    out = case()
                    seen.append(("ok", out))
                except Exception as e:  # noqa: BLE001
                    seen.append((type(e), str(e)))
        (a, x), (b, y) = seen
        assert a == b, (name, seen)
        if a == "ok" and x is not None:
            assert type(x) is type(y) and x.dtype == y.dtype, name
            torch.testing.assert_close(x, y, rtol=1e-6, atol=1e-6)
        elif a != "ok":
            assert x == y, name


@pytest.mark.parametrize("op", OPS)
def test_binding_saved_tensors(op):
    """Saved-tensor hooks see the saved tensors, an input changed in place after the forward is an
    error, and a graph is freed after its backward."""
    fn, tensors = _call(op, torch.float32)
    ins = [t.clone().requires_grad_() for t in tensors]
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t.shape) or t, lambda t: t):
        out = fn(*ins)
    assert ins[0].shape in packed
    torch.autograd.grad(out.sum(), ins)
    with pytest.raises(RuntimeError, match="second time|already been freed"):
        out.sum().backward()
    out = fn(*ins)
    with torch.no_grad():
        ins[1].add_(1.0)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        out.sum().backward()


def _other_layout(t):
    """The same values, channels first in memory."""
    return t.movedim(-1, 0).contiguous().movedim(0, -1)


@pytest.mark.parametrize("op", OPS)
def test_binding_saved_tensor_hooks(op):
    """What hooks make of the saved tensors reaches the kernels by its values: in another layout, or in
    bfloat16 (as if rounded to it and brought back). Other shapes and CPU tensors are refused."""
    fn, tensors = _call(op, torch.float32)

    def grads(unpack):
        ins = [t.detach().clone().requires_grad_() for t in tensors]
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t, unpack):
            out = fn(*ins)
        assert _is_binding(out, op)
        torch.manual_seed(5)
        return torch.autograd.grad(out, ins, _draw(*out.shape))

    def floats(f):
        return lambda t: f(t) if t.dtype == torch.float32 else t

    want, rounded = grads(lambda t: t), grads(floats(lambda t: t.bfloat16().float()))
    for got, expected in ((grads(_other_layout), want), (grads(floats(lambda t: t.bfloat16())), rounded)):
        for a, b in zip(got, expected, strict=True):
            assert a.dtype == b.dtype
            torch.testing.assert_close(a, b, rtol=1e-6, atol=1e-6)
    for wrong in (lambda t: t[..., :-1], lambda t: t[None], lambda t: t.cpu()):
        with pytest.raises((ValueError, RuntimeError), match="saved tensor|invalid gradient"):
            grads(wrong)


def test_binding_errors_keep_their_type():
    """A shape that only the library refuses raises MsdaError from the forward and from the backward."""
    q = _draw(1, 1, 8, 48)  # head_dim 48
    with pytest.raises(_native.MsdaError) as e:
        scaled_dot_product_attention(q, q, q)
    assert e.value.code == _native.ERR_UNSUPPORTED
    wide = ((2, 40000),)  # an image row too wide for the backward's LDS
    v = _draw(1, 80000, 64).requires_grad_()
    loc, attn = torch.rand(1, 3, 1, 1, 1, 2, device="cuda"), torch.ones(1, 3, 1, 1, device="cuda")
    out = ms_deform_attn_core_rows(v, wide, loc, attn)
    with pytest.raises(_native.MsdaError) as e:
        out.sum().backward()
    assert e.value.code == _native.ERR_UNSUPPORTED


def test_binding_module_and_threads():
    """The module's parameters take the binding, from several threads and streams at once."""
    import threading

    m = MSDeformAttn(32, 2, 4, 2).cuda()
    torch.manual_seed(1)
    q, x, ref = _draw(2, 9, 32), _draw(2, POSITIONS, 32), torch.rand(2, 9, 2, 4, device="cuda")
    want = m(q, ref, x, SHAPES)
    want_grads = torch.autograd.grad(want.sum(), list(m.parameters()))
    torch.cuda.synchronize()
    failed = []

    def work():
        try:
            s = torch.cuda.Stream()
            with torch.cuda.stream(s):
                for _ in range(20):
                    out = m(q, ref, x, SHAPES)
                    grads = torch.autograd.grad(out.sum(), list(m.parameters()))
            s.synchronize()
            torch.testing.assert_close(out, want)
            for a, b in zip(grads, want_grads):
                torch.testing.assert_close(a, b, rtol=1e-4, atol=1e-4)
        except Exception as e:  # noqa: BLE001
            failed.append(e)

    threads = [threading.Thread(target=work) for _ in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed, failed[0]
