"""Parity of the decoder self-attention kernels (msda_attention_fwd / _bwd through the C ABI, via
the torch mirror rfdetr_jax_amd.attention) on an MI355X.

Expected values: oracle/attention_ref.py (float64); for the module, torch's
``nn.MultiheadAttention`` in float64 on the CPU, run per (image, group). Tolerances
(``max|got - want| <= tol * max(1, max|want|)``): f32 forward 1e-5, gradients 1e-4; bf16 2e-2.
"""

from __future__ import annotations

import sys

import numpy as np
import pytest
import torch

from oracle import attention_ref as AT
from oracle.msda_ref import bf16_round
from rfdetr_jax_amd.attention import (
    MultiheadAttention,
    decoder_self_attention,
    grouped_attention,
    scaled_dot_product_attention,
)
from tests._util import assert_close

pytestmark = pytest.mark.gpu


def _dev():
    assert torch.cuda.is_available(), "GPU tests need a visible MI355X"
    return torch.device("cuda:0")


def _note(msg):
    sys.stderr.write(f"[gpu] {msg}\n")
    sys.stderr.flush()


def _t(a, dtype=None):
    t = torch.from_numpy(np.ascontiguousarray(a)).to(_dev())
    return t if dtype is None else t.to(dtype)


def _np(t):
    return t.detach().float().cpu().numpy()


SHAPES = {
    "decoder": (6, 8, 300, 32),   # 300 queries per group, 8 heads x 32 (config-2 slices, fewer of them)
    "small": (2, 3, 9, 32),
    "ragged": (2, 2, 37, 64),     # head_dim 64, rows not a multiple of 32
    "one": (1, 1, 1, 32),
    "long": (1, 2, 480, 32),      # 8 chunks of keys
    "long64": (1, 1, 1000, 64),   # head_dim 64, 16 chunks
}


@pytest.mark.parametrize("bf16", [False, True], ids=["f32", "bf16"])
@pytest.mark.parametrize("masked", [False, True], ids=["nomask", "mask"])
@pytest.mark.parametrize("shape", sorted(SHAPES))
def test_sdpa_against_oracle(shape, masked, bf16):
    b, h, length, d = SHAPES[shape]
    _note(f"sdpa {shape} masked={masked} bf16={bf16}")
    rng = np.random.default_rng(41)
    q, k, v, g = (rng.standard_normal((b, h, length, d)).astype(np.float32) for _ in range(4))
    mask = None
    if masked:
        mask = rng.uniform(0, 1, (length, length)) < 0.2
        mask[:, -3:] = True  # tests/test_attention.py:37-40
        mask[length // 2] = True  # a fully blocked row: uniform weights
    if bf16:
        q, k, v, g = (bf16_round(t) for t in (q, k, v, g))
    dt = torch.bfloat16 if bf16 else None
    tq, tk, tv = (_t(x, dt).requires_grad_(True) for x in (q, k, v))
    out = scaled_dot_product_attention(tq, tk, tv, None if mask is None else _t(mask))
    out.backward(_t(g, dt))
    torch.cuda.synchronize()
    tf, tg = (2e-2, 2e-2) if bf16 else (1e-5, 1e-4)
    assert_close(_np(out), AT.sdpa(q, k, v, mask), tf, "out")
    for name, t, want in zip("qkv", (tq, tk, tv), AT.sdpa_vjp(q, k, v, g, mask)):
        assert_close(_np(t.grad), want, tg, f"grad_{name}")


@pytest.mark.parametrize("bf16", [False, True], ids=["f32", "bf16"])
@pytest.mark.parametrize("order", ["rising", "falling"])
def test_sdpa_reference_score_moves(order, bf16):
    """The forward's running reference score moves only when a key chunk's maximum exceeds it by
    more than 8 (log2 units). Keys scaled up chunk by chunk (factors 1, 4, 7, 10, 13) move it at
    every chunk, with the partial sums rescaled each time; scaled down, it never moves after the
    first chunk and later weights are far below 1."""
    b, h, length, d = 2, 4, 300, 32
    _note(f"sdpa reference score {order} bf16={bf16}")
    rng = np.random.default_rng(43)
    q, k, v, g = (rng.standard_normal((b, h, length, d)).astype(np.float32) for _ in range(4))
    factor = 1.0 + 3.0 * (np.arange(length) // 64)
    k = k * (factor if order == "rising" else factor[::-1])[:, None].astype(np.float32)
    if bf16:
        q, k, v, g = (bf16_round(t) for t in (q, k, v, g))
    dt = torch.bfloat16 if bf16 else None
    tq, tk, tv = (_t(x, dt).requires_grad_(True) for x in (q, k, v))
    out = scaled_dot_product_attention(tq, tk, tv)
    out.backward(_t(g, dt))
    torch.cuda.synchronize()
    tf, tg = (2e-2, 2e-2) if bf16 else (1e-5, 1e-4)
    assert_close(_np(out), AT.sdpa(q, k, v, None), tf, "out")
    for name, t, want in zip("qkv", (tq, tk, tv), AT.sdpa_vjp(q, k, v, g, None)):
        assert_close(_np(t.grad), want, tg, f"grad_{name}")


def test_reference_known_answers():
    """tests/test_attention.py:104-119 (at head_dim 32): equal scores give the mean of V, and the
    padding of the key blocks takes no weight."""
    q = torch.ones((2, 3, 145, 32), device=_dev())
    k = -torch.ones((2, 3, 145, 32), device=_dev())
    v = _t(np.random.default_rng(0).standard_normal((2, 3, 145, 32)).astype(np.float32))
    out = _np(scaled_dot_product_attention(q, k, v))
    want = _np(v).astype(np.float64).mean(axis=2, keepdims=True)
    assert_close(out, np.broadcast_to(want, out.shape), 1e-5, "mean")


@pytest.mark.parametrize("bf16", [False, True], ids=["f32", "bf16"])
def test_grouped_rows_layout_against_split_groups(bf16):
    """[B, G * P, C] rows with q and k read in place from a fused [B, Q, 2C] projection (row stride
    2C): the same as splitting the groups onto the batch, attending per head and merging back."""
    batch, groups, per, heads, d = 2, 13, 30, 8, 32
    c = heads * d
    _note(f"grouped rows bf16={bf16}")
    rng = np.random.default_rng(42)
    qk = rng.standard_normal((batch, groups * per, 2 * c)).astype(np.float32)
    v = rng.standard_normal((batch, groups * per, c)).astype(np.float32)
    g = rng.standard_normal((batch, groups * per, c)).astype(np.float32)
    if bf16:
        qk, v, g = (bf16_round(x) for x in (qk, v, g))
    dt = torch.bfloat16 if bf16 else None
    tqk = _t(qk, dt).requires_grad_(True)
    tv = _t(v, dt).requires_grad_(True)
    out = grouped_attention(tqk[..., :c], tqk[..., c:], tv, heads, groups)
    out.backward(_t(g, dt))
    tf, tg = (2e-2, 2e-2) if bf16 else (1e-5, 1e-4)

    def heads_of(x):  # [G B, P, C] -> [G B, H, P, D]
        return x.reshape(x.shape[0], per, heads, d).transpose(0, 2, 1, 3)

    qs, ks, vs = (heads_of(AT.split_groups(x, per)) for x in (qk[..., :c], qk[..., c:], v))
    gs = heads_of(AT.split_groups(g, per))
    want = AT.merge_groups(AT.sdpa(qs, ks, vs).transpose(0, 2, 1, 3).reshape(groups * batch, per, c), batch)
    assert_close(_np(out), want, tf, "out")
    dq, dk, dv = (AT.merge_groups(x.transpose(0, 2, 1, 3).reshape(groups * batch, per, c), batch) for x in AT.sdpa_vjp(qs, ks, vs, gs))
    gqk = _np(tqk.grad)
    assert_close(gqk[..., :c], dq, tg, "grad_q")
    assert_close(gqk[..., c:], dk, tg, "grad_k")
    assert_close(_np(tv.grad), dv, tg, "grad_v")


def _torch_reference(m, tgt, pos, groups, heads, grad):
    """The decoder self-attention written with torch's float64 nn.MultiheadAttention on the CPU, one
    (image, group) block at a time, with the parameter gradients."""
    c = tgt.shape[-1]
    ref = torch.nn.MultiheadAttention(c, heads, batch_first=True, dtype=torch.float64)
    with torch.no_grad():
        ref.in_proj_weight.copy_(m.in_proj_weight.detach().double().cpu())
        ref.in_proj_bias.copy_(m.in_proj_bias.detach().double().cpu())
        ref.out_proj.weight.copy_(m.out_proj.weight.detach().double().cpu())
        ref.out_proj.bias.copy_(m.out_proj.bias.detach().double().cpu())
    t = torch.tensor(tgt, dtype=torch.float64, requires_grad=True)
    p = torch.tensor(pos, dtype=torch.float64)
    batch, total, _ = tgt.shape
    per = total // groups
    query = t + p
    outs = []
    for b in range(batch):
        row = []
        for g in range(groups):
            sl = slice(g * per, (g + 1) * per)
            o, _ = ref(query[b:b + 1, sl], query[b:b + 1, sl], t[b:b + 1, sl], need_weights=False)
            row.append(o)
        outs.append(torch.cat(row, 1))
    out = torch.cat(outs, 0)
    out.backward(torch.tensor(grad, dtype=torch.float64))
    grads = {"in_proj_weight": ref.in_proj_weight.grad, "in_proj_bias": ref.in_proj_bias.grad,
             "out_proj.weight": ref.out_proj.weight.grad, "out_proj.bias": ref.out_proj.bias.grad}
    return out.detach().numpy(), t.grad.numpy(), {k: v.numpy() for k, v in grads.items()}


@pytest.mark.parametrize("groups", [1, 3])
def test_decoder_self_attention_module(groups):
    """The whole block (fused q/k projection, attention per group, out_proj) and every gradient."""
    torch.manual_seed(0)
    heads, c, batch, per = 8, 256, 2, 40
    m = MultiheadAttention(c, heads).to(_dev())
    with torch.no_grad():
        m.in_proj_bias.normal_(0, 0.1)
        m.out_proj.bias.normal_(0, 0.1)
    rng = np.random.default_rng(43)
    tgt = rng.standard_normal((batch, groups * per, c)).astype(np.float32)
    pos = rng.standard_normal((batch, groups * per, c)).astype(np.float32)
    grad = rng.standard_normal((batch, groups * per, c)).astype(np.float32)
    tt = _t(tgt).requires_grad_(True)
    out = decoder_self_attention(tt, _t(pos), m, groups)
    out.backward(_t(grad))
    want, want_dt, want_grads = _torch_reference(m, tgt, pos, groups, heads, grad)
    assert_close(_np(out), want, 1e-5, "out")
    assert_close(_np(tt.grad), want_dt, 1e-4, "grad tgt")
    for name, p in m.named_parameters():
        assert_close(_np(p.grad), want_grads[name], 1e-4, f"grad {name}")


def test_single_gradient_requests():
    from rfdetr_jax_amd.attention import _Layout, attention_backward, attention_forward

    rng = np.random.default_rng(44)
    q, k, v, g = (rng.standard_normal((2, 2, 50, 32)).astype(np.float32) for _ in range(4))
    lay = _Layout(2, 1, 2, 50, 32)
    tq, tk, tv = _t(q), _t(k), _t(v)
    out, stats = attention_forward(tq, tk, tv, lay, lay.strides_bhld)
    want = AT.sdpa_vjp(q, k, v, g)
    for i in range(3):
        needs = tuple(j == i for j in range(3))
        got = attention_backward(tq, tk, tv, out, stats, _t(g), lay, lay.strides_bhld, None, needs)
        for j in range(3):
            if j == i:
                assert_close(_np(got[j]), want[j], 1e-4, f"gradient {j}")
            else:
                assert got[j] is None


FUSED_LENGTHS = [1, 17, 32, 33, 64, 65, 129, 200, 256, 257, 300, 319, 320, 321]


@pytest.mark.parametrize("bf16", [False, True], ids=["f32", "bf16"])
@pytest.mark.parametrize("length", FUSED_LENGTHS)
def test_fused_backward_against_two_kernel_path(length, bf16, tune):
    """Head_dim 32 without a mask, up to 320 rows: one fused backward kernel (one workgroup per
    (slice, head): a wave per key block, two waves that form dQ from the dS tiles) against the
    oracle, and against the two-kernel path (MSDA_ATTN_FUSED=0) on the same forward; both write
    rowsum(dO * O) into entry 2 of the statistics. 321 rows take the two kernels either way."""
    from rfdetr_jax_amd.attention import _Layout, attention_backward, attention_forward

    b, h, d = 2, 3, 32
    _note(f"fused backward L={length} bf16={bf16}")
    rng = np.random.default_rng(45 + length)
    q, k, v, g = (rng.standard_normal((b, h, length, d)).astype(np.float32) for _ in range(4))
    if bf16:
        q, k, v, g = (bf16_round(x) for x in (q, k, v, g))
    dt = torch.bfloat16 if bf16 else torch.float32
    tol, cross = (2e-2, 1e-2) if bf16 else (1e-4, 1e-4)
    lay = _Layout(b, 1, h, length, d)
    tq, tk, tv, tg = (_t(x, dt) for x in (q, k, v, g))
    out, stats = attention_forward(tq, tk, tv, lay, lay.strides_bhld)
    fused = attention_backward(tq, tk, tv, out, stats, tg, lay, lay.strides_bhld)
    torch.cuda.synchronize()
    dsum_fused = _np(stats).reshape(b * h * length, 4)[:, 2].copy()
    tune({"MSDA_ATTN_FUSED": 0})
    split = attention_backward(tq, tk, tv, out, stats, tg, lay, lay.strides_bhld)
    torch.cuda.synchronize()
    dsum_split = _np(stats).reshape(b * h * length, 4)[:, 2]
    want_dsum = (g.astype(np.float64) * _np(out).astype(np.float64)).sum(-1).reshape(-1)
    assert_close(dsum_fused, want_dsum, 1e-5, "rowsum(dO * O), fused")
    assert_close(dsum_split, want_dsum, 1e-5, "rowsum(dO * O), two kernels")
    want = AT.sdpa_vjp(q, k, v, g)
    for name, a, c, w in zip("qkv", fused, split, want):
        assert_close(_np(a), w, tol, f"grad_{name} fused")
        assert_close(_np(c), w, tol, f"grad_{name} two kernels")
        assert_close(_np(a), _np(c).astype(np.float64), cross, f"grad_{name} fused against two kernels")


D32_LENGTHS = [1, 17, 63, 64, 65, 128, 129, 300, 320, 321, 480, 512, 513]


@pytest.mark.parametrize("length", D32_LENGTHS)
def test_bf16_forward_d32_against_chunked(length, tune):
    """bf16, head_dim 32, no mask, 16-byte aligned key and value rows, up to 512 rows: the forward
    that stages the whole key and value slice in LDS (scores leave the MFMA scaled and shifted,
    row sums add the rounded weights) against the oracle and the chunked kernel
    (MSDA_ATTN_FWD_D32=0). Its statistics give log2 sum_k 2^x (x = q.k log2(e) / sqrt(D)) as
    m + log2 l, and drive the backward. 513 rows take the chunked kernel either way."""
    from rfdetr_jax_amd.attention import _Layout, attention_backward, attention_forward

    b, h, d = 2, 3, 32
    _note(f"bf16 forward d32 L={length}")
    rng = np.random.default_rng(47 + length)
    q, k, v, g = (bf16_round(rng.standard_normal((b, h, length, d)).astype(np.float32)) for _ in range(4))
    lay = _Layout(b, 1, h, length, d)
    tq, tk, tv, tg = (_t(x, torch.bfloat16) for x in (q, k, v, g))
    out, stats = attention_forward(tq, tk, tv, lay, lay.strides_bhld)
    grads = attention_backward(tq, tk, tv, out, stats, tg, lay, lay.strides_bhld)
    torch.cuda.synchronize()
    st = _np(stats).reshape(b, h, length, 4)
    tune({"MSDA_ATTN_FWD_D32": 0})
    out2, _ = attention_forward(tq, tk, tv, lay, lay.strides_bhld)
    torch.cuda.synchronize()
    assert_close(_np(out), AT.sdpa(q, k, v, None), 2e-2, "out")
    assert_close(_np(out), _np(out2).astype(np.float64), 1e-2, "out against the chunked kernel")
    x = np.einsum("bhqd,bhkd->bhqk", q.astype(np.float64), k.astype(np.float64)) * (np.log2(np.e) / np.sqrt(d))
    xm = x.max(-1)
    lse2 = xm + np.log2(np.exp2(x - xm[..., None]).sum(-1))
    err = np.abs(st[..., 0] + st[..., 1] - lse2).max()
    assert err <= 1e-2, f"m + log2 l against log2 sum 2^x: max error {err}"
    for name, a, w in zip("qkv", grads, AT.sdpa_vjp(q, k, v, g)):
        assert_close(_np(a), w, 2e-2, f"grad_{name}")


@pytest.mark.parametrize("case", ["far_below", "unaligned_rows"])
def test_bf16_forward_d32_edge_cases(case, tune):
    """far_below: every score about -65 (log2 units), below the reference score's low limit, so it
    moves at the first chunk; equal scores give the mean of V. unaligned_rows: key and value rows
    with a stride of 36 elements (not 16-byte aligned) take the chunked kernel."""
    from rfdetr_jax_amd.attention import _Layout, attention_forward

    _note(f"bf16 forward d32 {case}")
    b, h, length, d = 2, 2, 200, 32
    rng = np.random.default_rng(48)
    v = bf16_round(rng.standard_normal((b, h, length, d)).astype(np.float32))
    if case == "far_below":
        q = np.full((b, h, length, d), 8.0, np.float32)
        k = -np.ones((b, h, length, d), np.float32)
        lay = _Layout(b, 1, h, length, d)
        out, _ = attention_forward(_t(q, torch.bfloat16), _t(k, torch.bfloat16), _t(v, torch.bfloat16), lay, lay.strides_bhld)
        want = np.broadcast_to(v.astype(np.float64).mean(axis=2, keepdims=True), v.shape)
        assert_close(_np(out), want, 2e-2, "mean of V")
        return
    q, k = (bf16_round(rng.standard_normal((b, h, length, d)).astype(np.float32)) for _ in range(2))
    pad = np.zeros((b, h, length, 36), np.float32)
    tq = _t(q, torch.bfloat16)
    tk = _t(np.concatenate([k, pad[..., :4]], -1), torch.bfloat16)[..., :d]
    tv = _t(np.concatenate([v, pad[..., :4]], -1), torch.bfloat16)[..., :d]
    lay = _Layout(b, 1, h, length, d)
    out, _ = attention_forward(tq, tk, tv, lay, lay.strides_bhld)
    assert_close(_np(out), AT.sdpa(q, k, v, None), 2e-2, "out")


@pytest.mark.parametrize("bf16", [False, True], ids=["f32", "bf16"])
@pytest.mark.parametrize("needs", [(True, True, False), (True, False, True), (True, False, False), (False, True, True)],
                         ids=["qk", "qv", "q", "kv"])
def test_gradient_subsets_head_dim_32(needs, bf16):
    """Head_dim 32: grad_q with one of grad_k / grad_v (the fused kernel, skipping the missing
    store), grad_q alone and grad_k with grad_v (the two-kernel path's halves)."""
    from rfdetr_jax_amd.attention import _Layout, attention_backward, attention_forward

    _note(f"gradient subset {needs} bf16={bf16}")
    rng = np.random.default_rng(46)
    q, k, v, g = (rng.standard_normal((2, 2, 150, 32)).astype(np.float32) for _ in range(4))
    if bf16:
        q, k, v, g = (bf16_round(x) for x in (q, k, v, g))
    dt = torch.bfloat16 if bf16 else torch.float32
    lay = _Layout(2, 1, 2, 150, 32)
    tq, tk, tv = (_t(x, dt) for x in (q, k, v))
    out, stats = attention_forward(tq, tk, tv, lay, lay.strides_bhld)
    got = attention_backward(tq, tk, tv, out, stats, _t(g, dt), lay, lay.strides_bhld, None, needs)
    torch.cuda.synchronize()
    want = AT.sdpa_vjp(q, k, v, g)
    for j in range(3):
        if needs[j]:
            assert_close(_np(got[j]), want[j], 2e-2 if bf16 else 1e-4, f"gradient {j}")
        else:
            assert got[j] is None


@pytest.mark.parametrize("path", ["bf16", "bf16-two-kernels", "f32"])
def test_unaligned_output_rows(path, tune):
    """Every kernel stores its results as 16-byte row pieces through an LDS transpose when the
    output rows allow it, element by element otherwise. Here the forward output and the gradients
    start 8 bytes (bf16) or 4 bytes (f32) into a buffer, with a row stride of 36 elements; the
    elements between the rows stay untouched."""
    import ctypes

    from rfdetr_jax_amd import _native
    from rfdetr_jax_amd.attention import _DTYPES, _Layout, _ptr, _stream, attention_forward

    bf16 = path != "f32"
    if path == "bf16-two-kernels":
        tune({"MSDA_ATTN_FUSED": 0})
    b, h, length, d, rs = 2, 3, 300, 32, 36
    off = 4 if bf16 else 1
    dt = torch.bfloat16 if bf16 else torch.float32
    _note(f"unaligned output rows {path}")
    rng = np.random.default_rng(47)
    q, k, v, g = (rng.standard_normal((b, h, length, d)).astype(np.float32) for _ in range(4))
    if bf16:
        q, k, v, g = (bf16_round(x) for x in (q, k, v, g))
    lay = _Layout(b, 1, h, length, d)
    tq, tk, tv, tg = (_t(x, dt) for x in (q, k, v, g))
    n = b * h * length * rs
    row_strides = [h * length * rs, 0, length * rs, rs]

    def views(count):
        bufs = [torch.zeros(n + off, dtype=dt, device=_dev()) for _ in range(count)]
        return bufs, [x[off:].view(b, h, length, rs)[..., :d] for x in bufs]

    def untouched(bufs):
        for x in bufs:
            assert not _np(x[off:].view(b, h, length, rs)[..., d:]).any() and not _np(x[:off]).any()

    tf, tg_ = (2e-2, 2e-2) if bf16 else (1e-5, 1e-4)
    obufs, (out_u,) = views(1)
    stats_u = torch.empty(b * h * length * 4, dtype=torch.float32, device=_dev())
    s = lay.strides_bhld(tq) + lay.strides_bhld(tk) + lay.strides_bhld(tv) + row_strides
    rc = _native.lib().msda_attention_fwd(_ptr(tq), _ptr(tk), _ptr(tv), _DTYPES[dt], _ptr(out_u), _ptr(stats_u), b, 1, h, length, d,
                                          (ctypes.c_int64 * 16)(*s), None, _stream(_dev()))
    _native.check(rc)
    torch.cuda.synchronize()
    assert_close(_np(out_u), AT.sdpa(q, k, v, None), tf, "out")
    untouched(obufs)

    out, stats = attention_forward(tq, tk, tv, lay, lay.strides_bhld)
    gbufs, grads = views(3)
    s = []
    for t in (tq, tk, tv, out, tg):
        s += lay.strides_bhld(t)
    for _ in grads:
        s += row_strides
    rc = _native.lib().msda_attention_bwd(_ptr(tq), _ptr(tk), _ptr(tv), _ptr(out), _ptr(stats), _ptr(tg), _DTYPES[dt],
                                          _ptr(grads[0]), _ptr(grads[1]), _ptr(grads[2]), b, 1, h, length, d,
                                          (ctypes.c_int64 * 32)(*s), None, _stream(_dev()))
    _native.check(rc)
    torch.cuda.synchronize()
    for name, got, want in zip("qkv", grads, AT.sdpa_vjp(q, k, v, g)):
        assert_close(_np(got), want, tg_, f"grad_{name}")
    untouched(gbufs)


@pytest.mark.parametrize("bf16", [False, True], ids=["f32", "bf16"])
@pytest.mark.parametrize("seed", range(6))
def test_fused_backward_random_shapes(seed, bf16):
    """Seeded random shapes through the fused backward (head_dim 32, no mask): 1-3 images, 1-4
    heads, 1-320 rows, rows padded to a random stride (a multiple of 4 elements, as the interface
    requires), against the float64 oracle."""
    import ctypes

    from rfdetr_jax_amd import _native
    from rfdetr_jax_amd.attention import _DTYPES, _Layout, _ptr, _stream, attention_forward

    rng = np.random.default_rng(1000 + seed)
    b, h, length, d = int(rng.integers(1, 4)), int(rng.integers(1, 5)), int(rng.integers(1, 321)), 32
    rs = d + 4 * int(rng.integers(0, 4))
    _note(f"fused random shape seed={seed} bf16={bf16}: b={b} h={h} L={length} row stride {rs}")
    dt = torch.bfloat16 if bf16 else torch.float32
    q, k, v, g = (rng.standard_normal((b, h, length, d)).astype(np.float32) for _ in range(4))
    if bf16:
        q, k, v, g = (bf16_round(x) for x in (q, k, v, g))

    def padded(x):
        buf = torch.zeros((b, h, length, rs), dtype=dt, device=_dev())
        if x is not None:
            buf[..., :d] = _t(x, dt)
        return buf[..., :d]

    tq, tk, tv, tg = (padded(x) for x in (q, k, v, g))
    lay = _Layout(b, 1, h, length, d)
    out, stats = attention_forward(tq, tk, tv, lay, lay.strides_bhld)
    grads = [padded(None) for _ in range(3)]
    s = []
    for t in (tq, tk, tv, out, tg, *grads):
        s += lay.strides_bhld(t)
    rc = _native.lib().msda_attention_bwd(_ptr(tq), _ptr(tk), _ptr(tv), _ptr(out), _ptr(stats), _ptr(tg), _DTYPES[dt],
                                          _ptr(grads[0]), _ptr(grads[1]), _ptr(grads[2]), b, 1, h, length, d,
                                          (ctypes.c_int64 * 32)(*s), None, _stream(_dev()))
    _native.check(rc)
    torch.cuda.synchronize()
    for name, got, want in zip("qkv", grads, AT.sdpa_vjp(q, k, v, g)):
        assert_close(_np(got), want, 2e-2 if bf16 else 1e-4, f"grad_{name}")


# --------------------------------------------------------------------------------------------
# attention dropout (layers.py:537-544): the keep decisions come from dropout_keep_mask, the same
# hash the kernels evaluate; the expected values are the float64 oracle with that mask.

DROP_SHAPES = {
    "decoder": (3, 8, 300, 32),
    "ragged64": (2, 2, 77, 64),
    "one": (1, 1, 1, 32),
}


def _keep(batch, heads, length, rate, seed, groups=1):
    from rfdetr_jax_amd.attention import dropout_keep_mask

    return dropout_keep_mask(batch, heads, length, rate, seed, groups=groups, device=_dev())


def test_dropout_keep_mask_statistics():
    """Keep rate 1 - rate (overall, for even and odd keys, which share one hash, and across
    neighbouring queries, within six standard deviations); the same (rate, seed) gives the same
    mask, another seed or another slice an independent one (disagreement 2 r (1 - r))."""
    b, h, length = 4, 8, 300
    for rate in (0.1, 0.5, 0.9):
        keep = _keep(b, h, length, rate, 1234).float()
        n = keep.numel()
        sd = (rate * (1 - rate) / n) ** 0.5
        _note(f"dropout rate {rate}: kept {keep.mean().item():.5f}")
        assert abs(keep.mean().item() - (1 - rate)) < 6 * sd
        for part in (keep[..., 0::2], keep[..., 1::2]):
            assert abs(part.mean().item() - (1 - rate)) < 6 * sd * 2 ** 0.5
        both = (keep[..., 0:298:2] * keep[..., 1:299:2]).mean().item()  # the two halves of one hash
        rows = (keep[:, :, 0::2, :] * keep[:, :, 1::2, :]).mean().item()
        sd2 = ((1 - rate) ** 2 * (1 - (1 - rate) ** 2) / (n / 2)) ** 0.5
        assert abs(both - (1 - rate) ** 2) < 6 * sd2 and abs(rows - (1 - rate) ** 2) < 6 * sd2
    k1 = _keep(b, h, length, 0.1, 1234)
    assert torch.equal(k1, _keep(b, h, length, 0.1, 1234))
    other = (k1 != _keep(b, h, length, 0.1, 1235)).float().mean().item()
    slices = (k1[0, 0] != k1[0, 1]).float().mean().item()
    assert abs(other - 0.18) < 0.005 and abs(slices - 0.18) < 0.01
    assert bool((_keep(1, 2, 40, 0.0, 5) == 1).all())


@pytest.mark.parametrize("bf16", [False, True], ids=["f32", "bf16"])
@pytest.mark.parametrize("masked", [False, True], ids=["nomask", "mask"])
@pytest.mark.parametrize("shape", sorted(DROP_SHAPES))
def test_dropout_against_oracle(shape, masked, bf16):
    """Output and gradients with dropout (rate 0.1) against the float64 oracle given the kernels'
    keep mask, with and without a key mask (a fully blocked row included)."""
    b, h, length, d = DROP_SHAPES[shape]
    rate, seed = 0.1, 1000 + length
    _note(f"dropout {shape} masked={masked} bf16={bf16}")
    rng = np.random.default_rng(43)
    q, k, v, g = (rng.standard_normal((b, h, length, d)).astype(np.float32) for _ in range(4))
    mask = None
    if masked:
        mask = rng.uniform(0, 1, (length, length)) < 0.2
        mask[:, -3:] = True
        mask[length // 2] = True
    if bf16:
        q, k, v, g = (bf16_round(t) for t in (q, k, v, g))
    dt = torch.bfloat16 if bf16 else None
    tq, tk, tv = (_t(x, dt).requires_grad_(True) for x in (q, k, v))
    out = scaled_dot_product_attention(tq, tk, tv, None if mask is None else _t(mask), dropout=rate, seed=seed)
    out.backward(_t(g, dt))
    keep = _np(_keep(b, h, length, rate, seed)).astype(bool)
    torch.cuda.synchronize()
    tf, tg = (2e-2, 2e-2) if bf16 else (1e-5, 1e-4)
    assert_close(_np(out), AT.sdpa(q, k, v, mask, keep, rate), tf, "out")
    for name, t, want in zip("qkv", (tq, tk, tv), AT.sdpa_vjp(q, k, v, g, mask, keep, rate)):
        assert_close(_np(t.grad), want, tg, f"grad_{name}")


@pytest.mark.parametrize("bf16", [False, True], ids=["f32", "bf16"])
def test_grouped_dropout_rows_layout(bf16):
    """Dropout on [B, G * P, C] rows with G groups: slice z = g * B + b of the keep mask belongs to
    group g of image b (the order of _split_groups)."""
    batch, groups, per, heads, d = 2, 3, 40, 4, 32
    c = heads * d
    rate, seed = 0.2, 9
    rng = np.random.default_rng(44)
    q, k, v, g = (rng.standard_normal((batch, groups * per, c)).astype(np.float32) for _ in range(4))
    if bf16:
        q, k, v, g = (bf16_round(x) for x in (q, k, v, g))
    dt = torch.bfloat16 if bf16 else None
    tq, tk, tv = (_t(x, dt).requires_grad_(True) for x in (q, k, v))
    out = grouped_attention(tq, tk, tv, heads, groups, dropout=rate, seed=seed)
    out.backward(_t(g, dt))
    keep = _np(_keep(batch, heads, per, rate, seed, groups=groups)).astype(bool)  # [G B, H, P, P]
    tf, tg = (2e-2, 2e-2) if bf16 else (1e-5, 1e-4)

    def heads_of(x):  # [G B, P, C] -> [G B, H, P, D]
        return x.reshape(x.shape[0], per, heads, d).transpose(0, 2, 1, 3)

    def back(x):  # [G B, H, P, D] -> [B, G P, C]
        return AT.merge_groups(x.transpose(0, 2, 1, 3).reshape(groups * batch, per, c), batch)

    qs, ks, vs, gs = (heads_of(AT.split_groups(x, per)) for x in (q, k, v, g))
    assert_close(_np(out), back(AT.sdpa(qs, ks, vs, None, keep, rate)), tf, "out")
    for name, t, want in zip("qkv", (tq, tk, tv), AT.sdpa_vjp(qs, ks, vs, gs, None, keep, rate)):
        assert_close(_np(t.grad), back(want), tg, f"grad_{name}")


def test_dropout_module_training_and_eval():
    """MultiheadAttention(dropout=0.1): in training a call draws its seed from torch's generator
    (repeatable under torch.manual_seed, different otherwise) and its gradients are finite; in
    eval the module is the plain attention; rate 0 is the plain path bit for bit; rate 1 gives
    zeros (flax's Dropout at rate 1)."""
    torch.manual_seed(0)
    m = MultiheadAttention(64, 2, dropout=0.1).to(_dev())
    x = torch.randn(2, 50, 64, device=_dev(), requires_grad=True)
    m.train()
    torch.manual_seed(5)
    y1 = m(x, x, x)
    torch.manual_seed(5)
    y2 = m(x, x, x)
    torch.manual_seed(6)
    y3 = m(x, x, x)
    assert torch.equal(y1, y2) and not torch.equal(y1, y3)
    y1.square().sum().backward()
    assert torch.isfinite(x.grad).all() and torch.isfinite(m.in_proj_weight.grad).all()
    m.eval()
    plain = MultiheadAttention(64, 2).to(_dev())
    plain.load_state_dict(m.state_dict())
    with torch.no_grad():
        assert torch.equal(m(x, x, x), plain(x, x, x))
    q, k, v = (torch.randn(1, 2, 33, 32, device=_dev()) for _ in range(3))
    assert torch.equal(scaled_dot_product_attention(q, k, v, dropout=0.0, seed=3), scaled_dot_product_attention(q, k, v))
    assert not scaled_dot_product_attention(q, k, v, dropout=1.0).any()


SPLIT_RANGES = ["tiny", "large", "late_keys", "small_channels", "zero_first", "row_range"]


def _split_inputs(kind, shape):
    rng = np.random.default_rng(61)
    b, h, length, d = shape
    q, k, v, g = (rng.standard_normal(shape).astype(np.float32) for _ in range(4))
    if kind == "tiny":  # far below f16's range, some values below 2^-126
        k, v, g = k * np.float32(1e-32), v * np.float32(1e-36), g * np.float32(1e-30)
    elif kind == "large":  # far above it
        q, k, v, g = q * np.float32(1e-12), k * np.float32(1e12), v * np.float32(1e30), g * np.float32(1e-20)
    elif kind == "late_keys":  # rows past the first 64 overflow the scale taken from those
        first = min(64, length // 2)
        q, k[:, :, first:], v[:, :, first:] = q / np.float32(200), k[:, :, first:] * np.float32(200), v[:, :, first:] * np.float32(200)
    elif kind == "small_channels":  # channels that the shared scale would leave without their low bits
        v = v * np.where(np.arange(d) % 3 == 0, 1e-7, 1.0).astype(np.float32)
    elif kind == "zero_first":  # nothing to take a scale from
        k[:, :, :64], v[:, :, :64] = 0.0, 0.0
    else:  # rows of very different sizes
        size = 10.0 ** rng.uniform(-8, 0, (b, h, length, 1))
        q, g = (q * size).astype(np.float32), (g * size[:, :, ::-1]).astype(np.float32)
    return q, k, v, g


@pytest.mark.parametrize("kind", SPLIT_RANGES)
@pytest.mark.parametrize("shape", [(2, 2, 300, 32), (1, 3, 65, 64), (2, 1, 33, 32)], ids=str)
def test_split_operands_of_any_size(shape, kind):
    """f32 operands are split into 16-bit terms: sizes and spreads that 16 bits do not cover, against the
    float64 oracle. Errors are relative to the 2-norm of each output channel and of each grad_q row
    (a shared scale must not cost the small ones their bits): a few hundred terms at f32's 2^-24 and
    the rounding of the scores, 8e-6."""
    _note(f"sdpa split operands {kind} {shape}")
    q, k, v, g = _split_inputs(kind, shape)
    tq, tk, tv = (_t(x).requires_grad_(True) for x in (q, k, v))
    out = scaled_dot_product_attention(tq, tk, tv)
    out.backward(_t(g))
    torch.cuda.synchronize()

    def err(got, want, axes):
        got, want = got.detach().double().cpu().numpy(), np.asarray(want, np.float64)
        n = np.sqrt((want ** 2).sum(axes))
        # below 2^-120 f32 itself has few bits left
        ok = n > 2.0 ** -120
        return float((np.sqrt(((got - want) ** 2).sum(axes))[ok] / n[ok]).max()) if ok.any() else 0.0

    want = AT.sdpa(q, k, v)
    gq, gk, gv = AT.sdpa_vjp(q, k, v, g)
    _note(f"errors: {err(out, want, 2):.2g} {err(tq.grad, gq, 3):.2g} {err(tk.grad, gk, (2, 3)):.2g} {err(tv.grad, gv, (2, 3)):.2g}")
    assert err(out, want, 2) <= 8e-6, "out"
    assert err(tv.grad, gv, (2, 3)) <= 8e-6, "grad_v"
    if kind != "tiny":  # grad_q and grad_k are products of what is tiny: below f32's range
        assert err(tq.grad, gq, 3) <= 1e-4, "grad_q"  # a row's terms cancel: dP - rowsum(dO O)
        assert err(tk.grad, gk, (2, 3)) <= 1e-5, "grad_k"


@pytest.mark.parametrize("where", ["q", "k", "v", "g"])
@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, 3.4e38], ids=str)
def test_split_operands_nonfinite(tune, where, value):
    """An infinity, a NaN or a value that 16 bits round to infinity gives what the f32 kernels give: the
    forward with a mask that blocks nothing, the backward in its two-kernel form."""
    rng = np.random.default_rng(62)
    x = {n: rng.standard_normal((2, 2, 96, 32)).astype(np.float32) for n in "qkvg"}
    x[where][0, 1, 70, 5] = value
    if value == 3.4e38:  # finite scores: its partner is small
        x[{"q": "k", "k": "q", "v": "g", "g": "v"}[where]][0, 1, :, 5] *= 1e-36
    got, want = [], []
    for res, mask, fused in ((got, None, 1), (want, _t(np.zeros((96, 96), bool)), 0)):
        tune({"MSDA_ATTN_FUSED": fused})
        t = {n: _t(x[n]).requires_grad_(True) for n in "qkv"}
        out = scaled_dot_product_attention(t["q"], t["k"], t["v"], mask)
        res += [out, *torch.autograd.grad(out, list(t.values()), _t(x["g"]))]
    torch.cuda.synchronize()
    for name, a, b in zip(("out", "grad_q", "grad_k", "grad_v"), got, want):
        a, b = _np(a).astype(np.float64), _np(b).astype(np.float64)
        fine = np.isfinite(b)
        assert np.array_equal(fine, np.isfinite(a)), name
        assert np.array_equal(np.isnan(a), np.isnan(b)), name
        np.testing.assert_allclose(a[fine], b[fine], rtol=1e-4, atol=1e-5 * max(1.0, np.abs(b[fine]).max()))


@pytest.mark.parametrize("shape", [(2, 2, 1, 32), (2, 2, 50, 32), (1, 2, 300, 32), (2, 1, 62, 64), (1, 1, 600, 64)], ids=str)
def test_split_forward_statistics(shape):
    """The f32 forward's statistics: entry 0 + entry 1 is log2 of the sum of 2^x, and entry 1 (log2 of a sum in
    [1, 2) and what entry 0 rounds off, at most 2^-20 for entries below 16) is small, so that a backward's x -
    entry 0 - entry 1 is rounded at its own size. Bound: 32 sums a row and chunk of 2^-24 of the sum each, in log2
    units 2.8e-6, and as much for the scores (64 products of 2^-22 of a score of 8 at most, mostly far below)."""
    b, h, length, d = shape
    from rfdetr_jax_amd.attention import _Layout, attention_forward

    _note(f"split forward statistics {shape}")
    rng = np.random.default_rng(91 + length)
    q, k, v = (rng.standard_normal((b, h, length, d)).astype(np.float32) for _ in range(3))
    lay = _Layout(b, 1, h, length, d)
    _, stats = attention_forward(_t(q), _t(k), _t(v), lay, lay.strides_bhld)
    torch.cuda.synchronize()
    st = _np(stats).reshape(b, h, length, 4).astype(np.float64)
    x = np.einsum("bhqd,bhkd->bhqk", q.astype(np.float64), k.astype(np.float64)) * (np.log2(np.e) / np.sqrt(d))
    want = x.max(-1) + np.log2(np.exp2(x - x.max(-1, keepdims=True)).sum(-1))
    assert np.abs(st[..., 0] + st[..., 1] - want).max() <= 5.6e-6
    assert st[..., 1].min() >= -(2.0 ** -20) and st[..., 1].max() <= 1.0 + 2.0 ** -20


def _row_range_inputs(kind, shape):
    """Keys, values and queries whose rows differ so much in size that a scale shared by rows, or taken from
    the first of them, would cost some rows their low bits."""
    rng = np.random.default_rng(63)
    q, k, v = (rng.standard_normal(shape).astype(np.float32) for _ in range(3))
    if kind.startswith("zero_first"):  # nothing in the first chunk; scores of ordinary size from small keys
        size = np.float32(kind[len("zero_first_"):])
        k[:, :, :64] = 0.0
        q, k = q / size, k * size
    elif kind.startswith("large_row"):  # one value row far above the others, which no query attends to
        q[..., 0], k[:, :, 5, 0] = 3.0, -250.0
        v[:, :, 5] *= np.float32(kind[len("large_row_"):])
    elif kind == "value_rows":  # every query attends to its own key; values from 1e-8 to 1
        k = (k / np.linalg.norm(k, axis=-1, keepdims=True) * 12.0).astype(np.float32)
        q = k * np.float32(np.sqrt(shape[-1]) / 3.0)
        v = (v * 10.0 ** rng.uniform(-8, 0, (*shape[:3], 1))).astype(np.float32)
    else:  # keys from 1e-8 to 1
        k = (k * 10.0 ** rng.uniform(-8, 0, (*shape[:3], 1))).astype(np.float32)
    return q, k, v


ROW_RANGES = ["zero_first_1e-4", "zero_first_1e-6", "zero_first_1e4", "large_row_1e6", "large_row_1e8", "value_rows", "key_rows"]


@pytest.mark.parametrize("kind", ROW_RANGES)
@pytest.mark.parametrize("shape", [(2, 2, 300, 32), (1, 3, 130, 64)], ids=str)
def test_split_forward_keeps_every_row(shape, kind):
    """The maskless f32 forward (split operands) against the f32 matrix kernel (a mask that blocks nothing),
    row by row: the largest error of a query's output row, relative to the row's sum of weights times |values|,
    and of the statistics, is at most twice that kernel's and a rounding of f32 (2^-23; the statistics' log2
    of a sum near 2^8 is rounded at 2^-20)."""
    from rfdetr_jax_amd.attention import _Layout, attention_forward

    _note(f"split forward rows {kind} {shape}")
    q, k, v = _row_range_inputs(kind, shape)
    b, h, length, d = shape
    lay = _Layout(b, 1, h, length, d)
    x = np.matmul(q.astype(np.float64), k.astype(np.float64).swapaxes(-1, -2)) / np.sqrt(d)
    top = x.max(-1, keepdims=True)
    weights = np.exp(x - top)
    total = weights.sum(-1, keepdims=True)
    weights /= total
    want, size = weights @ v.astype(np.float64), weights @ np.abs(v.astype(np.float64))
    log2_sum = ((top + np.log(total)) * np.log2(np.e))[..., 0]
    errors = []
    for mask in (None, _t(np.zeros((length, length), bool))):
        out, stats = attention_forward(_t(q), _t(k), _t(v), lay, lay.strides_bhld, mask)
        torch.cuda.synchronize()
        st = _np(stats).reshape(b, h, length, 4).astype(np.float64)
        rows = np.linalg.norm(_np(out).astype(np.float64) - want, axis=-1) / np.linalg.norm(size, axis=-1)
        errors.append((rows.max(), np.abs(st[..., 0] + st[..., 1] - log2_sum).max()))
    (out_split, st_split), (out_f32, st_f32) = errors
    _note(f"rows: {out_split:.2g} against {out_f32:.2g}; statistics: {st_split:.2g} against {st_f32:.2g}")
    assert out_split <= 2 * out_f32 + 2.0 ** -23
    assert st_split <= 2 * st_f32 + 2.0 ** -20


@pytest.mark.parametrize("d", [32, 64])
def test_split_forward_of_one_key_returns_the_value(d):
    """With one key the weight is 1 and every bit of the value comes back, as from the f32 kernel."""
    rng = np.random.default_rng(64)
    q, k = (_t(rng.standard_normal((4, 8, 1, d)).astype(np.float32)) for _ in range(2))
    v = _t((rng.standard_normal((4, 8, 1, d)) * 10.0 ** rng.uniform(-9, 9, (4, 8, 1, d))).astype(np.float32))
    q[0] = 0.0  # a score of exactly 0, the others' weight is 2^x for a rounded x: f32's rounding of w v / w
    out = scaled_dot_product_attention(q, k, v)
    assert torch.equal(out[0], v[0])
    assert float(((out - v).abs() / v.abs()).max()) <= 2.0 ** -22


@pytest.mark.parametrize("where", ["g", "v", "k", "q"])
@pytest.mark.parametrize("length", [300, 33])
def test_split_backward_of_tiny_tensors(tune, where, length):
    """Elements of 1e-34, whose low bits leave bf16's range, cost the fused backward no bits: its gradients'
    errors against float64 are at most twice the two-kernel f32 backward's (and 2^-23)."""
    rng = np.random.default_rng(65)
    shape = (2, 2, length, 32)
    x = {n: rng.standard_normal(shape).astype(np.float32) for n in "qkvg"}
    x[where] *= np.float32(1e-34)
    if where in "qk":  # gradients within f32's range
        x["g"] *= np.float32(1e10)
        x["q" if where == "k" else "k"] *= np.float32(1e10)
    want = AT.sdpa_vjp(x["q"], x["k"], x["v"], x["g"])
    errors = []
    for fused in (1, 0):
        tune({"MSDA_ATTN_FUSED": fused})
        t = [_t(x[n]).requires_grad_(True) for n in "qkv"]
        got = torch.autograd.grad(scaled_dot_product_attention(*t), t, _t(x["g"]))
        torch.cuda.synchronize()
        errors.append([np.linalg.norm(_np(a).astype(np.float64) - b) / np.linalg.norm(b) for a, b in zip(got, want)])
    _note(f"tiny {where} {length}: {errors}")
    for name, split, f32 in zip("qkv", *errors):
        assert split <= 2 * f32 + 2.0 ** -23, name


def test_masked_attention_saved_tensor_hooks_and_types():
    """The Python autograd function (mask or dropout): saved tensors that hooks hand back in another type or layout
    reach the kernels by their values, other shapes and mixed input types are refused."""
    torch.manual_seed(4)
    ins = [torch.randn(2, 2, 40, 32, device=_dev()) for _ in range(3)]
    mask = torch.rand(40, 40, device=_dev()) < 0.2
    g = torch.randn(2, 2, 40, 32, device=_dev())

    def grads(unpack):
        t = [x.clone().requires_grad_() for x in ins]
        with torch.autograd.graph.saved_tensors_hooks(lambda x: x, unpack):
            out = scaled_dot_product_attention(*t, mask)
        return torch.autograd.grad(out, t, g)

    def floats(f):
        return lambda x: f(x) if x.dtype == torch.float32 else x

    pairs = ((floats(lambda x: x.bfloat16()), floats(lambda x: x.bfloat16().float())),
             (floats(lambda x: x.movedim(-1, 0).contiguous().movedim(0, -1)), lambda x: x))
    for got, want in pairs:
        for a, b in zip(grads(got), grads(want)):
            assert a.dtype == b.dtype and torch.equal(a, b)
    with pytest.raises(ValueError, match="other shapes"):
        grads(floats(lambda x: x[..., :-4]))
    for i in range(3):
        mixed = [x.bfloat16() if j == i else x for j, x in enumerate(ins)]
        with pytest.raises(TypeError, match="one type"):
            scaled_dot_product_attention(*mixed, mask)
        with pytest.raises(TypeError, match="one type"):
            scaled_dot_product_attention(*mixed)
