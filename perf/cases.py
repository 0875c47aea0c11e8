"""The work a user of this package has it do, as timed cases.

Each case is one pass through a public entry point of ``rfdetr_jax_amd``, at sizes of the RF-DETR
decoder: the deformable-attention core (inference, and training with its three gradients), the core
with the MSDeformAttn prologue fused, the value projection, the decoder's grouped self-attention,
the segmentation loss's point sampling, and the whole MSDeformAttn module. ``op`` names the entry
point; the other keys are its sizes. :func:`draw` gives further cases of the same ranges.
"""

import os
import sys

import torch
import torch.nn.functional as F

sys.path.insert(0, os.path.join(os.getcwd(), "rf-detr-jax_amd"))

from rfdetr_jax_amd import (  # noqa: E402
    MSDeformAttn,
    grouped_attention,
    ms_deform_attn_core_rows,
    ms_deform_attn_fused,
    point_sample,
    value_proj_rows,
)

DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16}


def listed():
    return [
        # Serving one or two images with the Nano decoder: the smallest call, launch latency.
        {"name": "core_infer_b2_f32", "op": "core", "train": False, "dtype": "f32", "batch": 2, "heads": 16, "head_dim": 16,
         "queries": 300, "levels": "24x24", "points": 2, "uniform": False},
        # Throughput inference at a larger resolution, bf16 memory, locations past the image border.
        {"name": "core_infer_b64_bf16", "op": "core", "train": False, "dtype": "bf16", "batch": 64, "heads": 16, "head_dim": 16,
         "queries": 300, "levels": "36x36", "points": 2, "uniform": True},
        # Group-DETR training of the Nano decoder: 13 groups x 300 queries (the package's headline shape).
        {"name": "core_train_group_f32", "op": "core", "train": True, "dtype": "f32", "batch": 8, "heads": 16, "head_dim": 16,
         "queries": 3900, "levels": "24x24", "points": 2, "uniform": False},
        # Training with two levels of a 640-pixel image, bf16 memory.
        {"name": "core_train_two_level_bf16", "op": "core", "train": True, "dtype": "bf16", "batch": 8, "heads": 16, "head_dim": 16,
         "queries": 300, "levels": "80x80,20x20", "points": 4, "uniform": False},
        # Training with MSDeformAttn's default sizes (8 heads x 32, 4 levels, 4 points), box reference
        # points and an image that is not square.
        {"name": "fused_train_four_level_f32", "op": "fused", "dtype": "f32", "batch": 8, "heads": 8, "head_dim": 32,
         "queries": 900, "levels": "64x85,32x43,16x22,8x11", "points": 4, "ref_dim": 4},
        # The value path of the Nano decoder in training: 8 images of 24 x 24 positions, some padded.
        {"name": "value_proj_train_f32", "op": "value_proj", "train": True, "dtype": "f32", "batch": 8, "heads": 16, "head_dim": 16,
         "length": 576, "padded": True},
        # The value path at two levels of a 640-pixel image (80 x 80 + 20 x 20 positions), bf16.
        {"name": "value_proj_train_bf16", "op": "value_proj", "train": True, "dtype": "bf16", "batch": 16, "heads": 16, "head_dim": 16,
         "length": 6800, "padded": False},
        # The decoder's self-attention in training: 13 query groups of 300, q and k from one product.
        {"name": "attention_train_f32", "op": "attention", "train": True, "dtype": "f32", "batch": 8, "groups": 13, "heads": 8,
         "head_dim": 32, "length": 300},
        # The same in bf16, twice the images.
        {"name": "attention_train_bf16", "op": "attention", "train": True, "dtype": "bf16", "batch": 16, "groups": 13, "heads": 8,
         "head_dim": 32, "length": 300},
        # The decoder's self-attention at inference: one group.
        {"name": "attention_infer_f32", "op": "attention", "train": False, "dtype": "f32", "batch": 32, "groups": 1, "heads": 8,
         "head_dim": 32, "length": 300},
        # The segmentation loss on 400 masks: candidate points, the chosen points with the gradient of
        # the logits, and the labels at the same points.
        {"name": "mask_points_train_f32", "op": "points", "masks": 400, "height": 112, "width": 112, "points": 784},
        # The whole cross-attention module at inference: a padded image that is not square.
        {"name": "module_infer_f32", "op": "module", "batch": 16, "heads": 16, "head_dim": 16, "queries": 300,
         "levels": "27x38", "points": 2},
    ]


def _between(rng, lo, hi):
    """A whole number, its logarithm uniform."""
    return max(lo, min(hi, round(lo * (hi / lo) ** rng.random())))


def _levels(rng, count, most):
    """`count` levels, each half the one before, of an image that is seldom square."""
    h, w = _between(rng, 16, most), _between(rng, 16, most)
    out = []
    for _ in range(count):
        out.append(f"{h}x{w}")
        h, w = max(2, -(-h // 2)), max(2, -(-w // 2))
    return ",".join(out)


def draw(rng):
    op = rng.choice(["core", "core", "fused", "value_proj", "attention", "attention", "points", "module"])
    dtype = rng.choice(["f32", "bf16"])
    heads, head_dim = rng.choice([(16, 16), (8, 32)])
    if op == "core":
        count = rng.choice([1, 1, 2, 4])
        return {"op": op, "train": rng.random() < 0.6, "dtype": dtype, "batch": _between(rng, 1, 8), "heads": heads,
                "head_dim": head_dim, "queries": _between(rng, 100, 3900 // count), "levels": _levels(rng, count, 60),
                "points": rng.choice([2, 4]) if count == 1 else 4, "uniform": rng.random() < 0.25}
    if op == "fused":
        count = rng.choice([1, 2, 4])
        return {"op": op, "dtype": dtype, "batch": _between(rng, 1, 8), "heads": heads, "head_dim": head_dim,
                "queries": _between(rng, 100, 900), "levels": _levels(rng, count, 64), "points": 2 if count == 1 else 4,
                "ref_dim": rng.choice([2, 4])}
    if op == "value_proj":
        return {"op": op, "train": rng.random() < 0.7, "dtype": dtype, "batch": _between(rng, 1, 16), "heads": heads,
                "head_dim": head_dim, "length": _between(rng, 300, 6800), "padded": rng.random() < 0.5}
    if op == "attention":
        return {"op": op, "train": rng.random() < 0.6, "dtype": dtype, "batch": _between(rng, 1, 8), "groups": rng.choice([1, 13]),
                "heads": 8, "head_dim": rng.choice([32, 32, 32, 64]), "length": _between(rng, 50, 300)}
    if op == "points":
        h, w = rng.randint(64, 112), rng.randint(64, 112)
        return {"op": op, "masks": _between(rng, 16, 400), "height": h, "width": w, "points": h * w // 16}
    return {"op": op, "batch": _between(rng, 1, 16), "heads": heads, "head_dim": head_dim, "queries": _between(rng, 100, 900),
            "levels": _levels(rng, rng.choice([1, 2]), 40), "points": rng.choice([2, 4])}


# -- sizes --------------------------------------------------------------------------------------


def _shapes(case):
    return tuple(tuple(int(x) for x in s.split("x")) for s in case["levels"].split(","))


def _positions(case):
    return sum(h * w for h, w in _shapes(case))


def work(case):
    op = case["op"]
    size = 2 if case.get("dtype") == "bf16" else 4
    if op in ("core", "fused"):
        heads, d = case["heads"], case["head_dim"]
        samples = case["batch"] * case["queries"] * heads * len(_shapes(case)) * case["points"]
        value = case["batch"] * heads * _positions(case) * d * size
        rows = case["batch"] * case["queries"] * heads * d * 4
        given = samples * 12 + (case["batch"] * case["queries"] * len(_shapes(case)) * case["ref_dim"] * 4 if op == "fused" else 0)
        train = op == "fused" or case["train"]
        # forward: value, samples in, rows out; backward: value, samples and rows in, gradients out
        return {"bytes": value + given + rows + (2 * value + 2 * given + rows if train else 0),
                "flops": samples * d * 8 * (4 if train else 1)}
    if op == "value_proj":
        m, c = case["batch"] * case["length"], case["heads"] * case["head_dim"]
        act, weight = m * c * size, (c * c + c) * 4
        mask = m if case["padded"] else 0
        if not case["train"]:
            return {"bytes": 2 * act + weight + mask, "flops": 2 * m * c * c}
        return {"bytes": 5 * act + 3 * weight + 2 * mask, "flops": 6 * m * c * c}
    if op == "attention":
        slices = case["batch"] * case["groups"] * case["heads"]
        act = slices * case["length"] * case["head_dim"] * size
        pair = slices * case["length"] ** 2 * case["head_dim"] * 2
        if not case["train"]:
            return {"bytes": 4 * act, "flops": 2 * pair}
        return {"bytes": 12 * act, "flops": 6 * pair}
    if op == "points":
        plane, n, p = case["height"] * case["width"], case["masks"], case["points"]
        # the logits read by both samplings and by none of the gradients; labels read at the points only
        return {"bytes": 4 * n * (plane + 3 * p * 3 + p * 3 + (plane + p * 3) + p * 4), "flops": n * p * 8 * 5}
    b, c, s, q = case["batch"], case["heads"] * case["head_dim"], _positions(case), case["queries"]
    samples = b * q * case["heads"] * len(_shapes(case)) * case["points"]
    per = case["heads"] * len(_shapes(case)) * case["points"] * 3
    return {"bytes": 4 * (b * s * c + 2 * b * q * c + b * q * len(_shapes(case)) * 4 + 2 * c * c + per * c) + b * s,
            "flops": 2 * b * s * c * c + 2 * b * q * c * (c + per) + samples * case["head_dim"] * 8}


def tolerance(case):
    # About four times the largest error against exact() that was measured: 32-bit sums 1.7e-7 (attention
    # 5.5e-7, the module with its four products 9.5e-7); bf16 results, rounded once per value, 2e-3
    # (attention, whose softmax weights and their gradients are rounded too, 2.5e-3).
    op, bf16 = case["op"], case.get("dtype") == "bf16"
    if bf16 and (op != "core" or case["train"]):
        return {"rel": 1e-2 if op == "attention" else 8e-3}
    return {"rel": {"attention": 2e-6, "module": 4e-6}.get(op, 1e-6)}


# -- inputs -------------------------------------------------------------------------------------


class _Draw:
    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(self, *shape, std=1.0):
        return torch.randn(shape, generator=self.g, device="cuda") * std

    def uniform(self, *shape, lo=0.0, hi=1.0):
        return torch.rand(shape, generator=self.g, device="cuda") * (hi - lo) + lo


def _reference(rng, batch, queries, levels, ref_dim):
    centre = rng.uniform(batch, queries, 1, 2, lo=0.05, hi=0.95)
    ref = centre if ref_dim == 2 else torch.cat([centre, rng.uniform(batch, queries, 1, 2, lo=0.05, hi=0.5)], -1)
    return ref.expand(-1, -1, levels, -1).contiguous()


def prepare(case, seed):
    rng = _Draw(seed)
    op, dt = case["op"], DTYPES[case.get("dtype", "f32")]
    state = {"case": case}
    if op in ("core", "fused"):
        b, h, d, q, p = case["batch"], case["heads"], case["head_dim"], case["queries"], case["points"]
        shapes = _shapes(case)
        levels = len(shapes)
        state["shapes"] = shapes
        train = op == "fused" or case["train"]
        value = rng.normal(b * h, _positions(case), d).to(dt)
        logits = rng.normal(b, q, h, levels * p)
        if op == "core":
            if case["uniform"]:
                loc = rng.uniform(b, q, h, levels, p, 2, lo=-0.1, hi=1.1)
            else:
                loc = rng.uniform(b, q, 1, 1, 1, 2) + rng.normal(b, q, h, levels, p, 2, std=0.05)
            inputs = [value, loc, torch.softmax(logits, -1)]
        else:
            inputs = [value, _reference(rng, b, q, levels, case["ref_dim"]), rng.normal(b, q, h, levels, p, 2, std=2.0), 2 * logits]
        state["inputs"] = [t.requires_grad_(train) for t in inputs]
        if train:
            state["grad"] = rng.normal(b, q, h * d)
    elif op == "value_proj":
        b, s, c = case["batch"], case["length"], case["heads"] * case["head_dim"]
        train = case["train"]
        x = rng.normal(b, s, c).to(dt)
        weight, bias = rng.normal(c, c, std=c ** -0.5), rng.normal(c)
        state["inputs"] = [t.requires_grad_(train) for t in (x, weight, bias)]
        state["mask"] = _padding(b, s) if case["padded"] else None
        if train:
            state["grad"] = rng.normal(b * case["heads"], s, case["head_dim"]).to(dt)
    elif op == "attention":
        rows, c = (case["batch"], case["groups"] * case["length"]), case["heads"] * case["head_dim"]
        qk, v = rng.normal(*rows, 2 * c).to(dt), rng.normal(*rows, c).to(dt)
        # q and k are halves of one product's rows, as the module has them
        state["inputs"] = [t.detach().requires_grad_(case["train"]) for t in (qk[..., :c], qk[..., c:], v)]
        if case["train"]:
            state["grad"] = rng.normal(*rows, c).to(dt)
    elif op == "points":
        n, p, hw = case["masks"], case["points"], (case["height"], case["width"])
        state["logits"] = rng.normal(n, 1, *hw).requires_grad_(True)
        state["labels"] = (rng.uniform(n, 1, *hw) > 0.5).float()
        state["candidates"] = rng.uniform(n, 3 * p, 2)
        state["chosen"] = rng.uniform(n, p, 2)
        state["grad"] = rng.normal(n, 1, p)
    else:
        b, q, c, shapes = case["batch"], case["queries"], case["heads"] * case["head_dim"], _shapes(case)
        m = MSDeformAttn(c, len(shapes), case["heads"], case["points"]).cuda()
        with torch.no_grad():  # as after some training: no projection is zero
            for lin, std in ((m.sampling_offsets, 0.5), (m.attention_weights, 1.0), (m.value_proj, 1.0), (m.output_proj, 1.0)):
                lin.weight.copy_(rng.normal(*lin.weight.shape, std=std * c ** -0.5))
                if lin is not m.sampling_offsets:
                    lin.bias.copy_(rng.normal(*lin.bias.shape, std=0.5))
        s = _positions(case)
        state.update(module=m.eval(), shapes=shapes, query=rng.normal(b, q, c), memory=rng.normal(b, s, c),
                     ref=_reference(rng, b, q, len(shapes), 4), mask=_padding(b, s))
    return state


def _padding(batch, length):
    """True on the padded tail of each image, from none of it to an eighth."""
    keep = length - (torch.arange(batch, device="cuda") * length) // (8 * max(1, batch - 1))
    return torch.arange(length, device="cuda")[None, :] >= keep[:, None]


# -- one pass -----------------------------------------------------------------------------------


def run(state):
    case = state["case"]
    op = case["op"]
    if op == "module":
        with torch.no_grad():
            return state["module"](state["query"], state["ref"], state["memory"], state["shapes"], state["mask"])
    if op == "points":
        logits = state["logits"]
        with torch.no_grad():
            candidates = point_sample(logits, state["candidates"])
            labels = point_sample(state["labels"], state["chosen"], mode="nearest")
        chosen = point_sample(logits, state["chosen"])
        (grad,) = torch.autograd.grad(chosen, logits, state["grad"])
        return {"candidates": candidates, "labels": labels, "chosen": chosen, "grad": grad}
    inputs = state["inputs"]
    if op == "core":
        value, loc, attn = inputs
        out = ms_deform_attn_core_rows(value, state["shapes"], loc, attn)
    elif op == "fused":
        value, ref, off, logits = inputs
        out = ms_deform_attn_fused(value, state["shapes"], ref, off, logits)
    elif op == "value_proj":
        out = value_proj_rows(*inputs, case["heads"], state["mask"])
    else:
        out = grouped_attention(*inputs, case["heads"], case["groups"])
    if "grad" not in state:
        return out
    return (out, *torch.autograd.grad(out, inputs, state["grad"]))


# -- the same in 64 bits ------------------------------------------------------------------------
# Pixel coordinates keep their 32-bit formula (their floor is part of the operation); all else is 64-bit.


def _pixel(loc, size):
    """((2 loc - 1 + 1) size - 1) / 2 in 32 bits, with the derivative d/dloc = size."""
    at = (((2 * loc.detach().float() - 1) + 1) * size - 1) / 2
    return at.double() + (loc - loc.detach()) * size


def _sample64(value, shapes, loc, attn):
    """value [B*H, S, D], loc [B, Q, H, L, P, 2], attn [B, Q, H, L*P] -> [B, Q, H*D], zero padding."""
    b, q, h, levels, p, _ = loc.shape
    d = value.shape[-1]
    attn = attn.view(b, q, h, levels, p)
    out, start = 0, 0
    for lv, (hh, ww) in enumerate(shapes):
        at = loc[:, :, :, lv].permute(0, 2, 1, 3, 4).reshape(b * h, q * p, 2)
        a = attn[:, :, :, lv].permute(0, 2, 1, 3).reshape(b * h, q * p)
        x, y = _pixel(at[..., 0], ww), _pixel(at[..., 1], hh)
        x0, y0 = x.detach().floor(), y.detach().floor()
        fx, fy = x - x0, y - y0
        total = 0
        for dy, wy in ((0, 1 - fy), (1, fy)):
            for dx, wx in ((0, 1 - fx), (1, fx)):
                cx, cy = (x0 + dx).long(), (y0 + dy).long()
                inside = (cx >= 0) & (cx < ww) & (cy >= 0) & (cy < hh)
                row = start + cy.clamp(0, hh - 1) * ww + cx.clamp(0, ww - 1)
                taken = torch.gather(value, 1, row[..., None].expand(-1, -1, d))
                total = total + taken * (wx * wy * inside * a)[..., None]
        out = out + total.view(b, h, q, p, d).sum(3)
        start += hh * ww
    return out.permute(0, 2, 1, 3).reshape(b, q, h * d)


def _locations64(ref, off, shapes, points):
    """Sampling locations from reference points and offsets: 32-bit values, 64-bit derivatives."""
    def form(r, o):
        if r.shape[-1] == 2:
            wh = torch.tensor([[w, h] for h, w in shapes], dtype=o.dtype, device=o.device)
            return r[:, :, None, :, None, :] + o / wh[None, None, None, :, None, :]
        return r[:, :, None, :, None, :2] + o / points * r[:, :, None, :, None, 2:] * 0.5
    wide = form(ref, off)
    return form(ref.detach().float(), off.detach().float()).double() + (wide - wide.detach())


def _bilinear64(plane, at, size):
    """Border sampling of plane [N, HW] at points [N, P, 2] of the unit square."""
    h, w = size
    g = 2 * at - 1  # 32 bits
    x, y = ((g[..., 0] + 1) * w - 1) / 2, ((g[..., 1] + 1) * h - 1) / 2
    x0, y0 = x.floor(), y.floor()
    fx, fy = (x - x0).double(), (y - y0).double()
    total = 0
    for dy, wy in ((0, 1 - fy), (1, fy)):
        for dx, wx in ((0, 1 - fx), (1, fx)):
            row = (y0 + dy).long().clamp(0, h - 1) * w + (x0 + dx).long().clamp(0, w - 1)
            total = total + torch.gather(plane, 1, row) * wx * wy
    return total


def exact(case, seed):
    state = prepare(case, seed)
    op = case["op"]
    if op == "module":
        m = state["module"].double()
        b, q, _ = state["query"].shape
        h, levels, p = m.n_heads, m.n_levels, m.n_points
        with torch.no_grad():
            query = state["query"].double()
            value = F.linear(state["memory"].double(), m.value_proj.weight, m.value_proj.bias).masked_fill(state["mask"][..., None], 0)
            value = value.view(b, -1, h, m.d_model // h).permute(0, 2, 1, 3).reshape(b * h, -1, m.d_model // h)
            off = F.linear(query, m.sampling_offsets.weight, m.sampling_offsets.bias).view(b, q, h, levels, p, 2)
            attn = torch.softmax(F.linear(query, m.attention_weights.weight, m.attention_weights.bias).view(b, q, h, -1), -1)
            out = _sample64(value, state["shapes"], _locations64(state["ref"].double(), off, state["shapes"], p), attn)
            return F.linear(out, m.output_proj.weight, m.output_proj.bias)
    if op == "points":
        n, size = case["masks"], (case["height"], case["width"])
        plane = state["logits"].detach().double().view(n, -1).requires_grad_(True)
        chosen = _bilinear64(plane, state["chosen"], size)
        (grad,) = torch.autograd.grad(chosen, plane, state["grad"].double().view(n, -1))
        with torch.no_grad():
            candidates = _bilinear64(plane, state["candidates"], size)
            g = 2 * state["chosen"] - 1
            x = (((g[..., 0] + 1) * size[1] - 1) / 2).round().long().clamp(0, size[1] - 1)
            y = (((g[..., 1] + 1) * size[0] - 1) / 2).round().long().clamp(0, size[0] - 1)
            labels = torch.gather(state["labels"].double().view(n, -1), 1, y * size[1] + x)
        return {"candidates": candidates[:, None], "labels": labels[:, None], "chosen": chosen.detach()[:, None],
                "grad": grad.view(n, 1, *size)}
    train = "grad" in state
    inputs = [t.detach().double().requires_grad_(train) for t in state["inputs"]]
    if op == "core":
        value, loc, attn = inputs
        out = _sample64(value, state["shapes"], loc, attn)
    elif op == "fused":
        value, ref, off, logits = inputs
        out = _sample64(value, state["shapes"], _locations64(ref, off, state["shapes"], case["points"]), torch.softmax(logits, -1))
    elif op == "value_proj":
        x, weight, bias = inputs
        # the layer casts its weight to the input's type
        used = weight + (weight.detach().to(DTYPES[case["dtype"]]).double() - weight.detach())
        out = F.linear(x, used, bias)
        if state["mask"] is not None:
            out = out.masked_fill(state["mask"][..., None], 0)
        out = out.view(*x.shape[:2], case["heads"], case["head_dim"]).permute(0, 2, 1, 3).reshape(-1, x.shape[1], case["head_dim"])
    else:
        b, g, n, h, d = (case[k] for k in ("batch", "groups", "length", "heads", "head_dim"))
        q, k, v = (t.reshape(b, g, n, h, d).transpose(2, 3).reshape(-1, n, d) for t in inputs)
        parts = []
        for z in range(0, q.shape[0], 256):  # a share of the slices at a time bounds the memory
            w = torch.softmax(torch.bmm(q[z:z + 256], k[z:z + 256].transpose(1, 2).contiguous()) * d ** -0.5, -1)
            parts.append(torch.bmm(w, v[z:z + 256].contiguous()))
        out = torch.cat(parts).view(b, g, h, n, d).transpose(2, 3).reshape(b, g * n, h * d)
    if not train:
        return out.detach()
    return (out.detach(), *torch.autograd.grad(out, inputs, state["grad"].double()))
