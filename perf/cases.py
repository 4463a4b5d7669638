"""What the speed of this framework is measured on: the sparse global-attention layer.

A VGGT / Pi3 global-attention layer sees ``views`` images of ``tokens`` tokens each (5 special
tokens and a grid of up to 37 x 37 patches of 14 pixels: 1374 tokens for a 518 x 518 image,
fewer for the other aspect ratios), 16 heads of 64, a lightning indexer of 4 x 64 and top-k
1024. A program calls the layer as a whole (``SparseGlobalAttention``), or the drop-ins it is
made of: the indexer's top-k, the sparse attention over the selected keys, the indexer's KL
loss, and their backward. Kinds of a case:

* ``infer``: the inference indexer, then the inference attention over its selection.
* ``attend``: the attention alone over a selection that the program holds, as a layer that
  reuses another layer's top-k does.
* ``layer``: ``SparseGlobalAttention.forward`` (projection, glue, indexer, attention, output
  projection).
* ``train``: one training step of indexer, attention with its attention mass, the indexer's KL
  loss and the backward of all of them. ``mass`` "detached" gives the loss the mass detached
  (the presets' choice); "joined" lets its gradient reach q, k and v as well.
* ``layer_train``: the same step through ``SparseGlobalAttention.forward_train``.

The order of the selected keys inside a row is unspecified, so a case returns what is computed
from the selection (attention outputs, losses, gradients) and not the index lists.
"""
import torch
import torch.nn.functional as F

from geoweave_amd import dsa_layer
from geoweave_amd.custom_flash_attn.sparse_index_flash_attn import (
    sparse_index_flash_attn_func,
    sparse_index_flash_attn_inference_bhtd_func,
    sparse_index_flash_attn_inference_func,
)
from geoweave_amd.custom_indexer import sparse_indexer_kl_loss, sparse_topk_indexer_func
from geoweave_amd.custom_indexer.indexer_kl_fused import sparse_attention_kl_loss
from geoweave_amd.custom_indexer.sparse_topk_indexer import sparse_topk_indexer_inference_func

DIM, HEADS, IDX_HEADS, HEAD_DIM = 1024, 16, 4, 64
SCALE = 0.125
EPS = 1e-6
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}


def _case(kind, views, grid_h=37, grid_w=37, batch=1, topk=1024, dtype="bf16", **more):
    return dict(kind=kind, views=views, grid_h=grid_h, grid_w=grid_w, batch=batch, topk=topk, dtype=dtype, **more)


def _tokens(case):
    return case["views"] * (5 + case["grid_h"] * case["grid_w"])


def listed():
    return [
        # An image pair through one layer: the smallest call, where launches and latency count.
        dict(_case("layer", 2, score_dtype="bf16"), name="layer, 2 views"),
        # Four views, the smallest of the repository's own configurations.
        dict(_case("infer", 4), name="infer, 4 views"),
        # A short clip of 518 x 392 frames in fp16: ragged token counts.
        dict(_case("infer", 12, 37, 28, dtype="fp16"), name="infer, 12 views of 37x28, fp16"),
        # The presets' layer: bf16 activations, fp16 scores, 16 views.
        dict(_case("layer", 16, score_dtype="fp16"), name="layer, 16 views, fp16 scores"),
        # A layer that reuses the selection of the layer before it, [B, H, T, D] layout.
        dict(_case("attend", 20, 37, 36, layout="bhtd"), name="attend, 20 views of 37x36"),
        # The headline layer: 32 views.
        dict(_case("infer", 32), name="infer, 32 views"),
        # Long context: 64 views.
        dict(_case("infer", 64), name="infer, 64 views"),
        # Training on few views, as at the start of a multi-view curriculum.
        dict(_case("train", 4, mass="detached"), name="train, 4 views"),
        # The training configuration: two scenes of 24 views.
        dict(_case("train", 24, batch=2, mass="detached"), name="train, 2 x 24 views"),
        # Training with the indexer's loss reaching the attention as well.
        dict(_case("train", 8, mass="joined"), name="train, 8 views, joined loss"),
        # The whole layer trained on 12 views of 518 x 294 frames.
        dict(_case("layer_train", 12, 21, 37, score_dtype="bf16"), name="layer training, 12 views of 21x37"),
    ]


def draw(rng):
    kind = rng.choice(["infer", "infer", "attend", "layer", "train", "train", "layer_train"])
    train = "train" in kind
    # One side of an image is 37 patches, the other 12 to 37.
    side = rng.randint(12, 37)
    grid = (37, side) if rng.random() < 0.5 else (side, 37)
    top = 65.0 if not train else 33.0
    views = int(2.0 * (top / 2.0) ** rng.random())
    # The product of batch and square of the tokens stays within the largest listed case of its kind.
    batch = 2 if views <= (24 if train else 40) and rng.random() < 0.3 else 1
    topk = rng.choice([512, 1024, 1024, 1024] if train else [512, 1024, 1024, 1024, 2048])
    more = {}
    if kind == "attend":
        more["layout"] = rng.choice(["bthd", "bhtd"])
    if kind in ("layer", "layer_train"):
        more["score_dtype"] = rng.choice(["bf16", "fp16"])
    dtype = "bf16" if kind in ("layer", "layer_train") else rng.choice(["bf16", "bf16", "fp16"])
    if kind == "train":
        more["mass"] = "joined" if views <= 8 and rng.random() < 0.3 else "detached"
    return _case(kind, views, grid[0], grid[1], batch, topk, dtype, **more)


# ---------------------------------------------------------------------------------------------
# Inputs


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda")


def _indexer_inputs(g, batch, n, dtype):
    """Projections of unit-variance tokens: q, k about N(0, 1), gates 1 with a spread."""
    qs, ks, ws = [], [], []
    for _ in range(batch):
        x = _randn(g, n, DIM)
        qs.append((x @ (_randn(g, DIM, IDX_HEADS * HEAD_DIM) / DIM ** 0.5)).view(n, IDX_HEADS, HEAD_DIM))
        ks.append((x @ (_randn(g, DIM, IDX_HEADS * HEAD_DIM) / DIM ** 0.5)).view(n, IDX_HEADS, HEAD_DIM))
        ws.append(1.0 + x @ (_randn(g, DIM, IDX_HEADS) * (0.5 / DIM ** 0.5)))
    return [torch.stack(t).to(dtype) for t in (qs, ks, ws)]


def _layer(g, case):
    """A layer with random weights (there are no checkpoints to load): unit-variance
    projections, LayerNorm gains about 1, the indexer's gates about 1."""
    score = None if case["score_dtype"] == "bf16" else "float16"
    layer = dsa_layer.SparseGlobalAttention(DIM, HEADS, indexer_heads=IDX_HEADS, topk=case["topk"], score_dtype=score).cuda()
    with torch.no_grad():
        for name, p in layer.named_parameters():
            if p.dim() == 2:
                p.copy_(_randn(g, *p.shape) * ((0.25 if "w_proj" in name else 1.0) / p.shape[1] ** 0.5))
            elif "norm" in name and name.endswith("weight"):
                p.copy_(1 + 0.1 * _randn(g, *p.shape))
            elif "w_proj" in name:
                p.fill_(1.0)
            else:
                p.copy_(0.02 * _randn(g, *p.shape))
    return layer.to(torch.bfloat16)


def _inputs(case, seed):
    g = _gen(seed)
    b, n, dtype = case["batch"], _tokens(case), DTYPES[case["dtype"]]
    if case["kind"] in ("layer", "layer_train"):
        s = {"layer": _layer(g, case), "x": _randn(g, b, n, DIM).to(dtype)}
        pos = dsa_layer.grid_positions(case["views"], case["grid_h"], case["grid_w"], device="cuda")
        s["pos"] = pos.reshape(1, n, 2).expand(b, -1, -1).contiguous()
        s["rope_len"] = max(case["grid_h"], case["grid_w"]) + 1
        if case["kind"] == "layer_train":
            s["dout"] = _randn(g, b, n, DIM).to(dtype)
        return s
    s = {}
    s["qi"], s["ki"], s["wi"] = _indexer_inputs(g, b, n, dtype)
    shape = (b, HEADS, n, HEAD_DIM) if case.get("layout") == "bhtd" else (b, n, HEADS, HEAD_DIM)
    for name in ("q", "k", "v") + (("do",) if case["kind"] == "train" else ()):
        s[name] = _randn(g, *shape).to(dtype)
    return s


def prepare(case, seed):
    s = _inputs(case, seed)
    s["case"] = case
    if case["kind"] == "attend":
        idx, _ = sparse_topk_indexer_inference_func(s.pop("qi"), s.pop("ki"), s.pop("wi"), None, case["topk"], SCALE)
        s["idx"] = idx
    if case["kind"] == "train":
        for name in ("qi", "ki", "wi", "q", "k", "v"):
            s[name].requires_grad_()
    if case["kind"] == "layer_train":
        s["x"].requires_grad_()
    return s


# ---------------------------------------------------------------------------------------------
# One pass


def run(s):
    case = s["case"]
    kind, topk = case["kind"], case["topk"]
    if kind == "infer":
        idx, _ = sparse_topk_indexer_inference_func(s["qi"], s["ki"], s["wi"], None, topk, SCALE)
        o, _ = sparse_index_flash_attn_inference_func(s["q"], s["k"], s["v"], idx, softmax_scale=SCALE)
        return {"o": o}
    if kind == "attend":
        f = sparse_index_flash_attn_inference_bhtd_func if case["layout"] == "bhtd" else sparse_index_flash_attn_inference_func
        o, _ = f(s["q"], s["k"], s["v"], s["idx"], softmax_scale=SCALE)
        return {"o": o}
    if kind == "layer":
        return {"out": s["layer"](s["x"], s["pos"], rope_len=s["rope_len"])}
    if kind == "train":
        ins = [s[n] for n in ("q", "k", "v", "qi", "ki", "wi")]
        idx, scores = sparse_topk_indexer_func(s["qi"], s["ki"], s["wi"], None, topk, SCALE, 256, 0)
        if case["mass"] == "joined":
            o, _, loss = sparse_attention_kl_loss(s["q"], s["k"], s["v"], idx, scores, EPS, SCALE)
        else:
            o, attn = sparse_index_flash_attn_func(s["q"], s["k"], s["v"], idx, None, False, SCALE)
            p = attn.detach().to(o.dtype)
            p = p / (p.sum(dim=-1, keepdim=True) + EPS)
            loss = sparse_indexer_kl_loss(p, scores, EPS)
        grads = torch.autograd.grad([o, loss], ins, [s["do"], torch.ones_like(loss)])
        return {"o": o.detach(), "loss": loss.detach(), **dict(zip(("dq", "dk", "dv", "dqi", "dki", "dwi"), grads))}
    if kind == "layer_train":
        out, attn, scores, _ = s["layer"].forward_train(s["x"], s["pos"], rope_len=s["rope_len"])
        p = attn.detach().to(out.dtype)
        p = p / (p.sum(dim=-1, keepdim=True) + EPS)
        loss = sparse_indexer_kl_loss(p, scores, EPS)
        names, params = zip(*s["layer"].named_parameters())
        grads = torch.autograd.grad([out, loss], [s["x"], *params], [s["dout"], torch.ones_like(loss)])
        return {"out": out.detach(), "loss": loss.detach(), "grads": dict(zip(("x",) + names, grads))}
    raise ValueError(kind)


# ---------------------------------------------------------------------------------------------
# What a pass cannot do without


def work(case):
    """Inputs read once, outputs written once, and the products over what is needed: the
    indexer scores every (query, key) pair, the attention the selected pairs."""
    b, n = case["batch"], _tokens(case)
    k = min(case["topk"], n)
    rows = b * n * DIM * 2  # one [B, N, 1024] tensor of 16-bit values
    idx_rows = 2 * b * n * (2 * IDX_HEADS * HEAD_DIM + IDX_HEADS)
    score_flops = 2 * b * n * n * IDX_HEADS * HEAD_DIM
    attn_flops = 4 * b * n * k * HEADS * HEAD_DIM
    kind = case["kind"]
    if kind == "infer":
        return {"bytes": 4 * rows + idx_rows, "flops": score_flops + attn_flops}
    if kind == "attend":
        return {"bytes": 4 * rows + 4 * b * n * k, "flops": attn_flops}
    weights = DIM * (4 * DIM + 2 * IDX_HEADS * HEAD_DIM + IDX_HEADS)
    proj_flops = 2 * b * n * weights
    if kind == "layer":
        return {"bytes": 2 * rows + 2 * weights + 8 * b * n, "flops": proj_flops + score_flops + attn_flops}
    # backward: five products over the selected pairs, and two for the indexer's gradients
    step = score_flops + attn_flops + 10 * b * n * k * HEADS * HEAD_DIM + 6 * b * n * k * IDX_HEADS * HEAD_DIM
    if kind == "train":
        return {"bytes": 8 * rows + 2 * idx_rows, "flops": step}
    return {"bytes": 4 * rows + 4 * weights + 8 * b * n, "flops": step + 3 * proj_flops}


def tolerance(case):
    # About four times the 2-norm errors against 64 bits, which are the outputs' own rounding:
    # 1.9e-3 in bf16, 3e-4 to 6e-4 in fp16, 4e-3 behind a layer's projections, 3e-3 for the
    # gradients. A selection that differs where two scores tie within fp32 rounding moves single
    # rows by up to a key's weight, hence "max".
    if case["kind"] in ("layer", "layer_train"):
        return {"rel": 1.6e-2, "max": 0.9}
    if case["kind"] == "train":
        return {"rel": 1.2e-2, "max": 0.9}
    return {"rel": 8e-3 if case["dtype"] == "bf16" else 2e-3, "max": 0.9}


# ---------------------------------------------------------------------------------------------
# The same in 64 bits, from plain torch


def _exact_topk(qi, ki, wi, topk):
    """Selected pairs of one batch element as a [T, S] mask, and their scores (0 elsewhere)."""
    n, s = qi.shape[0], ki.shape[0]
    k = min(topk, s)
    mask = torch.zeros(n, s, dtype=torch.bool, device="cuda")
    for a in range(0, n, 1024):
        score = _exact_scores(qi[a:a + 1024], ki, wi)
        mask[a:a + 1024].scatter_(1, score.topk(k, dim=1, sorted=False).indices, True)
    return mask


def _exact_scores(qi, ki, wi):
    score = 0
    for h in range(qi.shape[1]):
        score = torch.relu(qi[:, h].double() @ ki[:, h].double().t()).mul_(SCALE * wi[:, h].double()[None]).add_(score)
    return score


def _exact_attention(q, k, v, mask, mass=False):
    """q, k, v [N, H, D] of one batch element, in 64 bits."""
    o = torch.empty_like(q)
    for a in range(0, q.shape[0], 1024):
        off = ~mask[a:a + 1024]
        for h in range(q.shape[1]):
            p = torch.softmax((q[a:a + 1024, h] @ k[:, h].t()).mul_(SCALE).masked_fill_(off, float("-inf")), dim=1)
            o[a:a + 1024, h] = p @ v[:, h]
    return o


def _exact_step(q, k, v, qi, ki, wi, do, case, mask, rows):
    """(o, the sum of the loss over this batch element's rows, gradients) in 64 bits."""
    dtype = DTYPES[case["dtype"]]
    joined = case["mass"] == "joined"
    n, heads = q.shape[0], q.shape[1]
    o, loss = torch.empty_like(q), 0.0
    grads = [torch.zeros_like(t) for t in (q, k, v, qi, ki, wi)]
    dq, dk, dv, dqi, dki, dwi = grads
    for a in range(0, n, 512):
        c = slice(a, min(a + 512, n))
        on = mask[c]
        logits = [(q[c, h] @ k[:, h].t()).mul_(SCALE).masked_fill_(~on, float("-inf")) for h in range(heads)]
        mass = 0
        for h in range(heads):
            logits[h] = torch.softmax(logits[h], dim=1)
            mass = mass + logits[h]
            o[c, h] = logits[h] @ v[:, h]
        a_in = mass if joined else mass.to(dtype).double()
        total = a_in.sum(1, keepdim=True) + EPS
        p = a_in / total
        if not joined:  # the loss normalises what it is given once more
            p = p / (p.sum(1, keepdim=True) + EPS)
        z = _exact_scores(qi[c], ki, wi).to(dtype).double().masked_fill_(~on, float("-inf"))
        log_soft = torch.log_softmax(z, dim=1).masked_fill_(~on, 0.0)
        term = torch.where(on, (p + EPS).log() - log_soft, 0.0)
        loss = loss + (p * term).sum()
        dz = torch.where(on, torch.softmax(z, dim=1) - p, 0.0) / rows
        da = 0.0
        if joined:
            dp = torch.where(on, term + p / (p + EPS), 0.0) / rows
            da = (dp - (dp * p).sum(1, keepdim=True)) / total
        for h in range(heads):
            w = logits[h]
            dw_h = (do[c, h] @ v[:, h].t()).add_(da)
            ds = w * (dw_h - (w * dw_h).sum(1, keepdim=True)) * SCALE
            dq[c, h] = ds @ k[:, h]
            dk[:, h] += ds.t() @ q[c, h]
            dv[:, h] += w.t() @ do[c, h]
        for h in range(qi.shape[1]):
            y = qi[c, h] @ ki[:, h].t()
            gate = dz * (y > 0)
            dqi[c, h] = SCALE * (gate * wi[:, h][None]) @ ki[:, h]
            dki[:, h] += SCALE * wi[:, h][:, None] * (gate.t() @ qi[c, h])
            dwi[:, h] += SCALE * (gate * y).sum(0)
    return o, loss, grads


def _exact_rope(t, pos):
    """t [N, H, 64] in 64 bits, rotated by (y, x): dims 0-31 with y, 32-63 with x."""
    freq = 100.0 ** (-torch.arange(0, 32, 2, device="cuda").double() / 32)
    halves = []
    for axis, x in enumerate(t.chunk(2, dim=-1)):
        angle = pos[:, axis].double()[:, None] * freq
        cos, sin = angle.cos()[:, None], angle.sin()[:, None]
        x1, x2 = x.chunk(2, dim=-1)
        halves += [x1 * cos - x2 * sin, x2 * cos + x1 * sin]
    return torch.cat(halves, dim=-1)


def _exact_layer(case, seed):
    """The layer with the 16-bit tensors that it hands from stage to stage, each stage in 64 bits."""
    s = _inputs(case, seed)
    layer, dtype = s["layer"], DTYPES[case["dtype"]]
    cut = lambda t: t.to(dtype).double()  # noqa: E731
    score = (lambda t: t.to(torch.float16).double()) if case["score_dtype"] == "fp16" else (lambda t: t)
    ix = layer.indexer

    def linear(m, x):
        return x @ m.weight.double().t() + m.bias.double()

    def norm(m, t):
        return F.layer_norm(t, (HEAD_DIM,), m.weight.double(), m.bias.double(), m.eps)

    outs = []
    with torch.no_grad():
        for b in range(case["batch"]):
            x, pos = s["x"][b].double(), s["pos"][b]
            q, k, v = cut(linear(layer.qkv, x)).view(-1, 3, HEADS, HEAD_DIM).unbind(1)
            qi = cut(linear(ix.q_proj, x)).view(-1, IDX_HEADS, HEAD_DIM)
            ki = cut(linear(ix.k_proj, x)).view(-1, IDX_HEADS, HEAD_DIM)
            wi = score(cut(linear(ix.w_proj, x)))
            q, k = (score(cut(_exact_rope(norm(m, t), pos))) for m, t in ((layer.q_norm, q), (layer.k_norm, k)))
            qi, ki = score(cut(_exact_rope(qi, pos))), score(cut(_exact_rope(norm(ix.k_norm, ki), pos)))
            o = _exact_attention(q, k, score(v), _exact_topk(qi, ki, wi, case["topk"]))
            outs.append(linear(layer.proj, cut(o).reshape(-1, DIM)))
    return {"out": torch.stack(outs)}


def exact(case, seed):
    kind = case["kind"]
    if kind == "layer_train":
        return None  # gradients through every 16-bit stage have no one value; the other cases hold each of them
    if kind == "layer":
        return _exact_layer(case, seed)
    s = _inputs(case, seed)
    bhtd = case.get("layout") == "bhtd"
    batch, rows = case["batch"], case["batch"] * _tokens(case)
    outs, loss, grads = [], 0.0, []
    for b in range(batch):
        qi, ki, wi = (s[n][b] for n in ("qi", "ki", "wi"))
        q, k, v = ((s[n][b].transpose(0, 1) if bhtd else s[n][b]).double() for n in ("q", "k", "v"))
        mask = _exact_topk(qi, ki, wi, case["topk"])
        if kind == "train":
            o, part, g = _exact_step(q, k, v, qi.double(), ki.double(), wi.double(), s["do"][b].double(), case, mask, rows)
            loss = loss + part / rows
            grads.append(g)
        else:
            o = _exact_attention(q, k, v, mask)
        outs.append(o.transpose(0, 1) if bhtd else o)
        del mask
    out = {"o": torch.stack(outs)}
    if kind == "train":
        out["loss"] = loss
        out.update(zip(("dq", "dk", "dv", "dqi", "dki", "dwi"), (torch.stack(t) for t in zip(*grads))))
    return out
