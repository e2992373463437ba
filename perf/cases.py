"""What this framework is timed on: its layers, called as a model calls them.

A case is a dict of plain values; its "kind" names the part of a sparse
attention layer that one pass runs, through the public entry points of
sparse.ops, sparse.builders and lsrm_hip:

  pool    key (and value) block compression
  select  per-query-block top-k selection
  layer   compression + selection + selected attention, inference
  train   selection + selected attention, forward and backward
  aware   3D-aware per-token rows (builder) + selected attention, forward and
          (train) backward
  learned compressed attention + learned top-k + selected attention, inference
  score   learned top-k alone
  gate    gated merge of the branch outputs, forward and backward
  window  block-diagonal (window) attention, forward and backward

The selection of every layer is a new tensor in each pass, as in a model, so
the plan of the attention kernels is part of the pass.  Sizes are those of
lsrm_hip.workloads (four token counts from 4096 to 524288, LSRM's decoder
heads among them) and of the tests; inputs have their distributions.
"""

import math
import os
import sys
from types import SimpleNamespace

import numpy as np
import torch

PACKAGE = os.path.abspath("large-sparse-reconstruction-model_amd")
if PACKAGE not in sys.path:
    sys.path.insert(1, PACKAGE)

import lsrm_hip  # noqa: E402
import sparse.builders as builders  # noqa: E402
import sparse.ops as ops  # noqa: E402

DEVICE = "cuda"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}

# Of one pass of the largest listed cases; drawn cases stay below both.
MOST_FLOPS = 7.5e12
MOST_ROWS = 524288 * 4 * 32  # selection entries (kv heads x tokens x topk)


def _attention(name, kind, n, hq, hkv, d, topk, blocks, lo, hi, dtype="bf16", batch=1, images=0,
               lowrank=0, train=False):
    return {"name": name, "kind": kind, "n": n, "hq": hq, "hkv": hkv, "d": d, "topk": topk,
            "blocks": blocks, "lo": lo, "hi": hi, "dtype": dtype, "batch": batch,
            "images": images, "lowrank": lowrank, "train": train}


def listed():
    return [
        # one small tensor's block means: launch latency decides
        {"name": "pool_small", "kind": "pool", "n": 4099, "c": 256, "pair": False, "dtype": "bf16",
         "out": "bf16", "blocks": "uniform", "lo": 16, "hi": 128},
        # keys and values of a full decoder layer (hidden 1536), one launch
        # pair; the keys' means in fp32 for the selection
        {"name": "pool_kv_full", "kind": "pool", "n": 131072, "c": 1536, "pair": True,
         "dtype": "bf16", "out": "fp32", "blocks": "scene", "lo": 32, "hi": 512},
        # selection over thousands of heavy-tailed blocks with near ties
        _attention("select_stress", "select", 524288, 4, 4, 64, 32, "lognormal", 8, 1024,
                   lowrank=4),
        # the smallest layer: host work, launches and the plan decide
        _attention("layer_small", "layer", 4096, 4, 4, 64, 8, "uniform", 16, 128),
        # the full decoder layer: 8 image blocks, always selected, and
        # 122880 voxel tokens
        _attention("layer_full", "layer", 131072, 24, 24, 64, 16, "scene", 32, 512, images=8),
        # a training step's attention at mid scale
        _attention("train_mid", "train", 32768, 16, 16, 64, 16, "uniform", 32, 256),
        # one GPU's head shard of the sequence-parallel layout, training
        _attention("train_stress", "train", 524288, 4, 4, 64, 32, "lognormal", 8, 1024,
                   lowrank=4),
        # LSRM's decoder heads over 3D-aware per-token rows of a 64^3 volume
        # in 8^3 blocks, training
        _attention("aware_train", "aware", 122880, 32, 2, 32, 16, "grid", 64, 8, train=True),
        # learned per-token selection at the full layer's heads, inference
        _attention("learned_full", "learned", 131072, 24, 24, 64, 16, "scene", 32, 512),
        # learned top-k alone at LSRM's decoder heads, odd token count
        _attention("score_decoder", "score", 100003, 32, 2, 32, 16, "uniform", 64, 512),
        # three gated branches of a full layer, training
        {"name": "gate_full", "kind": "gate", "n": 131072, "hidden": 1536, "branches": 3,
         "dtype": "bf16"},
        # window branch in fp16 at head dim 128, odd token count, training
        _attention("window_fp16", "window", 30011, 8, 8, 128, 1, "uniform", 64, 512,
                   dtype="fp16"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["pool", "select", "layer", "layer", "train", "train", "aware", "learned",
                       "score", "gate", "window"])
    dtype = rng.choice(["bf16", "bf16", "fp16"])
    if kind == "pool":
        dtype = rng.choice(["bf16", "bf16", "fp16", "fp32"])
        c = rng.choice([192, 256, 512, 768, 1024, 1536])
        n = _log_int(rng, 700, 131072)
        return {"kind": kind, "n": n, "c": c, "pair": rng.random() < 0.5, "dtype": dtype,
                "out": rng.choice([dtype, "fp32"]), "blocks": rng.choice(["uniform", "lognormal"]),
                "lo": 16, "hi": rng.choice([128, 256, 512])}
    if kind == "gate":
        return {"kind": kind, "n": _log_int(rng, 500, 100000),
                "hidden": rng.choice([256, 768, 1000, 1024, 1536]),
                "branches": rng.choice([2, 3]), "dtype": dtype}
    while True:
        if kind == "aware":
            res = rng.choice([32, 64])
            hq, hkv, d = rng.choice([(32, 2, 32), (16, 2, 64), (8, 8, 64)])
            case = _attention("", kind, int(res ** 3 * rng.uniform(0.03, 0.45)), hq, hkv, d,
                              rng.choice([8, 16, 32]), "grid", res, 8, dtype,
                              train=rng.random() < 0.5)
        else:
            hq, hkv, d = rng.choice([(4, 4, 64), (16, 16, 64), (24, 24, 64), (32, 2, 32),
                                     (8, 2, 64), (8, 8, 128)])
            blocks = rng.choice(["uniform", "uniform", "lognormal"])
            lo, hi = (8, 1024) if blocks == "lognormal" else rng.choice(
                [(16, 128), (32, 256), (32, 512)])
            topk = 1 if kind == "window" else rng.choice([4, 8, 12, 16, 32])
            case = _attention("", kind, _log_int(rng, 600, 524288), hq, hkv, d, topk, blocks, lo,
                              hi, dtype, batch=rng.choice([1, 1, 2]), train=kind == "train")
            if kind == "layer" and case["n"] >= 8192 and topk >= 8:
                case["images"] = rng.choice([0, 4])  # blocks that are always selected
        del case["name"]
        if kind in ("select", "score") and \
                min(len(p) for p in _partition(case, 0)) < 2 * case["topk"]:
            continue  # nothing to choose
        w = work(case)
        if w["flops"] <= MOST_FLOPS and case["n"] * hkv * case["topk"] <= MOST_ROWS and \
                case["n"] * hq * d <= 131072 * 1536:
            return case


# ------------------------------------------------------------------ inputs --

def _sizes(blocks, n, lo, hi, rng):
    """Contiguous block sizes covering n tokens; a last block shorter than lo
    joins the one before it."""
    if blocks == "lognormal":
        s = np.clip(np.round(rng.lognormal(math.log(64.0), 1.0, n // lo + 1)), lo, hi)
    else:
        s = rng.integers(lo, hi + 1, n // lo + 1)
    s = s.astype(np.int64)
    ends = np.cumsum(s)
    count = int(np.searchsorted(ends, n)) + 1
    s = s[:count]
    s[-1] -= ends[count - 1] - n
    if count > 1 and s[-1] < lo:
        s[-2] += s[-1]
        s = s[:-1]
    return s


def _partition(case, seed):
    """Block sizes of every batch element: the case's own sizes (as many
    blocks for every seed, so that outputs keep their shapes) in the seed's
    order."""
    sizes, order = np.random.default_rng(case["n"]), np.random.default_rng(seed)
    n, lo, hi = case["n"], case["lo"], case["hi"]
    if case["blocks"] == "scene":  # 8 image blocks, then voxel blocks
        image = n // 128
        voxel = order.permutation(_sizes("uniform", n - 8 * image, lo, hi, sizes))
        return [np.concatenate([np.full(8, image), voxel])]
    batch = case.get("batch", 1)
    lens = [n // batch + (n % batch if e == 0 else 0) for e in range(batch)]
    return [order.permutation(_sizes(case["blocks"], m, lo, hi, sizes)) for m in lens]


def _offsets(counts):
    return torch.tensor(np.concatenate([[0], np.cumsum(counts)]), dtype=torch.int32,
                        device=DEVICE)


def _meta(case, seed):
    parts = _partition(case, seed)
    return SimpleNamespace(cu=_offsets(np.concatenate(parts)),
                           cu_sb=_offsets([len(p) for p in parts]),
                           cu_q=_offsets([int(p.sum()) for p in parts]))


def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _qkv(case, gen, dtype):
    n, hq, hkv, d = case["n"], case["hq"], case["hkv"], case["d"]

    def randn(*shape):
        return torch.randn(shape, generator=gen, device=DEVICE)

    if case["lowrank"]:  # a tenth of the variance shared: near-tied block scores
        r = case["lowrank"]
        u = randn(n, r)
        mix = [(u[:, :, None] * randn(1, r, h * d)).sum(1).view(n, h, d) / math.sqrt(r)
               for h in (hq, hkv)]
        q, k = (math.sqrt(0.9) * randn(n, h, d) + math.sqrt(0.1) * m
                for h, m in zip((hq, hkv), mix))
        return q.to(dtype), k.to(dtype), randn(n, hkv, d).to(dtype)
    return tuple((0.5 * randn(n, h, d)).to(dtype) for h in (hq, hkv, hkv))


def _mean64(x, cu):
    """Block means of [N, C] in 64 bits."""
    lens = (cu[1:] - cu[:-1]).long()
    ids = torch.repeat_interleave(torch.arange(lens.numel(), device=x.device), lens)
    out = torch.zeros(lens.numel(), x.shape[1], dtype=torch.float64, device=x.device)
    for c in range(0, x.shape[1], 256):
        out[:, c:c + 256].index_add_(0, ids, x[:, c:c + 256].double())
    return out / lens[:, None]


def _volume(case, gen):
    """Occupied cells of a res^3 volume in block order -> coords [N, 4] int32
    (batch, c1, c2, c3)."""
    res, bs = case["lo"], case["hi"]
    cells = torch.randperm(res ** 3, generator=gen, device=DEVICE)[:case["n"]]
    c = torch.stack([cells // (res * res), (cells // res) % res, cells % res], 1)
    per = res // bs
    block = ((c[:, 0] // bs) * per + c[:, 1] // bs) * per + c[:, 2] // bs
    inside = ((c[:, 0] % bs) * bs + c[:, 1] % bs) * bs + c[:, 2] % bs
    c = c[torch.argsort(block * bs ** 3 + inside)]
    return torch.cat([torch.zeros_like(c[:, :1]), c], 1).to(torch.int32).contiguous()


def prepare(case, seed):
    gen = _generator(seed)
    kind, dtype = case["kind"], DTYPES[case["dtype"]]
    s = SimpleNamespace(case=case, kind=kind)
    if kind == "gate":
        n, hidden, m = case["n"], case["hidden"], case["branches"]
        s.gate = torch.sigmoid(torch.randn(n, m * hidden, generator=gen, device=DEVICE)).to(dtype)
        s.branches = [torch.randn(n, hidden, generator=gen, device=DEVICE).to(dtype)
                      for _ in range(m)]
        s.dout = torch.randn(n, hidden, generator=gen, device=DEVICE).to(dtype)
        for t in [s.gate] + s.branches:
            t.requires_grad_()
        return s
    if kind == "aware":
        s.coords = _volume(case, gen)
        s.args = SimpleNamespace(block_size=case["hi"], volume_res=case["lo"], bbox_radius=1.0,
                                 topk_volume=case["topk"], use_3d_aware_attn=True)
        s.cu_q = torch.tensor([0, case["n"]], dtype=torch.int32, device=DEVICE)
    else:
        m = _meta(case, seed)
        s.cu, s.cu_sb, s.cu_q = m.cu, m.cu_sb, m.cu_q
    if kind == "pool":
        s.x = [(0.5 * torch.randn(case["n"], case["c"], generator=gen, device=DEVICE)).to(dtype)
               for _ in range(2 if case["pair"] else 1)]
        s.out = DTYPES[case["out"]]
        return s
    s.q, s.k, s.v = _qkv(case, gen, dtype)
    s.forced = list(range(case["images"]))
    s.forced_ids = torch.tensor(s.forced, dtype=torch.int32, device=DEVICE)
    if kind in ("learned", "score"):  # an earlier module has compressed keys and values
        n, hkv, d = s.k.shape
        s.ck, s.cv = (_mean64(t.view(n, -1), s.cu).to(dtype).view(-1, hkv, d)
                      for t in (s.k, s.v))
    if kind == "score":  # natural-log lse of the compressed attention
        s.lse = _compressed64(s, out=False)[1].float()
    if kind == "window" or case["train"]:
        s.do = torch.randn(s.q.shape, generator=gen, device=DEVICE).to(dtype)
    if kind == "window" or case["train"] or kind == "train":
        for t in (s.q, s.k, s.v):
            t.requires_grad_()
        if not hasattr(s, "do"):
            s.do = torch.randn(s.q.shape, generator=gen, device=DEVICE).to(dtype)
    return s


# -------------------------------------------------------------------- passes --

def run(s):
    kind = s.kind
    if kind == "pool":
        if len(s.x) == 2:
            return lsrm_hip.block_mean_pool2(s.x[0], s.x[1], s.cu, s.out, None)
        return ops.block_mean_pool(s.x[0], s.cu, s.out)
    if kind == "gate":
        out = ops.gate_merge(s.gate, *s.branches)
        return (out.detach(),) + torch.autograd.grad(out, [s.gate] + s.branches, s.dout)
    if kind == "score":
        return ops.get_block_score(s.q, s.ck, s.lse, s.case["topk"], s.cu_q, s.cu_sb, None, None)
    if kind == "window":
        out = ops.sparse_window_attention(s.q, s.k, s.v, s.cu)
        return (out.detach(),) + torch.autograd.grad(out, [s.q, s.k, s.v], s.do)
    if kind == "learned":
        with torch.no_grad():
            cmp_out, lse = ops.compressed_attention(s.q, s.ck, s.cv, s.cu_q, s.cu_sb)
            rows = ops.get_block_score(s.q, s.ck, lse, s.case["topk"], s.cu_q, s.cu_sb, None,
                                       None)
            return cmp_out, rows, _attend(s, rows)
    if kind == "layer":
        n, hkv, d = s.k.shape
        with torch.no_grad():
            ck, cv = lsrm_hip.block_mean_pool2(s.k.view(n, -1), s.v.view(n, -1), s.cu,
                                               torch.float32, None)
            rows, _ = lsrm_hip.select_blocks(s.q, s.k, s.cu_sb, s.cu, s.case["topk"],
                                             s.forced_ids, True, pooled_k=ck)
            return ck, cv, rows, _attend(s, rows)
    if kind == "aware":
        made = builders.build_volume_to_volume_attn(s.coords, s.args, s.case["hkv"])
        s.cu, s.cu_sb, rows = (made["cu_block_include_tokens"], made["cu_seqblocks"],
                               made["block_topk"])
    else:
        with torch.no_grad():
            rows = ops.select_blocks(s.q, s.k, s.cu_sb, s.cu, s.case["topk"], s.forced, True)
        if kind == "select":
            return rows
    if not s.q.requires_grad:
        return rows, _attend(s, rows)
    out = _attend(s, rows)
    return (rows, out.detach()) + torch.autograd.grad(out, [s.q, s.k, s.v], s.do)


def _attend(s, rows):
    return ops.spatial_selection_attention(s.q, s.k, s.v, rows, s.cu_sb, s.cu, s.cu_q, s.cu_q,
                                           None, None)


# ---------------------------------------------------------------------- work --

def _attended(case):
    """Keys that a query attends on average: blocks are chosen by the product
    of means of independent values, so a block's score spreads as
    1 / sqrt(its size) and small blocks are chosen more often."""
    if case["blocks"] == "grid":
        blocks = (case["lo"] // case["hi"]) ** 3
        return min(case["topk"], blocks) * case["n"] / blocks
    rng = np.random.default_rng(0)
    total = weight = 0.0
    for sizes in _partition(case, 0):
        nb = len(sizes)
        own = rng.integers(0, nb, min(nb, 256))
        if case["kind"] == "window":
            total += float((sizes * sizes).sum())
            weight += float(sizes.sum())
            continue
        z = rng.standard_normal((len(own), nb)) / np.sqrt(sizes)
        if case["kind"] in ("layer", "train"):
            z[np.arange(len(own)), own] = np.inf
        z[:, :case["images"]] = np.inf
        top = np.argsort(-z, axis=1)[:, :case["topk"]]
        w = sizes[own] * (sizes.sum() / sizes[own].sum())
        total += float((sizes[top].sum(1) * w).sum())
        weight += float(w.sum())
    return total / weight


def work(case):
    """Each input read once and each output written once; products of the
    attention forward count 4, of its backward 10 operations per attended
    (query head, key) pair and channel."""
    kind, n = case["kind"], case["n"]
    size = {"bf16": 2, "fp16": 2, "fp32": 4}[case["dtype"]]
    if kind == "gate":
        m, cells = case["branches"], n * case["hidden"]
        # forward reads gate and branches; backward reads dout, writes as many
        return {"bytes": (2 * m + 1 + 1 + 2 * m) * cells * size, "flops": 5 * m * cells}
    if kind == "pool":
        out = {"bf16": 2, "fp16": 2, "fp32": 4}[case["out"]]
        nb, c = len(np.concatenate(_partition(case, 0))), case["c"]
        means = nb * c * (out + (size if case["pair"] else 0))
        tensors = 2 if case["pair"] else 1
        return {"bytes": tensors * n * c * size + means, "flops": tensors * n * c}
    hq, hkv, d, topk = case["hq"], case["hkv"], case["d"], case["topk"]
    q, k, rows = n * hq * d * size, n * hkv * d * size, 4 * hkv * n * topk
    nb = (case["lo"] // case["hi"]) ** 3 if kind == "aware" else \
        len(np.concatenate(_partition(case, 0)))
    batch = case["batch"]
    if kind == "select":
        return {"bytes": q + k + rows, "flops": 2 * nb * nb // batch * hkv * d + (hq + hkv) * n * d}
    if kind == "score":
        return {"bytes": q + nb * hkv * d * size + 4 * hq * n + rows,
                "flops": 2 * n * hq * d * nb // batch}
    pairs = n * hq * _attended(case)
    bytes_, flops = 2 * q + 2 * k + (0 if kind == "window" else rows), 4 * pairs * d
    if kind == "layer":
        bytes_ += nb * hkv * d * (4 + size)
    if kind == "learned":
        bytes_ += q + 2 * nb * hkv * d * size
        flops += 4 * n * hq * d * nb // batch
    if kind in ("train", "window") or case["train"]:
        bytes_ += 2 * q + 2 * k  # dout, and the three gradients
        flops += 10 * pairs * d
    return {"bytes": int(bytes_), "flops": int(flops)}


def tolerance(case):
    kind = case["kind"]
    if kind in ("select", "gate"):
        return "exact"  # block ids; products and sums rounded one by one
    if kind == "pool":
        # sums in 32 bits, rounded once to the output's type
        return {"rel": 2e-3 if case["out"] == "bf16" or case["dtype"] == "bf16" and case["pair"]
                else 3e-4 if case["out"] == "fp16" or case["dtype"] == "fp16" and case["pair"]
                else 1e-6}
    if kind == "score":
        return {"differ": 1e-3}  # keys whose 32-bit scores are tied
    rel = 1e-2 if case["dtype"] == "bf16" else 1.2e-3
    if kind == "learned":
        return {"rel": 3 * rel, "max": 0.9, "differ": 1e-3}
    return {"rel": rel, "max": 0.2}


# ------------------------------------------------------- 64-bit counterparts --

def _select64(q, k, cu, cu_sb, topk, forced, force_self):
    """Per-query-block selection -> rows [Hkv, N, topk] int32."""
    n, hq, d = q.shape
    hkv = k.shape[1]
    mq = _mean64(q.reshape(n, -1), cu).view(-1, hkv, hq // hkv, d).sum(2)
    mk = _mean64(k.reshape(n, -1), cu).view(-1, hkv, d)
    nb = mq.shape[0]
    compact = torch.full((hkv, nb, topk), -1, dtype=torch.int32, device=q.device)
    for e in range(cu_sb.numel() - 1):
        b0, b1 = int(cu_sb[e]), int(cu_sb[e + 1])
        for h in range(hkv):
            score = mq[b0:b1, h].contiguous() @ mk[b0:b1, h].t().contiguous()
            score[:, forced] = math.inf
            if force_self:
                score.fill_diagonal_(math.inf)
            m = min(topk, b1 - b0)
            compact[h, b0:b1, :m] = score.topk(m, 1).indices.sort(1).values.int()
    return compact.repeat_interleave((cu[1:] - cu[:-1]).long(), 1)


def _attend64(q, k, v, rows, cu, cu_sb, cu_q, do=None):
    """Selected attention in 64 bits, block by block over the queries that
    list the block; the logits of these inputs need no maximum taken off."""
    n, hq, d = q.shape
    hkv = k.shape[1]
    g, nb, topk, scale = hq // hkv, cu.numel() - 1, rows.shape[2], 1.0 / math.sqrt(d)
    base = torch.repeat_interleave(cu_sb[:-1].long(), (cu_q[1:] - cu_q[:-1]).long())
    bounds = cu.tolist()
    out, dq = torch.empty(n, hq, d, dtype=torch.float64, device=q.device), None
    if do is not None:
        dq = torch.empty_like(out)
        dk = torch.zeros(k.shape, dtype=torch.float64, device=q.device)
        dv = torch.zeros_like(dk)
    for h in range(hkv):
        ids = torch.where(rows[h] >= 0, rows[h] + base[:, None], nb).reshape(-1)
        token = torch.argsort(ids, stable=True) // topk
        ends = torch.bincount(ids, minlength=nb + 1).cumsum(0).tolist()
        qh = q[:, h * g:(h + 1) * g].double() * scale
        kh, vh = k[:, h].double(), v[:, h].double()
        o = torch.zeros(n, g, d, dtype=torch.float64, device=q.device)
        total = torch.zeros(n, g, 1, dtype=torch.float64, device=q.device)

        def pieces():
            for b in range(nb):
                k0, k1 = bounds[b], bounds[b + 1]
                step = max(1, (1 << 26) // (g * max(1, k1 - k0)))
                for t in range(ends[b - 1] if b else 0, ends[b], step):
                    yield k0, k1, token[t:min(t + step, ends[b])]

        for k0, k1, at in pieces():
            p = (qh[at].view(-1, d) @ kh[k0:k1].t()).exp_()
            o[at] += (p @ vh[k0:k1]).view(-1, g, d)
            total[at] += p.sum(1).view(-1, g, 1)
        o /= total
        out[:, h * g:(h + 1) * g] = o
        if do is None:
            continue
        doh = do[:, h * g:(h + 1) * g].double()
        delta = (doh * o).sum(2, keepdim=True)
        dqh = torch.zeros_like(qh)
        for k0, k1, at in pieces():
            qa, da = qh[at].view(-1, d), doh[at].view(-1, d)
            p = (qa @ kh[k0:k1].t()).exp_() / total[at].view(-1, 1)
            dv[k0:k1, h] += p.t() @ da
            ds = p.mul_(da @ vh[k0:k1].t() - delta[at].view(-1, 1))
            dqh[at] += (ds @ kh[k0:k1]).view(-1, g, d) * scale
            dk[k0:k1, h] += ds.t() @ qa
        dq[:, h * g:(h + 1) * g] = dqh
    return (out,) if do is None else (out, dq, dk, dv)


def _compressed64(s, out=True):
    """Attention over the compressed keys of the token's batch element ->
    (out or None, natural-log lse [Hq, N])."""
    n, hq, d = s.q.shape
    g = hq // s.ck.shape[1]
    o = torch.empty(n, hq, d, dtype=torch.float64, device=DEVICE) if out else None
    lse = torch.empty(hq, n, dtype=torch.float64, device=DEVICE)
    tokens, keys = s.cu_q.tolist(), s.cu_sb.tolist()
    for h in range(hq):
        for (t0, t1), (c0, c1) in zip(zip(tokens, tokens[1:]), zip(keys, keys[1:])):
            for t in range(t0, t1, 65536):
                e = min(t + 65536, t1)
                x = s.q[t:e, h].double() @ s.ck[c0:c1, h // g].double().t() / math.sqrt(d)
                lse[h, t:e] = x.logsumexp(1)
                if out:
                    o[t:e, h] = x.softmax(1) @ s.cv[c0:c1, h // g].double()
    return o, lse


def _score64(s, lse):
    """The topk best compressed keys per token and kv head, ascending."""
    n, hq, d = s.q.shape
    hkv, topk = s.ck.shape[1], s.case["topk"]
    g = hq // hkv
    rows = torch.full((hkv, n, topk), -1, dtype=torch.int32, device=DEVICE)
    tokens, keys = s.cu_q.tolist(), s.cu_sb.tolist()
    for h in range(hkv):
        for (t0, t1), (c0, c1) in zip(zip(tokens, tokens[1:]), zip(keys, keys[1:])):
            m = min(topk, c1 - c0)
            for t in range(t0, t1, 16384):
                e = min(t + 16384, t1)
                x = s.q[t:e, h * g:(h + 1) * g].double().reshape(-1, d) @ \
                    s.ck[c0:c1, h].double().t() / math.sqrt(d)
                p = (x.view(e - t, g, -1) - lse[h * g:(h + 1) * g, t:e].t()[:, :, None].double())
                rows[h, t:e, :m] = p.exp_().sum(1).topk(m, 1).indices.sort(1).values.int()
    return rows


def _nearest64(s):
    """3D-aware rows: the blocks whose centroids are nearest to each token."""
    case, c = s.case, s.coords[:, 1:].long()
    res, bs = case["lo"], case["hi"]
    per = res // bs
    block = ((c[:, 0] // bs) * per + c[:, 1] // bs) * per + c[:, 2] // bs
    counts = torch.unique_consecutive(block, return_counts=True)[1]
    cu = torch.cat([counts.new_zeros(1), counts.cumsum(0)])
    den = torch.tensor(res - 1, dtype=torch.float32, device=DEVICE)
    points = (2.0 * (c.flip(1).float() / den - 0.5) * np.float32(1.05).item())
    centres = _mean64(points, cu).float().double()
    m = min(case["topk"], counts.numel())
    rows = torch.full((case["n"], case["topk"]), -1, dtype=torch.int32, device=DEVICE)
    for t in range(0, case["n"], 16384):
        x = points[t:t + 16384].double()
        dist = sum((x[:, i:i + 1] - centres[None, :, i]) ** 2 for i in range(3))
        rows[t:t + 16384, :m] = dist.topk(m, 1, largest=False).indices.sort(1).values.int()
    cu_sb = torch.tensor([0, counts.numel()], dtype=torch.int32, device=DEVICE)
    return rows.expand(case["hkv"], -1, -1).contiguous(), cu.int(), cu_sb


def exact(case, seed):
    s = prepare(case, seed)
    kind = s.kind
    with torch.no_grad():
        if kind == "pool":
            means = [_mean64(x, s.cu) for x in s.x]
            return tuple(means) if len(means) == 2 else means[0]
        if kind == "gate":
            parts = [g.double() for g in s.gate.chunk(len(s.branches), 1)]
            dout = s.dout.double()
            out = sum(g * b.double() for g, b in zip(parts, s.branches))
            return (out, torch.cat([dout * b.double() for b in s.branches], 1)) + \
                tuple(dout * g for g in parts)
        if kind == "score":
            return _score64(s, s.lse)
        if kind == "learned":
            out, lse = _compressed64(s)
            rows = _score64(s, lse)
            return out, rows, _attend64(s.q, s.k, s.v, rows, s.cu, s.cu_sb, s.cu_q)[0]
        if kind == "aware":
            rows, cu, cu_sb = _nearest64(s)
        else:
            cu, cu_sb = s.cu, s.cu_sb
            if kind == "window":
                lens = (cu[1:] - cu[:-1]).long()
                first = torch.repeat_interleave(cu_sb[:-1].long(),
                                                (cu_sb[1:] - cu_sb[:-1]).long())
                local = torch.arange(lens.numel(), device=DEVICE) - first
                rows = local.int().repeat_interleave(lens).expand(s.k.shape[1], -1)[:, :, None]
            else:
                rows = _select64(s.q, s.k, cu, cu_sb, case["topk"], s.forced, True)
        if kind == "select":
            return rows
        do = getattr(s, "do", None)
        got = _attend64(s.q, s.k, s.v, rows, cu, cu_sb, s.cu_q, do)
        if kind == "window":
            return got
        if kind == "layer":
            n = s.k.shape[0]
            return (_mean64(s.k.view(n, -1), cu), _mean64(s.v.view(n, -1), cu), rows, got[0])
        return (rows,) + got
