"""The work that programs have this library do, as timed cases through its public entry points.

Six kinds of call, each over the range that a Gemma 4 31B program meets:

* ``decode``: one new token of each sequence against its cached keys (inference);
* ``extend``: a chunk of new tokens after a cached prefix, global layers (chunked
  prefill, a prompt after a shared prefix, verification of drafted tokens);
* ``layer``: one whole sliding attention layer over a prompt (projections, norms, RoPE,
  attention, output projection), the call that a compiled prefill makes per layer;
* ``kv_prep``: the global layers' K and V from their shared projection, forward and
  backward;
* ``train_fixed``: forward and backward of one short sequence through the fixed adapters;
* ``train_packed``: forward and backward of packed sequences, text or multimodal.

``listed`` gives the cases that are always timed, ``draw`` further ones of the same ranges.
Sequence lengths and vision blocks follow from a case's own ``shape`` number, values from the
seed given to ``prepare``.
"""

import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "gemma4-fa4-kernels_amd"))

import gemma4_fa4_amd as g4  # noqa: E402
from gemma4_fa4_amd import torch_ops  # noqa: E402

WINDOW = 1024  # sliding layers
HIDDEN = 5376
Q_HEADS = 32
KV_HEADS = {"local": 16, "global": 4}
HEAD_DIM = {"local": 256, "global": 512}
ROTARY = 128  # global layers: a quarter of the head dim
EPS = 1e-6
DEVICE = "cuda"


def listed():
    return [
        # One user's chat on a sliding layer: the smallest call, 50 times per generated token.
        {"name": "decode_local_1", "kind": "decode", "layer": "local", "batch": 1, "cache": 1024,
         "shape": 0},
        # The same step on a global layer with an 8K conversation in its StaticCache backing.
        {"name": "decode_global_8k", "kind": "decode", "layer": "global", "batch": 1,
         "cache": 8192, "shape": 0},
        # A serving step: 16 conversations of 4K to 8K tokens, packed.
        {"name": "decode_global_batch16", "kind": "decode", "layer": "global", "batch": 16,
         "cache": 8192, "shape": 1},
        # A 500-token message appended to a 12K conversation (chunked prefill).
        {"name": "extend_500_after_12k", "kind": "extend", "new": 500, "prefix": 12000},
        # One sliding layer of a 1000-token prompt, whole.
        {"name": "layer_local_1000", "kind": "layer", "seqlen": 1000},
        # K and V of the global layers in an 8K training step.
        {"name": "kv_prep_8k", "kind": "kv_prep", "seqlen": 8192, "tables": "fp32"},
        # Fine-tuning on short samples, one at a time: both layer kinds, odd lengths.
        {"name": "train_fixed_local_777", "kind": "train_fixed", "layer": "local", "seqlen": 777,
         "vision": True, "shape": 2},
        {"name": "train_fixed_global_1000", "kind": "train_fixed", "layer": "global",
         "seqlen": 1000, "vision": False, "shape": 0},
        # The headline benchmark: one 8K sequence on a global layer.
        {"name": "train_global_8k", "kind": "train_packed", "layer": "global", "tokens": 8192,
         "segments": 1, "vision": False, "documents": False, "shape": 0},
        # A packed batch of many short samples on a global layer.
        {"name": "train_global_32k_in_32", "kind": "train_packed", "layer": "global",
         "tokens": 32768, "segments": 32, "vision": False, "documents": False, "shape": 3},
        # One multimodal 8K sample on a sliding layer.
        {"name": "train_local_8k_vision", "kind": "train_packed", "layer": "local",
         "tokens": 8192, "segments": 1, "vision": True, "documents": False, "shape": 4},
        # A large packed multimodal batch on a sliding layer, document IDs given.
        {"name": "train_local_128k_vision_documents", "kind": "train_packed", "layer": "local",
         "tokens": 131072, "segments": 8, "vision": True, "documents": True, "shape": 5},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    most = work(listed()[-1])["flops"]
    while True:
        case = _draw(rng)
        if work(case)["flops"] <= 0.8 * most:
            return case


def _draw(rng):
    kind = rng.choice(["decode", "extend", "layer", "kv_prep", "train_fixed", "train_packed"])
    shape = rng.randrange(1 << 30)
    layer = rng.choice(["local", "global"])
    if kind == "decode":
        cache = rng.randint(64, WINDOW) if layer == "local" else _log_uniform(rng, 128, 32768)
        return {"kind": kind, "layer": layer, "batch": _log_uniform(rng, 1, 32), "cache": cache,
                "shape": shape}
    if kind == "extend":
        return {"kind": kind, "new": _log_uniform(rng, 8, 2048),
                "prefix": _log_uniform(rng, 512, 32768)}
    if kind == "layer":
        return {"kind": kind, "seqlen": _log_uniform(rng, 16, 1024)}
    if kind == "kv_prep":
        return {"kind": kind, "seqlen": _log_uniform(rng, 64, 32768),
                "tables": rng.choice(["fp32", "bf16"])}
    if kind == "train_fixed":
        seqlen = rng.randint(64, 1025) if layer == "local" else _log_uniform(rng, 64, 2048)
        return {"kind": kind, "layer": layer, "seqlen": seqlen,
                "vision": layer == "local" and rng.random() < 0.5, "shape": shape}
    tokens = _log_uniform(rng, 2048, 131072 if layer == "local" else 32768)
    vision = layer == "local" and rng.random() < 0.7
    return {"kind": kind, "layer": layer, "tokens": tokens,
            "segments": _log_uniform(rng, 1, min(32, tokens // 256)), "vision": vision,
            "documents": vision and rng.random() < 0.5, "shape": shape}


# ---------------------------------------------------------------------------
# geometry of a case
# ---------------------------------------------------------------------------


def _lengths(case):
    """Key lengths of the sequences."""
    kind = case["kind"]
    if kind in ("layer", "train_fixed"):
        return [case["seqlen"]]
    if kind == "extend":
        return [case["prefix"] + case["new"]]
    rng = np.random.default_rng(case["shape"])
    if kind == "decode":
        top, n = case["cache"], case["batch"]
        return [top] + [int(x) for x in rng.integers(max(1, top // 2), top + 1, n - 1)]
    n, total = case["segments"], case["tokens"]
    if n == 1:
        return [total]
    shares = rng.uniform(0.05, 1.0, n)
    lengths = np.maximum(1, np.floor(shares / shares.sum() * total)).astype(int)
    lengths[int(np.argmax(lengths))] += total - int(lengths.sum())
    return [int(x) for x in lengths]


def _vision(case):
    """Vision-block ID of every token (-1: text): runs of 256 to 1120 tokens, about 15% of a sample."""
    if not case.get("vision"):
        return None
    rng = np.random.default_rng(case["shape"] + 1)
    lengths = _lengths(case)
    ids = np.full(sum(lengths), -1, dtype=np.int32)
    start = block = 0
    for n in lengths:
        at = 0
        while True:
            gap, size = int(rng.integers(64, 7000)), int(rng.integers(256, 1121))
            if n < 2000:  # a short sample holds one image
                gap, size = n // 4, min(size, n // 2)
            if at + gap + size > n or size < 1:
                break
            ids[start + at + gap: start + at + gap + size] = block
            block += 1
            at += gap + size
            if n < 2000:
                break
        start += n
    return ids


def _window(case):
    layer = case.get("layer", "global" if case["kind"] == "extend" else "local")
    return WINDOW if layer == "local" else None


def _pairs(case):
    """Allowed (query, key) pairs of one head."""
    window, kind = _window(case), case["kind"]
    total = 0
    for n in _lengths(case):
        first = n - 1 if kind == "decode" else n - case["new"] if kind == "extend" else 0
        seen = np.arange(first + 1, n + 1, dtype=np.int64)
        total += int((seen if window is None else np.minimum(seen, window)).sum())
    ids = _vision(case)
    if ids is not None:  # the later keys of a row's own block
        change = np.flatnonzero(np.diff(ids)) + 1
        for run in np.split(np.arange(ids.size), change):
            if ids[run[0]] >= 0:
                total += run.size * (run.size - 1) // 2
    return total


def work(case):
    kind = case["kind"]
    if kind == "kv_prep":
        s, d, h = case["seqlen"], HEAD_DIM["global"], KV_HEADS["global"]
        rows, kb = s * h * d, 4 if case["tables"] == "fp32" else 2
        tables = 2 * s * ROTARY * kb + 4 * d
        # forward: Z in, K and V out; backward: Z, dK and dV in, dZ and dW out
        return {"bytes": rows * (2 + kb + 2) + rows * (2 + kb + 2 + 2) + 2 * tables + 4 * d,
                "flops": 0}
    layer = case.get("layer", "global" if kind == "extend" else "local")
    d, hkv = HEAD_DIM[layer], KV_HEADS[layer]
    pairs, keys = _pairs(case), sum(_lengths(case))
    queries = case["batch"] if kind == "decode" else case["new"] if kind == "extend" else keys
    forward = 2.0 * Q_HEADS * pairs * 2 * d
    qo, kv, lse = queries * Q_HEADS * d * 2, keys * hkv * d * 2, queries * Q_HEADS * 4
    if kind == "layer":
        proj = HIDDEN * d * (2 * Q_HEADS + 2 * hkv)
        return {"bytes": 2 * proj + 4 * keys * HIDDEN + 4 * keys * d + lse,
                "flops": 2.0 * keys * proj + forward}
    if kind in ("decode", "extend"):
        return {"bytes": 2 * qo + 2 * kv + lse, "flops": forward}
    # q, dO in, O, dQ out; K, V in, dK, dV out
    return {"bytes": 4 * qo + 4 * kv + lse, "flops": 3.5 * forward}


def tolerance(case):
    # Four times what the path differs from 64 bits by: bf16 results of 32-bit sums over
    # bf16-rounded P and dS (2.5e-3), of element-wise work (2e-3), and of a whole layer with
    # its bf16 intermediates (5.3e-3).
    return {"rel": {"kv_prep": 8e-3, "layer": 2e-2}.get(case["kind"], 1e-2)}


# ---------------------------------------------------------------------------
# inputs and calls
# ---------------------------------------------------------------------------


class _Values:
    def __init__(self, seed):
        self.g = torch.Generator(device=DEVICE).manual_seed(seed)

    def normal(self, *shape, std=1.0):
        return torch.randn(*shape, generator=self.g, device=DEVICE).mul_(std).to(torch.bfloat16)

    def uniform(self, *shape, lo, hi):
        return torch.rand(*shape, generator=self.g, device=DEVICE).mul_(hi - lo).add_(lo)


def _rope(seqlen, dim, theta, dtype):
    inv = theta ** (-torch.arange(0, dim, 2, device=DEVICE, dtype=torch.float64) / dim)
    angle = torch.arange(seqlen, device=DEVICE, dtype=torch.float64)[:, None] * inv
    angle = torch.cat((angle, angle), dim=1)
    return angle.cos().to(dtype), angle.sin().to(dtype)


def _cu(lengths):
    return torch.tensor([0, *np.cumsum(lengths).tolist()], dtype=torch.int32, device=DEVICE)


def prepare(case, seed):
    kind, r = case["kind"], _Values(seed)
    st = {"case": case}
    if kind == "kv_prep":
        s, h, d = case["seqlen"], KV_HEADS["global"], HEAD_DIM["global"]
        dt = torch.float32 if case["tables"] == "fp32" else torch.bfloat16
        st["z"] = r.normal(1, h, s, d).requires_grad_(True)
        st["w"] = r.uniform(d, lo=0.15, hi=0.3).requires_grad_(True)
        st["cos"], st["sin"] = _rope(s, ROTARY, 1e6, dt)
        st["dk"], st["dv"] = r.normal(1, h, s, d).to(dt), r.normal(1, h, s, d)
        return st
    if kind == "layer":
        s, d, h = case["seqlen"], HEAD_DIM["local"], KV_HEADS["local"]
        cos, sin = _rope(s, d, 1e4, torch.bfloat16)
        std = HIDDEN ** -0.5
        st["args"] = [
            r.normal(1, s, HIDDEN), cos[None].contiguous(), sin[None].contiguous(),
            torch.arange(s, device=DEVICE)[None].contiguous(),
            torch.zeros(1, s, dtype=torch.int64, device=DEVICE),
            r.normal(Q_HEADS * d, HIDDEN, std=std), r.normal(h * d, HIDDEN, std=std),
            r.normal(h * d, HIDDEN, std=std), r.normal(HIDDEN, Q_HEADS * d, std=(Q_HEADS * d) ** -0.5),
            r.uniform(d, lo=0.2, hi=0.3).to(torch.bfloat16),
            r.uniform(d, lo=0.2, hi=0.3).to(torch.bfloat16)]
        return st
    layer = case.get("layer", "global")
    d, h, lengths = HEAD_DIM[layer], KV_HEADS[layer], _lengths(case)
    keys = sum(lengths)
    std = d ** -0.25  # logits of unit variance at softmax scale 1
    if kind == "extend" or (kind == "decode" and layer == "global" and case["batch"] == 1):
        new = case.get("new", 1)
        st["q"] = r.normal(1, new, Q_HEADS, d, std=std)
        # the filled part of a StaticCache backing (heads outside tokens) with room left
        room = (keys // 1024 + 2) * 1024
        st["k"] = r.normal(1, h, room, d, std=std)[:, :, :keys].transpose(1, 2)
        st["v"] = r.normal(1, h, room, d)[:, :, :keys].transpose(1, 2)
        return st
    queries = case["batch"] if kind == "decode" else keys
    st["q"] = r.normal(queries, Q_HEADS, d, std=std)
    st["k"], st["v"] = r.normal(keys, h, d, std=std), r.normal(keys, h, d)
    st["cu_k"] = _cu(lengths)
    st["max_k"] = max(lengths)
    if kind == "decode":
        st["cu_q"], st["max_q"] = _cu([1] * queries), 1
        return st
    st["cu_q"], st["max_q"] = st["cu_k"], st["max_k"]
    st["do"] = r.normal(queries, Q_HEADS, d)
    ids = _vision(case)
    st["vision"] = None if ids is None else torch.from_numpy(ids).to(DEVICE)
    st["documents"] = None
    if case.get("documents"):
        st["documents"] = torch.repeat_interleave(
            torch.arange(len(lengths), dtype=torch.int32, device=DEVICE),
            torch.tensor(lengths, device=DEVICE))
    if kind == "train_fixed":
        for name in ("q", "k", "v", "do"):
            st[name] = st[name][None]
        if ids is not None:
            st["vision"] = st["vision"][None]
    for name in ("q", "k", "v"):
        st[name].requires_grad_(True)
    return st


def run(st):
    case = st["case"]
    kind, layer = case["kind"], case.get("layer")
    if kind == "kv_prep":
        k, v = g4.prepare_global_kv_from_projection_source(
            st["z"], k_norm_weight=st["w"], cos=st["cos"], sin=st["sin"])
        dz, dw = torch.autograd.grad((k, v), (st["z"], st["w"]), (st["dk"], st["dv"]))
        return {"k": k, "v": v, "dz": dz, "dw": dw}
    if kind == "layer":
        with torch.inference_mode():
            out, lse = torch_ops.local_layer_fwd(*st["args"])
        return {"out": out, "lse": lse}
    q, k, v = st["q"], st["k"], st["v"]
    if "cu_q" not in st:
        with torch.inference_mode():
            out, lse = g4.fa4_global_forward_only(q, k, v)
        return {"out": out, "lse": lse}
    lengths = {"max_seqlen_q": st["max_q"], "max_seqlen_k": st["max_k"]}
    if kind == "decode":
        call = g4.fa4_local_varlen_forward if layer == "local" else g4.fa4_global_varlen_forward_only
        with torch.no_grad():
            out, lse = call(q, k, v, st["cu_q"], st["cu_k"], **lengths)
        return {"out": out, "lse": lse}
    if kind == "train_fixed":
        if layer == "global":
            out, lse = g4.fa4_global_text_forward(q, k, v)
        else:
            out, lse = g4.fa4_local_forward(q, k, v, vision_block_ids=st["vision"])
    elif layer == "global":
        out, lse = g4.fa4_global_varlen_forward(q, k, v, st["cu_q"], st["cu_k"], **lengths)
    else:
        out, lse = g4.fa4_local_varlen_forward(
            q, k, v, st["cu_q"], st["cu_k"], vision_block_ids=st["vision"],
            document_ids=st["documents"], **lengths)
    dq, dk, dv = torch.autograd.grad(out, (q, k, v), st["do"])
    return {"out": out, "lse": lse, "dq": dq, "dk": dk, "dv": dv}


# ---------------------------------------------------------------------------
# the same results in 64 bits
# ---------------------------------------------------------------------------


def _rms(x):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS)


def _rotate(x, cos, sin):
    half = cos.shape[-1] // 2
    head, rest = x[..., : 2 * half], x[..., 2 * half:]
    turned = torch.cat((-head[..., half:], head[..., :half]), -1)
    return torch.cat((head * cos + turned * sin, rest), -1)


def _attention64(q, k, v, do, lengths_q, lengths_k, window, ids):
    """THD in any type -> O, LSE and, with do, dQ, dK, dV, all in 64 bits; a chunk of rows at a time."""
    hq, hkv, d = q.shape[1], k.shape[1], q.shape[2]
    group = hq // hkv
    out = torch.zeros(q.shape, dtype=torch.float64, device=q.device)
    lse = torch.zeros(hq, q.shape[0], dtype=torch.float64, device=q.device)
    dq = dk = dv = None
    if do is not None:
        dq = torch.zeros_like(out)
        dk = torch.zeros(k.shape, dtype=torch.float64, device=q.device)
        dv = torch.zeros_like(dk)
    q0 = k0 = 0
    for lq, lk in zip(lengths_q, lengths_k):
        kh = k[k0: k0 + lk].double().transpose(0, 1).contiguous()  # (Hkv, Lk, D)
        vh = v[k0: k0 + lk].double().transpose(0, 1).contiguous()
        seg = None if ids is None else ids[k0: k0 + lk]
        rows = 256 if window else max(1, min(512, (1 << 27) // (hq * lk)))
        for a in range(0, lq, rows):
            b = min(lq, a + rows)
            pos = torch.arange(a, b, device=q.device) + (lk - lq)
            lo = 0 if window is None else max(0, int(pos[0]) - window + 1)
            hi = int(pos[-1]) + 1
            if seg is not None:  # a vision row sees its block's later keys
                mine = seg[int(pos[0]): hi]
                mine = mine[mine >= 0]
                if mine.numel():
                    hi = max(hi, int(torch.isin(seg, mine).nonzero().max()) + 1)
            key = torch.arange(lo, hi, device=q.device)
            allowed = key[None, :] <= pos[:, None]
            if seg is not None:
                same = (seg[pos][:, None] == seg[key][None, :]) & (seg[pos] >= 0)[:, None]
                allowed = allowed | same
            if window is not None:
                allowed = allowed & (key[None, :] > pos[:, None] - window)

            def heads(t):  # (rows, Hq, D) -> (Hkv, group * rows, D)
                t = t[q0 + a: q0 + b].double().view(b - a, hkv, group, d)
                return t.permute(1, 2, 0, 3).reshape(hkv, group * (b - a), d)

            def tokens(t):
                return t.view(hkv, group, b - a, d).permute(2, 0, 1, 3).reshape(b - a, hq, d)

            qc, kc, vc = heads(q), kh[:, lo:hi].contiguous(), vh[:, lo:hi].contiguous()
            s = torch.bmm(qc, kc.transpose(1, 2).contiguous())
            s.view(hkv, group, b - a, hi - lo).masked_fill_(~allowed, -math.inf)
            l = torch.logsumexp(s, -1, keepdim=True)
            p = s.sub_(l).exp_()
            o = torch.bmm(p, vc)
            out[q0 + a: q0 + b] = tokens(o)
            lse[:, q0 + a: q0 + b] = l.view(hq, b - a)
            if do is not None:
                doc = heads(do)
                dv[k0 + lo: k0 + hi] += torch.bmm(p.transpose(1, 2).contiguous(), doc).transpose(0, 1)
                dp = torch.bmm(doc, vc.transpose(1, 2).contiguous())
                ds = dp.sub_((o * doc).sum(-1, keepdim=True)).mul_(p)
                dq[q0 + a: q0 + b] = tokens(torch.bmm(ds, kc))
                dk[k0 + lo: k0 + hi] += torch.bmm(ds.transpose(1, 2).contiguous(), qc).transpose(0, 1)
        q0, k0 = q0 + lq, k0 + lk
    return out, lse, dq, dk, dv


@torch.no_grad()
def _attention_exact(case, st):
    q, k, v, do = (st.get(n) for n in ("q", "k", "v", "do"))
    fixed = q.ndim == 4
    if fixed:
        q, k, v, do = (None if t is None else t[0] for t in (q, k, v, do))
    lengths = _lengths(case)
    new = [1] * len(lengths) if case["kind"] == "decode" else \
        [case["new"]] if case["kind"] == "extend" else lengths
    ids = st.get("vision")
    out, lse, dq, dk, dv = _attention64(q, k, v, do, new, lengths, _window(case),
                                        None if ids is None else ids.view(-1))
    got = {"out": out, "lse": lse}
    if do is not None:
        got.update(dq=dq, dk=dk, dv=dv)
    return {n: t[None] for n, t in got.items()} if fixed else got


@torch.no_grad()
def _layer_exact(st):
    x, cos, sin, _, _, wq, wk, wv, wo, qn, kn = (t.double() for t in st["args"])
    d, s = HEAD_DIM["local"], x.shape[1]
    cos, sin = cos[0][:, None], sin[0][:, None]
    q, k, v = ((x[0] @ w.t().contiguous()).view(s, -1, d) for w in (wq, wk, wv))
    q, k, v = _rotate(_rms(q) * qn, cos, sin), _rotate(_rms(k) * kn, cos, sin), _rms(v)
    o, lse, *_ = _attention64(q, k, v, None, [s], [s], WINDOW, None)
    return {"out": (o.reshape(s, -1) @ wo.t().contiguous())[None], "lse": lse[None]}


def _kv_prep_exact(st):
    z, w = (st[n].detach().double().requires_grad_(True) for n in ("z", "w"))
    cos, sin = st["cos"].double(), st["sin"].double()
    n = _rms(z)
    k = _rotate(n * w, cos, sin)
    dz, dw = torch.autograd.grad((k, n), (z, w), (st["dk"].double(), st["dv"].double()))
    return {"k": k.detach(), "v": n.detach(), "dz": dz, "dw": dw}


def exact(case, seed):
    st = prepare(case, seed)
    if case["kind"] == "kv_prep":
        return _kv_prep_exact(st)
    if case["kind"] == "layer":
        return _layer_exact(st)
    return _attention_exact(case, st)
