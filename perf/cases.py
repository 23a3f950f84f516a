"""What this framework is timed on: the calls of a GDN training or serving program.

Each case is one call (or one forward with its backward) of ``cqgdn.gated_delta_net`` or
``cqgdn.events`` on GPU tensors, at the sizes of this repository's benchmark configurations
and at generic ones between them.  The kinds:

* ``recurrent``      the recurrent step of N sequences, state updated in place;
* ``layer_decode``   one layer's whole decode step between its projections;
* ``train``          ``delta`` forward and backward over packed documents with read-only queries;
* ``prefill``        the precise forward with every document's final state;
* ``layer_train``    one layer between its projections, forward and backward, on an image-CQ plan;
* ``layer_prefill``  the same layer's inference prefill with the cache a decoder continues from;
* ``conv``           the packed causal conv1d, forward and backward.

``exact`` restates each call in float64 torch.
"""

import math
import random
import sys
from pathlib import Path
from types import SimpleNamespace

import torch
import torch.nn.functional as F

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "cq-pretrain_amd"))

from cqgdn import events  # noqa: E402
from cqgdn import gated_delta_net as gdn  # noqa: E402

D = 128  # the head dimension, the only one the framework takes
DEV = "cuda"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}


def listed():
    return [
        # one sequence's decode in an interactive session: a content token and its read-only query
        dict(name="decode_one", kind="recurrent", sequences=1, events=2, heads=16, dtype="bf16"),
        # a serving batch, one token each: the state is read and written once
        dict(name="decode_batch", kind="recurrent", sequences=64, events=1, heads=16, dtype="bf16"),
        # a layer's decode step with fewer key heads than value heads, an odd batch
        dict(name="layer_decode", kind="layer_decode", sequences=23, heads=32, key_heads=16, kernel=4),
        # the smallest training calls: one short document per step, one rank of a head-sharded layer
        dict(name="train_short", kind="train", content=317, docs=1, queries=0, heads=8, dtype="bf16", decay=1.0),
        # an image-generation step: 2048 content tokens, then one block of 256 read-only queries
        dict(name="train_image", kind="train", content=2048, docs=1, queries=256, heads=16, dtype="bf16", decay=1.0),
        # the headline: 8192 content tokens with four blocks of 256 queries between them
        dict(name="train_long", kind="train", content=8192, docs=1, queries=1024, heads=16, dtype="bf16", decay=1.0),
        # a pretraining microbatch: 32768 tokens of packed documents of 256 to 4096 tokens
        dict(name="train_packed", kind="train", content=32768, docs=15, queries=0, heads=16, dtype="bf16", decay=1.0),
        # a model trained in fp16, more heads, a few ragged documents, gates of a trained layer (long memory)
        dict(name="train_fp16", kind="train", content=5003, docs=3, queries=256, heads=32, dtype="fp16", decay=0.02),
        # a long prompt before decoding
        dict(name="prefill_long", kind="prefill", content=8192, docs=1, queries=0, heads=16, dtype="bf16", decay=1.0),
        # one layer of the width-2048 model on an image-CQ step: 2048 content tokens, 1675 queries, two image groups
        dict(name="layer_train", kind="layer_train", content=2048, queries=1675, image=249, docs=1, heads=16,
             key_heads=16, kernel=4),
        # the prompt of that model's larger sibling (32 value heads over 16 key heads), two packed prompts
        dict(name="layer_prefill", kind="layer_prefill", content=1537, queries=130, image=64, docs=2, heads=32,
             key_heads=16, kernel=4),
        # the layer's short convolution by itself (a layer with separate projections), one long document
        dict(name="conv_long", kind="conv", content=8192, docs=1, channels=6144, kernel=4),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("recurrent", "layer_decode", "train", "train", "train", "prefill", "layer_train",
                       "layer_prefill", "conv"))
    heads = rng.choice((4, 8, 16, 16, 32))
    most = 32768 * 16 // heads  # the largest listed case's event rows
    if kind == "recurrent":
        return dict(kind=kind, sequences=_log(rng, 1, 2048 // heads), events=rng.choice((1, 1, 2)), heads=heads,
                    dtype=rng.choice(("bf16", "bf16", "fp16")))
    if kind == "layer_decode":
        key_heads = rng.choice([x for x in (4, 8, 16, 32) if x <= heads and heads % x == 0])
        return dict(kind=kind, sequences=_log(rng, 1, 2048 // heads), heads=heads, key_heads=key_heads,
                    kernel=rng.choice((2, 3, 4, 4)))
    if kind in ("train", "prefill"):
        docs = rng.choice((1, 1, 1, _log(rng, 2, 40)))
        content = _log(rng, max(64, 32 * docs), most // 2)
        return dict(kind=kind, content=content, docs=docs, queries=256 * rng.choice((0, 0, 1, 4)), heads=heads,
                    dtype=rng.choice(("bf16", "bf16", "fp16")),
                    decay=round(math.exp(rng.uniform(math.log(0.005), 0.0)), 4))
    if kind in ("layer_train", "layer_prefill"):
        key_heads = rng.choice([x for x in (4, 8, 16, 32) if x <= heads and heads % x == 0])
        docs = rng.choice((1, 1, 2, 5))
        content = docs * _log(rng, 100, 4096 * 16 // heads // docs)
        return dict(kind=kind, content=content, queries=rng.randrange(content), image=rng.choice((0, 16, 49)),
                    docs=docs, heads=heads, key_heads=key_heads, kernel=rng.choice((2, 4, 4)))
    return dict(kind="conv", content=_log(rng, 64, 16384), docs=rng.choice((1, 1, 7)),
                channels=8 * _log(rng, 64, 1024), kernel=rng.choice((2, 3, 4, 4)))


# ---- inputs --------------------------------------------------------------------------------


def _bounds(total, docs, rnd):
    """Document bounds (0, ..., total): `docs` documents of uneven lengths, none empty."""
    weights = [rnd.uniform(1, 16) for _ in range(docs)]
    bounds, at = [0], 0.0
    for i, w in enumerate(weights):
        at += w / sum(weights)
        left = docs - 1 - i
        bounds.append(total if left == 0 else min(max(bounds[-1] + 1, round(total * at)), total - left))
    return tuple(bounds)


def _readonly(content, queries, docs, rnd):
    """(events, bounds, read-only mask): query blocks of 256 at seeded places of the packed documents (a
    single block follows the content)."""
    blocks = queries // 256
    if blocks == 0:
        return content, _bounds(content, docs, rnd), None
    cuts = [content] if blocks == 1 else sorted(rnd.randrange(content + 1) for _ in range(blocks))
    mask = torch.zeros(content + queries, dtype=torch.bool)
    for i, cut in enumerate(cuts):
        mask[cut + 256 * i:cut + 256 * (i + 1)] = True
    return content + queries, _bounds(content + queries, docs, rnd), mask


def _randn(gen, *shape, dtype=torch.bfloat16):
    return torch.randn(*shape, generator=gen, device=DEV).to(dtype)


def _qkv(gen, T, H, dtype, decay, mask):
    q, k, v = (_randn(gen, 1, T, H, D, dtype=dtype) for _ in range(3))
    beta = torch.randn(1, T, H, generator=gen, device=DEV).sigmoid()
    g = -decay * F.softplus(torch.randn(1, T, H, generator=gen, device=DEV))
    if mask is not None:  # read-only queries write nothing: no key, no value, no gate
        keep = (~mask.to(DEV)).view(1, T, 1)
        k, v = k * keep[..., None], v * keep[..., None]
        g, beta = g * keep, beta * keep
    return q, k, v, g, beta


def _document_plan(content, queries, image, kernel, rnd):
    """One document: content rows in order (an image group of `image` tokens is written, then read again),
    each query reading before a random group.  Lists of (q source, row written) per event and the rows' events."""
    groups, at = [], 0
    start = rnd.randrange(content - image + 1) if image else -1
    while at < content:
        size = image if at == start else 1
        groups.append(range(at, at + size))
        at += size
    waiting = {}
    for j in range(queries):
        waiting.setdefault(rnd.randrange(len(groups)), []).append(j)
    reads, history, out_c, out_q = [], [None] * queries, [0] * content, [0] * queries
    for i, group in enumerate(groups):
        for j in waiting.get(i, ()):
            history[j] = [group[0] - kernel + 1 + x for x in range(kernel - 1)]
            out_q[j] = len(reads)
            reads.append(("q", j, None))
        for c in group:
            out_c[c] = len(reads)
            reads.append(("c", c, c))
        if len(group) > 1:
            for c in group:
                out_c[c] = len(reads)
                reads.append(("c", c, None))
    return reads, history, out_c, out_q


def _plan(case, rnd):
    """The event plan of a packed microbatch: hidden rows are all content rows, then all queries."""
    nc, nq, docs, K = case["content"], case["queries"], case["docs"], case["kernel"]
    cb = [nc * i // docs for i in range(docs + 1)]
    qb = [nq * i // docs for i in range(docs + 1)]
    eq, ew, hist, out_c, out_q, eb = [], [], [], [], [], [0]
    for d in range(docs):
        c0, q0, e0 = cb[d], qb[d], len(eq)
        reads, h, oc, oq = _document_plan(cb[d + 1] - c0, qb[d + 1] - q0, case["image"], K, rnd)
        eq += [c0 + i if what == "c" else nc + q0 + i for what, i, _ in reads]
        ew += [nc if w is None else c0 + w for _, _, w in reads]
        hist += [[c0 + x if x >= 0 else nc for x in row] for row in h]
        out_c += [e0 + e for e in oc]
        out_q += [e0 + e for e in oq]
        eb.append(len(eq))
    long = lambda xs: torch.tensor(xs, dtype=torch.long)  # noqa: E731
    return SimpleNamespace(
        content_order=torch.arange(nc), event_q=long(eq), event_write=long(ew),
        query_source=torch.arange(nc, nc + nq), query_history=long(hist).reshape(nq, K - 1),
        content_bounds=tuple(cb), event_bounds=tuple(eb), hidden_length=nc + nq,
        hidden_event=long(out_c + out_q), padding_hidden=torch.zeros(0, dtype=torch.long))


def _layer_parameters(gen, H, HK, K):
    C = (2 * HK + H) * D
    w = (torch.rand(C, K, generator=gen, device=DEV) - 0.5).bfloat16()
    A_log = (0.5 + 4 * torch.rand(H, generator=gen, device=DEV)).log()
    dt_bias = torch.randn(H, generator=gen, device=DEV) - 3.0
    norm = 1 + 0.1 * torch.randn(D, generator=gen, device=DEV)
    return w, A_log, dt_bias, norm


def prepare(case, seed):
    gdn.initialize()
    gen = torch.Generator(device=DEV).manual_seed(seed)
    rnd = random.Random(seed)
    s = SimpleNamespace(kind=case["kind"], case=case)
    H = case.get("heads")
    dtype = DTYPES[case.get("dtype", "bf16")]
    if s.kind == "recurrent":
        N, E = case["sequences"], case["events"]
        q, k, v = (torch.randn(N, E, H, D, generator=gen, device=DEV) for _ in range(3))
        g = -F.softplus(torch.randn(N, E, H, generator=gen, device=DEV))
        beta = torch.randn(N, E, H, generator=gen, device=DEV).sigmoid()
        if E == 2:  # the second event is the read-only query
            k[:, 1], v[:, 1], g[:, 1], beta[:, 1] = 0, 0, 0, 0
        q, k = (x * torch.rsqrt(x.square().sum(-1, keepdim=True) + 1e-6) for x in (q, k))
        s.q, s.k, s.v, s.g, s.beta = q.to(dtype), k.to(dtype), v.to(dtype), g, beta
        s.state = 0.02 * torch.randn(N, H, D, D, generator=gen, device=DEV)
        s.out = torch.empty_like(s.v)
    elif s.kind == "layer_decode":
        N, HK, K = case["sequences"], case["key_heads"], case["kernel"]
        s.parameters = _layer_parameters(gen, H, HK, K)
        s.proj = _randn(gen, N, 2, (2 * HK + 2 * H) * D + 2 * H)
        s.cache = dict(conv=_randn(gen, N, K - 1, (2 * HK + H) * D),
                       state=0.02 * torch.randn(N, H, D, D, generator=gen, device=DEV))
    elif s.kind in ("train", "prefill"):
        T, s.bounds, mask = _readonly(case["content"], case["queries"], case["docs"], rnd)
        xs = _qkv(gen, T, H, dtype, case["decay"], mask)
        if s.kind == "train":
            s.inputs = [x.requires_grad_() for x in xs]
            s.grad = _randn(gen, 1, T, H, D, dtype=dtype)
            s.cu = torch.tensor(s.bounds, device=DEV)
        else:
            s.inputs = xs
    elif s.kind in ("layer_train", "layer_prefill"):
        HK, K = case["key_heads"], case["kernel"]
        s.plan = _plan(case, rnd)
        events.event_plan(s.plan, K, torch.device(DEV, torch.cuda.current_device()))  # one plan serves every layer
        s.proj = _randn(gen, s.plan.hidden_length, (2 * HK + 2 * H) * D + 2 * H)
        s.parameters = _layer_parameters(gen, H, HK, K)
        if s.kind == "layer_train":
            s.inputs = [x.requires_grad_() for x in (s.proj, *s.parameters)]
            s.grad = _randn(gen, s.plan.hidden_length, H * D)
    else:
        s.bounds = _bounds(case["content"], case["docs"], rnd)
        s.cu = torch.tensor(s.bounds, device=DEV)
        C, K = case["channels"], case["kernel"]
        s.inputs = [_randn(gen, 1, case["content"], C).requires_grad_(),
                    (torch.rand(C, K, generator=gen, device=DEV) - 0.5).bfloat16().requires_grad_()]
        s.grad = _randn(gen, 1, case["content"], C)
    return s


# ---- one pass ------------------------------------------------------------------------------


def run(s):
    case = s.case
    if s.kind == "recurrent":
        return gdn.recurrent(s.q, s.k, s.v, s.g, s.beta, s.state, s.out), s.state
    if s.kind == "layer_decode":
        out = events.layer_decode_step(s.proj, *s.parameters, s.cache, heads=case["heads"],
                                       key_heads=case["key_heads"])
        return out, s.cache["conv"], s.cache["state"]
    if s.kind == "train":
        o, _ = gdn.delta(*s.inputs, use_qk_l2norm_in_kernel=True, cu_seqlens=s.cu, cu_seqlens_cpu=s.bounds)
        return (o, *torch.autograd.grad(o, s.inputs, s.grad))
    if s.kind == "prefill":
        return gdn.prefill(*s.inputs, s.bounds)
    if s.kind == "layer_train":
        out = events.layer_core(*s.inputs, s.plan, heads=case["heads"], key_heads=case["key_heads"])
        return (out, *torch.autograd.grad(out, s.inputs, s.grad))
    if s.kind == "layer_prefill":
        out, cache = events.layer_prefill(s.proj, *s.parameters, s.plan, heads=case["heads"],
                                          key_heads=case["key_heads"])
        return out, cache["state"], cache["conv"]
    y, _ = gdn.conv(*s.inputs, activation="silu", cu_seqlens=s.cu, cu_seqlens_cpu=s.bounds)
    return (y, *torch.autograd.grad(y, s.inputs, s.grad))


# ---- work and tolerance --------------------------------------------------------------------


def _gdn_flops(T, H, backward):
    """The chunked form's least contractions at chunk 64 (cqgdn/workmodel.py), per event and head."""
    c = 64
    fwd = 10 * c * c * D + 6 * c * D * D + 2 * c ** 3 / 3
    bwd = 20 * c * c * D + 12 * c * D * D + 4 * c ** 3
    return T * H / c * (fwd + (bwd if backward else 0))


def work(case):
    kind, H, E = case["kind"], case.get("heads"), case.get("events")
    if kind == "recurrent":
        rows = case["sequences"] * H
        return {"bytes": rows * (2 * D * D * 4 + E * (4 * D * 2 + 8)), "flops": rows * E * 7 * D * D}
    if kind == "layer_decode":
        N, HK, K = case["sequences"], case["key_heads"], case["kernel"]
        C = (2 * HK + H) * D
        row = 2 * (C + H * D + 2 * H) * 2 + 2 * (K - 1) * C * 2 + 2 * H * D * 2 + 2 * H * D * D * 4
        return {"bytes": N * row + C * K * 2, "flops": N * H * 9 * D * D}
    if kind == "train":
        T = case["content"] + case["queries"]
        return {"bytes": T * H * (8 * D * 2 + 4 * 4), "flops": _gdn_flops(T, H, True)}
    if kind == "prefill":
        T = case["content"] + case["queries"]
        return {"bytes": T * H * (4 * D * 2 + 8) + case["docs"] * H * D * D * 4, "flops": _gdn_flops(T, H, False)}
    if kind in ("layer_train", "layer_prefill"):
        HK, K, rows = case["key_heads"], case["kernel"], case["content"] + case["queries"]
        P = (2 * HK + 2 * H) * D + 2 * H
        T = rows + case["image"] * case["docs"]
        if kind == "layer_train":  # the projection and its gradient, the output and its gradient
            return {"bytes": rows * 2 * (2 * P + 2 * H * D), "flops": _gdn_flops(T, H, True)}
        state = case["docs"] * H * D * D * 4
        return {"bytes": rows * 2 * (P + H * D) + state, "flops": _gdn_flops(T, H, False)}
    n = case["content"] * case["channels"]
    return {"bytes": 4 * n * 2, "flops": n * (6 * case["kernel"] + 20)}


def tolerance(case):
    kind = case["kind"]
    if kind in ("recurrent", "conv"):  # fp32 arithmetic, each 16-bit output rounded once
        return {"rel": 4e-3}
    if kind == "layer_decode":  # 16-bit q, k, v and y between the layer's parts
        return {"rel": 8e-3}
    if kind == "prefill":  # fp16 operands, o rounded once to 16 bits
        return {"rel": 6e-3}
    if kind == "train" and case["dtype"] == "fp16":
        return {"rel": 3e-3}
    return {"rel": 2e-2}  # bf16 operands through the chunked chain


# ---- the same in 64 bits -------------------------------------------------------------------


def _delta64(q, k, v, g, beta, bounds, scale=D ** -0.5):
    """The gated delta rule over packed documents in float64, chunked: o [T, H, D] and the final states
    [docs, H, K, V].  Documents are padded to one length with events that change nothing."""
    n, H = len(bounds) - 1, q.shape[1]
    chunks = max(1, max((b - a + 63) // 64 for a, b in zip(bounds, bounds[1:])))
    pad = chunks * 64
    slot = torch.cat([torch.arange(b - a) + i * pad for i, (a, b) in enumerate(zip(bounds, bounds[1:]))]).to(q.device)

    def chunked(x):  # [T, H, ...] -> [docs, H, chunks, 64, ...]
        y = x.new_zeros(n * pad, *x.shape[1:]).index_copy(0, slot, x)
        return y.reshape(n, chunks, 64, *x.shape[1:]).movedim(3, 1)

    norm = lambda x: x * torch.rsqrt(x.square().sum(-1, keepdim=True) + 1e-6)  # noqa: E731
    q, k, v, g, beta = (chunked(x) for x in (norm(q) * scale, norm(k), v, g, beta))
    G = g.cumsum(-1)
    lower = torch.ones(64, 64, dtype=torch.bool, device=q.device).tril()
    gates = (G[..., :, None] - G[..., None, :]).masked_fill(~lower, -math.inf).exp()
    A = (k @ k.transpose(-1, -2) * gates * beta[..., None]).tril(-1)
    X = torch.eye(64, dtype=q.dtype, device=q.device) - A  # (I + A)^-1 = (I - A)(I + A^2)(I + A^4) ...
    P = A
    for _ in range(5):
        P = P @ P
        X = X + X @ P
    U = X @ (beta[..., None] * v)
    W = X @ ((beta * G.exp())[..., None] * k)
    scores = q @ k.transpose(-1, -2) * gates
    q_in, k_out = q * G.exp()[..., None], k * (G[..., -1:] - G).exp()[..., None]
    S, outs = q.new_zeros(n, H, D, D), []
    for c in range(chunks):
        new = U[:, :, c] - W[:, :, c] @ S
        outs.append(q_in[:, :, c] @ S + scores[:, :, c] @ new)
        S = S * G[:, :, c, -1, None, None].exp() + k_out[:, :, c].transpose(-1, -2) @ new
    o = torch.stack(outs, 2).movedim(1, 3).reshape(n * pad, H, D)
    return o.index_select(0, slot), S


def _conv64(x, w, bounds):
    K = w.shape[1]
    y = []
    for a, b in zip(bounds, bounds[1:]):
        rows = F.pad(x[a:b], (0, 0, K - 1, 0))
        y.append(sum(rows[i:i + b - a] * w[:, i] for i in range(K)))
    return F.silu(torch.cat(y))


def _layer64(proj, w, A_log, dt_bias, norm, plan, H, HK):
    SK, SV = HK * D, H * D
    raw, z, a, b = proj.split((2 * SK + SV, SV, H, H), -1)
    dev = lambda t: t.to(proj.device)  # noqa: E731
    order, source, history = dev(plan.content_order), dev(plan.query_source), dev(plan.query_history)
    read, write = dev(plan.event_q), dev(plan.event_write)
    rows = raw.index_select(0, order)
    q, k, v = _conv64(rows, w, plan.content_bounds).split((SK, SK, SV), -1)
    before = torch.cat((rows[:, :SK], rows.new_zeros(1, SK)))
    query = raw[:, :SK].index_select(0, source) * w[:SK, -1]
    for j in range(w.shape[1] - 1):
        query = query + before.index_select(0, history[:, j]) * w[:SK, j]
    wide = lambda x: x.reshape(-1, HK, D).repeat_interleave(H // HK, dim=1)  # noqa: E731
    q = torch.cat((wide(q), wide(F.silu(query)))).index_select(0, read)
    pick = lambda x: torch.cat((x, x.new_zeros(1, *x.shape[1:]))).index_select(0, write)  # noqa: E731
    a, b = a.index_select(0, order), b.index_select(0, order)
    y, state = _delta64(q, pick(wide(k)), pick(v.reshape(-1, H, D)), pick(-A_log.exp() * F.softplus(a + dt_bias)),
                        pick(b.sigmoid()), plan.event_bounds)
    y = y.index_select(0, dev(plan.hidden_event))
    y = y * torch.rsqrt(y.square().mean(-1, keepdim=True) + 1e-6) * norm * F.silu(z.reshape(-1, H, D))
    return y.flatten(1), state, rows


def _step64(q, k, v, g, beta, state):
    """One event of every sequence: q, k, v [N, H, D], state [N, H, V, K]; returns the output and the state."""
    state = state * g.exp()[..., None, None]
    new = beta[..., None] * (v - (state @ k[..., None])[..., 0])
    state = state + new[..., None] * k[..., None, :]
    return D ** -0.5 * (state @ q[..., None])[..., 0], state


def exact(case, seed):
    s = prepare(case, seed)
    if s.kind == "recurrent":
        q, k, v, g, beta, state = (x.double() for x in (s.q, s.k, s.v, s.g, s.beta, s.state))
        outs = []
        for e in range(case["events"]):
            o, state = _step64(q[:, e], k[:, e], v[:, e], g[:, e], beta[:, e], state)
            outs.append(o)
        return torch.stack(outs, 1), state
    H = case.get("heads")
    if s.kind == "layer_decode":
        HK = case["key_heads"]
        SK, SV = HK * D, H * D
        w, A_log, dt_bias, norm = (x.double() for x in s.parameters)
        raw, z, a, b = s.proj.double().split((2 * SK + SV, SV, H, H), -1)
        past = torch.cat((s.cache["conv"].double(), raw[:, :1]), 1)  # K rows: the history, then the new token
        q, k, v = F.silu((past * w.t()).sum(1)).split((SK, SK, SV), -1)
        query = F.silu((past[:, 1:, :SK] * w[:SK, :-1].t()).sum(1) + raw[:, 1, :SK] * w[:SK, -1])
        unit = lambda x: x * torch.rsqrt(x.square().sum(-1, keepdim=True) + 1e-6)  # noqa: E731
        wide = lambda x: unit(x.reshape(-1, HK, D)).repeat_interleave(H // HK, dim=1)  # noqa: E731
        g = -A_log.exp() * F.softplus(a[:, 0] + dt_bias)
        o, state = _step64(wide(q), wide(k), v.reshape(-1, H, D), g, b[:, 0].sigmoid(), s.cache["state"].double())
        o2 = D ** -0.5 * (state @ wide(query)[..., None])[..., 0]
        y = torch.stack((o, o2), 1)
        y = y * torch.rsqrt(y.square().mean(-1, keepdim=True) + 1e-6) * norm * F.silu(z.reshape(-1, 2, H, D))
        return y, past[:, 1:], state
    if s.kind == "train":
        xs = [x.detach()[0].double().requires_grad_() for x in s.inputs]
        o, _ = _delta64(*xs, s.bounds)
        return tuple(x[None] for x in (o.detach(), *torch.autograd.grad(o, xs, s.grad[0].double())))
    if s.kind == "prefill":
        o, state = _delta64(*(x[0].double() for x in s.inputs), s.bounds)
        return o[None], state
    if s.kind == "layer_train":
        xs = [x.detach().double().requires_grad_() for x in s.inputs]
        y, _, _ = _layer64(*xs, s.plan, H, case["key_heads"])
        return (y.detach(), *torch.autograd.grad(y, xs, s.grad.double()))
    if s.kind == "layer_prefill":
        y, state, rows = _layer64(s.proj.double(), *(x.double() for x in s.parameters), s.plan, H, case["key_heads"])
        K = case["kernel"]
        tail = F.pad(rows[:-1], (0, 0, K - 1, 0))[len(rows) - 1:]  # the K-1 content rows before the last one
        return y, state.transpose(-1, -2), tail[None]
    xs = [x.detach().double().requires_grad_() for x in s.inputs]
    y = _conv64(xs[0][0], xs[1], s.bounds)
    return (y.detach()[None], *torch.autograd.grad(y, xs, s.grad[0].double()))
