"""What a user has this framework do, as timed cases.

A case is one call (or one training step) through the public operators: block selection
(``m3_index_score_topk``), the indexer score with its gradients, top-k alone, sparse
attention forward (prefill) and forward + backward (training), and a whole sparse layer
with the indexer's KL loss. Sizes are the benchmark's configurations (1 280 to 65 536
tokens), ragged packs of odd lengths, head dims 64 to 256 and the three input types.

``exact`` restates every operator densely in float64 with plain torch.
"""

from __future__ import annotations

import torch

import msa_triton_amd as msa

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
DEVICE = "cuda"
KL_WEIGHT = 0.1  # weight of the indexer loss beside the layer's own gradient

# A serving batch: many requests of uneven length.
REQUESTS = ("1837,96,411,733,1290,57,208,1544,367,905,129,640,1021,288,77,1466,512,353,842,190,"
            "1127,33,675,1713,246,401,989,150,1358,568,301,784")


def listed():
    return [
        # Smallest training step: the benchmark's two-sequence configuration (c1), called as a drop-in
        # (plain cu_seqlens): selection, attention, KL and all gradients. Launches and host work count.
        dict(name="layer_small", op="layer", dtype="bf16", lengths="512,768", hq=8, g=2, d=64, di=64, block=128,
             topk=4, local=1, prepared=False),
        # A training step of one layer on a ragged pack (c3's size, odd lengths) with prepared metadata.
        dict(name="layer_varlen", op="layer", dtype="bf16", lengths="2047,3071,5003,6151", hq=32, g=4, d=128,
             di=128, block=128, topk=16, local=1, prepared=True),
        # The headline benchmark (c4): attention forward + backward of one 32K sequence.
        dict(name="train_32k", op="train", dtype="bf16", lengths="32768", hq=32, g=4, d=128, block=128, topk=16,
             local=1, prepared=False),
        # fp16 training at 8K (c2).
        dict(name="train_fp16", op="train", dtype="fp16", lengths="8192", hq=32, g=4, d=128, block=128, topk=16,
             local=1, prepared=True),
        # fp32 training, as used to check a model before it goes to 16 bits: a small ragged pack.
        dict(name="train_fp32", op="train", dtype="fp32", lengths="701,1347", hq=16, g=2, d=128, block=128, topk=8,
             local=1, prepared=False),
        # A model with wide heads at 8K.
        dict(name="train_d256", op="train", dtype="bf16", lengths="8192", hq=16, g=2, d=256, block=128, topk=16,
             local=1, prepared=True),
        # Prefill of a serving batch: forward only, many short requests.
        dict(name="prefill_batch", op="prefill", dtype="bf16", lengths=REQUESTS, hq=32, g=4, d=128, block=128,
             topk=16, local=1, prepared=True),
        # Block selection of one 32K sequence (c4) in inference.
        dict(name="select_32k", op="select", dtype="bf16", lengths="32768", g=4, di=128, block=128, topk=16,
             local=1, prepared=True),
        # Block selection in fp16 at 8K.
        dict(name="select_fp16", op="select", dtype="fp16", lengths="8192", g=4, di=128, block=128, topk=16,
             local=1, prepared=True),
        # Block selection in fp32, beside the fp32 training case.
        dict(name="select_fp32", op="select", dtype="fp32", lengths="701,1347", g=2, di=128, block=128, topk=8,
             local=1, prepared=False),
        # Indexer scores with gradients on c3's pack.
        dict(name="score_train", op="score", dtype="bf16", lengths="2048,3072,5120,6144", g=4, di=128, block=128,
             prepared=True),
        # Top-k of the largest configuration (c5): 64K tokens, 512 blocks, 32 slots.
        dict(name="topk_64k", op="topk", dtype="fp32", lengths="65536", g=8, block=128, topk=32, local=2,
             prepared=True),
    ]


def _lengths(rng, tokens, most):
    """`tokens` tokens in 1 to `most` sequences of uneven length."""
    n = min(rng.choice([1, 1, 2, 3, 5, 8, 13, 24]), most, max(1, tokens // 40))
    cuts = sorted(rng.sample(range(1, tokens), n - 1)) if n > 1 else []
    return ",".join(str(b - a) for a, b in zip([0, *cuts], [*cuts, tokens]))


def _log_uniform(rng, low, high):
    return int(round(low * (high / low) ** rng.random()))


def draw(rng):
    op = rng.choice(["layer", "train", "train", "prefill", "select", "select", "score", "topk"])
    dtype = "bf16" if op in ("layer", "score", "prefill") else rng.choice(["bf16", "bf16", "fp16", "fp32"])
    if op == "topk":
        dtype = "fp32"
    high = {"layer": 16000, "train": 16000, "prefill": 16000, "select": 32000, "score": 16000, "topk": 48000}[op]
    if op in ("train", "select") and dtype != "bf16":
        high = 8000 if dtype == "fp16" else 2000
    case = dict(op=op, dtype=dtype, block=rng.choice([128, 128, 128, 64]), prepared=rng.random() < 0.5)
    wide = op in ("train", "prefill") and dtype != "fp32" and rng.random() < 0.25
    if wide:
        high = 8000
    if op != "topk":
        case["lengths"] = _lengths(rng, _log_uniform(rng, 300, high), 24)
    else:
        case["lengths"] = _lengths(rng, _log_uniform(rng, 1000, high), 8)
    case["g"] = rng.choice([2, 4]) if op != "topk" else rng.choice([2, 4, 8])
    if op in ("layer", "train", "prefill"):
        case["hq"] = case["g"] * rng.choice([4, 8])
        if dtype == "fp32":
            case["hq"] = case["g"] = 2
            case["hq"] *= rng.choice([4, 8])
        case["d"] = rng.choice([64, 128]) if op == "layer" else rng.choice([64, 96, 128, 128])
        if wide:
            case["hq"], case["g"] = 16, 2
            case["d"] = rng.choice([192, 256])
    if op in ("layer", "select", "score"):
        case["di"] = rng.choice([64, 128, 128])
    if op != "score":
        case["topk"] = rng.choice([4, 8, 16] if dtype != "fp32" or op == "topk" else [4, 8])
        if op == "topk":
            case["topk"] = rng.choice([8, 16, 32])
        case["local"] = rng.choice([1, 1, 2])
    return case


# ---------------------------------------------------------------------------- inputs


def _bounds(case):
    lengths = [int(x) for x in case["lengths"].split(",")]
    bounds = [0]
    for n in lengths:
        bounds.append(bounds[-1] + n)
    return bounds


def _max_blocks(case):
    bounds = _bounds(case)
    return -(-max(b - a for a, b in zip(bounds, bounds[1:])) // case["block"])


def _positions(bounds):
    """Position of each token in its sequence."""
    pos = [torch.arange(b - a) for a, b in zip(bounds, bounds[1:])]
    return torch.cat(pos).to(DEVICE)


def _block_scores(case, gen):
    """Indexer-like block scores [T, G, NB] (some blocks more popular than others), -inf for blocks after the
    query's."""
    bounds = _bounds(case)
    total, nb = bounds[-1], _max_blocks(case)
    s = torch.randn(total, case["g"], nb, generator=gen, device=DEVICE)
    s += 0.3 * torch.randn(1, case["g"], nb, generator=gen, device=DEVICE)
    own = _positions(bounds) // case["block"]
    s.masked_fill_((torch.arange(nb, device=DEVICE)[None, :] > own[:, None])[:, None], float("-inf"))
    return s


def _selection(case, scores):
    """The selection the operators' contract gives for these scores: the current block and its predecessors
    (``local``) first, then by score; -1 where fewer blocks exist."""
    nb, k = scores.shape[2], case["topk"]
    own = (_positions(_bounds(case)) // case["block"])[:, None, None]
    b = torch.arange(nb, device=DEVICE)[None, None]
    s = scores.masked_fill((b <= own) & (b > own - case["local"]), float("inf"))
    v, ids = torch.topk(s, min(k, nb), dim=2)
    ids = torch.where(v == float("-inf"), -1, ids).to(torch.int32)
    pad = torch.full((*ids.shape[:2], k - ids.shape[2]), -1, dtype=torch.int32, device=DEVICE)
    return torch.cat([ids, pad], dim=2).contiguous()


def _inputs(case, seed):
    gen = torch.Generator(device=DEVICE).manual_seed(1000003 * int(seed) + 71)
    bounds = _bounds(case)
    total = bounds[-1]
    dtype = DTYPES[case["dtype"]]

    def randn(*shape):
        return torch.randn(*shape, generator=gen, device=DEVICE).to(dtype)

    x = {"max": max(b - a for a, b in zip(bounds, bounds[1:]))}
    op = case["op"]
    if op in ("layer", "select", "score"):
        x["iq"] = randn(total, case["g"], case["di"])
        x["ik"] = randn(total, 1, case["di"])
    if op in ("layer", "train", "prefill"):
        x["q"] = randn(total, case["hq"], case["d"])
        x["k"] = randn(total, case["g"], case["d"])
        x["v"] = randn(total, case["g"], case["d"])
    if op in ("layer", "train"):
        x["dout"] = randn(total, case["hq"], case["d"])
    if op in ("train", "prefill"):
        x["ids"] = _selection(case, _block_scores(case, gen))
    if op == "score":  # what a loss on the scores sends back: zero for blocks that do not exist
        own = (_positions(bounds) // case["block"])[:, None, None]
        ds = torch.randn(total, case["g"], _max_blocks(case), generator=gen, device=DEVICE)
        x["ds"] = ds * (torch.arange(ds.shape[2], device=DEVICE)[None, None] <= own)
    if op == "topk":
        x["scores"] = _block_scores(case, gen)
    return x


def prepare(case, seed):
    x = _inputs(case, seed)
    cu = torch.tensor(_bounds(case), dtype=torch.int32, device=DEVICE)
    x["cu"] = msa.prepare_sequences(cu, block_size=case["block"]) if case["prepared"] else cu
    x["case"] = case
    if case["op"] in ("layer", "train", "score"):
        for name in ("iq", "ik", "q", "k", "v"):
            if name in x:
                x[name].requires_grad_()
    return x


# ---------------------------------------------------------------------------- one pass


def run(x):
    case = x["case"]
    op, block = case["op"], case["block"]
    if op == "topk":
        return msa.m3_topk(x["scores"], x["cu"], block_size=block, topk_blocks=case["topk"],
                           local_blocks=case["local"])
    if op == "select":
        with torch.no_grad():
            return msa.m3_index_score_topk(x["iq"], x["ik"], x["cu"], x["max"], block_size=block,
                                           topk_blocks=case["topk"], local_blocks=case["local"])
    if op == "score":
        s = msa.m3_index_score(x["iq"], x["ik"], x["cu"], x["max"], block_size=block)
        return s.detach(), *torch.autograd.grad(s, (x["iq"], x["ik"]), x["ds"])
    if op == "prefill":
        with torch.no_grad():
            return msa.m3_sparse_attention(x["q"], x["k"], x["v"], x["ids"], x["cu"], x["max"], block_size=block)
    if op == "train":
        out = msa.m3_sparse_attention(x["q"], x["k"], x["v"], x["ids"], x["cu"], x["max"], block_size=block)
        return out.detach(), *torch.autograd.grad(out, (x["q"], x["k"], x["v"]), x["dout"])
    # layer: selection without gradient, attention, KL of the indexer against the attention
    with torch.no_grad():
        _, ids = msa.m3_index_score_topk(x["iq"], x["ik"], x["cu"], x["max"], block_size=block,
                                         topk_blocks=case["topk"], local_blocks=case["local"])
    out, lse = msa.m3_sparse_attention(x["q"], x["k"], x["v"], ids, x["cu"], x["max"], block_size=block,
                                       return_lse=True)
    kl = msa.m3_indexer_kl(x["iq"], x["ik"], x["q"].detach(), x["k"].detach(), ids, x["cu"], x["max"],
                           block_size=block, index_scale=case["di"] ** -0.5, teacher_lse=lse)
    loss = KL_WEIGHT * case["g"] * out.shape[0] * kl  # summed over the pairs, as dout is per token
    grads = torch.autograd.grad((out, loss), (x["q"], x["k"], x["v"], x["iq"], x["ik"]),
                                (x["dout"], torch.ones_like(loss)))
    return out.detach(), lse, kl.detach(), *grads


# ---------------------------------------------------------------------------- work


def work(case):
    bounds = _bounds(case)
    total, b, g = bounds[-1], case["block"], case["g"]
    pos = torch.cat([torch.arange(n1 - n0) for n0, n1 in zip(bounds, bounds[1:])]).double()
    own = torch.div(pos, b, rounding_mode="floor")
    blocks = float((own + 1).sum()) * g  # causal (token, group, block) triples
    size = DTYPES[case["dtype"]].itemsize
    op = case["op"]
    flops = moved = 0.0
    if op in ("select", "score", "layer"):
        di = case["di"]
        index = total * (g + 1) * di * size
        flops += 2.0 * di * g * float((pos + 1).sum())
        moved += index
        if op != "layer":
            moved += blocks * 4
        if op == "score":  # one winner row each way per block score; gradients of the scores and the inputs
            flops += 4.0 * di * blocks
            moved += blocks * 4 + index
    if op == "topk":
        moved += blocks * 4
    if "topk" in case and op != "score":
        moved += total * g * case["topk"] * 4
    if op in ("train", "prefill", "layer"):
        keys = g * float((pos % b + 1 + b * (torch.clamp(own + 1, max=case["topk"]) - 1)).sum())
        d, hq = case["d"], case["hq"]
        qkv = total * (hq + 2 * g) * d * size
        flops += keys * (hq // g) * 4.0 * d
        moved += qkv + total * hq * d * size
        if op != "prefill":
            flops += keys * (hq // g) * 10.0 * d
            moved += qkv + total * hq * d * size
        if op == "layer":
            flops += keys * (2.0 * d * (hq // g) + 6.0 * case["di"])
            moved += total * (g + 1) * case["di"] * size + total * hq * 4
    return {"bytes": moved, "flops": flops}


def tolerance(case):
    # Scores and selections are defined bit for bit (the exact winning dot, rounded once).
    if case["op"] in ("topk", "select"):
        return "exact"
    # Four times the distance from the float64 result, which is the rounding of the outputs themselves:
    # 2^-9 (bf16), 2^-12 (fp16) and 2^-25 (fp32) of a value, over sqrt(3).
    return {"bf16": {"rel": 7e-3, "max": 3e-2}, "fp16": {"rel": 9e-4, "max": 4e-3},
            "fp32": {"rel": 2e-7, "max": 4e-6}}[case["dtype"]]


# ---------------------------------------------------------------------------- float64


def _exact_scores(case, x, want_grad):
    """Block maxima [T, G, NB] in float64; with `want_grad` also dq and dk (the gradient goes to the winning key)."""
    bounds, b, g = _bounds(case), case["block"], case["g"]
    nb = _max_blocks(case)
    iq, ik = x["iq"].double(), x["ik"][:, 0].double()
    out = torch.full((bounds[-1], g, nb), float("-inf"), dtype=torch.float64, device=DEVICE)
    dq = torch.zeros_like(iq) if want_grad else None
    dk = torch.zeros_like(ik) if want_grad else None
    for n0, n1 in zip(bounds, bounds[1:]):
        step = max(1, (1 << 27) // max(1, (n1 - n0) * g))
        for t0 in range(n0, n1, step):
            t1 = min(n1, t0 + step)
            last = (t1 - 1 - n0) // b + 1
            keys = min(n1 - n0, last * b)
            s = iq[t0:t1].reshape(-1, iq.shape[2]) @ ik[n0:n0 + keys].T
            s = s.view(t1 - t0, g, keys)
            future = torch.arange(n0, n0 + keys, device=DEVICE)[None] > torch.arange(t0, t1, device=DEVICE)[:, None]
            s.masked_fill_(future[:, None], float("-inf"))
            s = torch.nn.functional.pad(s, (0, last * b - keys), value=float("-inf"))
            m, at = s.view(t1 - t0, g, last, b).max(dim=3)
            out[t0:t1, :, :last] = m
            if want_grad:
                w = torch.zeros_like(s).view(t1 - t0, g, last, b)
                w.scatter_(3, at[..., None], x["ds"][t0:t1, :, :last, None].double())
                w = w.view(t1 - t0, g, last * b)[:, :, :keys].reshape(-1, keys)
                dq[t0:t1] = (w @ ik[n0:n0 + keys]).view(t1 - t0, g, -1)
                dk[n0:n0 + keys] += w.T @ iq[t0:t1].reshape(-1, iq.shape[2])
    return out, dq, dk[:, None] if want_grad else None


def _exact_attention(case, x, ids):
    """Dense masked attention in float64, with the gradients and the KL terms that the case returns."""
    bounds, b, g, r = _bounds(case), case["block"], case["g"], case["hq"] // case["g"]
    q, k, v = (x[n].detach().double() for n in ("q", "k", "v"))
    d = q.shape[2]
    total = bounds[-1]
    train, layer = "dout" in x, case["op"] == "layer"
    out = torch.zeros_like(q)
    lse = torch.zeros(total, case["hq"], dtype=torch.float64, device=DEVICE)
    dout = x["dout"].double() if train else None
    dq, dk, dv = (torch.zeros_like(z) if train else None for z in (q, k, v))
    if layer:
        iq, ik = x["iq"].detach().double(), x["ik"].detach()[:, 0].double()
        diq, dik, kl = torch.zeros_like(iq), torch.zeros_like(ik), 0.0
        si = case["di"] ** -0.5
    for n0, n1 in zip(bounds, bounds[1:]):
        step = max(1, (1 << 26) // max(1, (n1 - n0) * r))
        for t0 in range(n0, n1, step):
            t1 = min(n1, t0 + step)
            c, keys = t1 - t0, t1 - n0
            nb = -(-keys // b)
            causal = torch.arange(n0, t1, device=DEVICE)[None] <= torch.arange(t0, t1, device=DEVICE)[:, None]
            for h in range(g):
                sel = torch.zeros(c, nb + 1, dtype=torch.bool, device=DEVICE)
                at = ids[t0:t1, h].long()
                sel.scatter_(1, torch.where(at < 0, nb, at), True)
                seen = sel[:, :nb].repeat_interleave(b, dim=1)[:, :keys] & causal
                heads = slice(h * r, h * r + r)
                qc, kc, vc = q[t0:t1, heads].reshape(-1, d), k[n0:t1, h], v[n0:t1, h]
                s = (qc @ kc.T * d ** -0.5).view(c, r, keys).masked_fill_(~seen[:, None], float("-inf"))
                lse[t0:t1, heads] = torch.logsumexp(s, dim=2)
                p = torch.softmax(s, dim=2)
                o = p.view(-1, keys) @ vc
                out[t0:t1, heads] = o.view(c, r, d)
                if train:
                    do = dout[t0:t1, heads].reshape(-1, d)
                    dp = do @ vc.T - (do * o).sum(1, keepdim=True)
                    dp = dp.mul_(p.view(-1, keys)).mul_(d ** -0.5)
                    dq[t0:t1, heads] = (dp @ kc).view(c, r, d)
                    dk[n0:t1, h] += dp.T @ qc
                    dv[n0:t1, h] += p.view(-1, keys).T @ do
                if layer:
                    teacher = p.mean(dim=1)
                    z = (iq[t0:t1, h] @ ik[n0:t1].T * si).masked_fill_(~seen, float("-inf"))
                    logs = torch.log_softmax(z, dim=1).masked_fill_(~seen, 0.0)
                    kl += float((torch.xlogy(teacher, teacher) - teacher * logs).sum())
                    dz = (torch.softmax(z, dim=1) - teacher) * si * KL_WEIGHT
                    diq[t0:t1, h] = dz @ ik[n0:t1]
                    dik[n0:t1] += dz.T @ iq[t0:t1, h]
    if layer:
        kl = torch.tensor(kl / (total * g), dtype=torch.float64, device=DEVICE)
        return out, lse, kl, dq, dk, dv, diq, dik[:, None]
    return (out, dq, dk, dv) if train else out


def exact(case, seed):
    if case["op"] == "topk":
        return None  # no computed numbers
    x = _inputs(case, seed)
    if case["op"] == "select":
        return _exact_scores(case, x, False)[0], None
    if case["op"] == "score":
        return _exact_scores(case, x, True)
    if case["op"] == "layer":
        ids = _selection(case, _exact_scores(case, x, False)[0].float())
    else:
        ids = x["ids"]
    return _exact_attention(case, x, ids)
