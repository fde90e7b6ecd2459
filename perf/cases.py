"""What is timed: the operators that a streaming GRPO/OPD program calls, through their public entry points.

A case is a dict of plain values; its ``op`` names one of the entry points below, the rest are sizes and
options.  ``listed()`` holds the named cases, ``draw()`` gives further ones of the same ranges, ``prepare()``
makes what the caller holds before the call, ``run()`` is one pass.  ``exact()`` computes the same outputs in
64 bits from plain torch operations.
"""

from __future__ import annotations

import math

import torch

from thundersync_amd import attention, forest, fused_logprob, fused_lora, rms_norm

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
CHUNK = 512  # tokens of a retained chunk


def listed():
    return [
        # A short turn scored without gradients: a few dozen new tokens over a conversation's retained chunks.
        {"name": "turn_infer", "op": "turn", "rows": 48, "context": 4096, "hq": 32, "hkv": 8, "dim": 128,
         "dtype": "bf16"},
        # One 512-token chunk of a streamed completion with its backward, over 8k tokens of retained chunks.
        {"name": "chunk_grad", "op": "chunk", "rows": 512, "context": 7680, "hq": 32, "hkv": 8, "dim": 128,
         "dtype": "bf16"},
        # One layer's attention of a whole forest: a shared prompt and eight sibling completions.
        {"name": "forest_grad", "op": "forest", "prompt": 2048, "siblings": 8, "low": 256, "high": 4096, "hq": 32,
         "hkv": 8, "dim": 128, "dtype": "bf16"},
        # One layer's attention of a pack of turns, each over the shared prompt and its own earlier chunk, with the
        # heads of a larger decoder (five query heads on each KV head).
        {"name": "pack_grad", "op": "pack", "prompt": 1500, "segments": 6, "low": 200, "high": 1500, "hq": 40,
         "hkv": 8, "dim": 128, "dtype": "bf16"},
        # A long tail over its prefix at head dim 256, six query heads on each KV head.
        {"name": "branch_grad", "op": "turn_grad", "rows": 9288, "context": 3000, "hq": 24, "hkv": 4, "dim": 256,
         "dtype": "bf16"},
        # A cohort of independent sequences of a small decoder (head dim 64) in half precision.
        {"name": "ragged_d64", "op": "ragged", "segments": 8, "low": 128, "high": 2048, "context": 512, "hq": 16,
         "hkv": 8, "dim": 64, "dtype": "fp16"},
        # The head over a whole batch's scored tokens: logprob and entropy, gradient to the hidden states.
        {"name": "head_gated", "op": "head", "rows": 11469, "hidden": 4096, "vocab": 151936, "entropy": True,
         "train": False, "dtype": "bf16"},
        # The head over one streamed turn: predictors gathered from the chunk, frozen weight.
        {"name": "head_turn", "op": "head_turn", "rows": 400, "hidden": 4096, "vocab": 151936, "dtype": "bf16"},
        # A trainable head: hidden and weight gradients of a medium batch of a smaller decoder.
        {"name": "head_train", "op": "head", "rows": 4096, "hidden": 2048, "vocab": 151936, "entropy": False,
         "train": True, "dtype": "bf16"},
        # The head at fp32, trainable, as small single-precision runs have it.
        {"name": "head_fp32", "op": "head", "rows": 2048, "hidden": 1024, "vocab": 32000, "entropy": True,
         "train": True, "dtype": "fp32"},
        # A decoder's norm over a batch of tokens, forward and backward.
        {"name": "norm_grad", "op": "norm", "rows": 16384, "width": 4096, "dtype": "bf16"},
        # A query projection with a merged adapter, forward and backward.
        {"name": "lora_grad", "op": "lora", "rows": 16384, "inp": 4096, "out": 4096, "rank": 16, "dtype": "bf16"},
    ]


def _log_int(rng, low, high):
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


HEADS_128 = ((32, 8), (16, 8), (40, 8))


def draw(rng):
    op = rng.choice(("turn", "chunk", "forest", "pack", "turn_grad", "ragged", "head", "head_turn", "head_train",
                     "head_fp32", "norm", "lora"))
    heads = rng.choice(((128, *rng.choice(HEADS_128)),) * 3 + ((256, 24, 4),))
    dims = {"dim": heads[0], "hq": heads[1], "hkv": heads[2], "dtype": "bf16"}
    if op == "turn":
        return {"op": op, "rows": _log_int(rng, 1, 512), "context": _log_int(rng, 256, 32768), **dims}
    if op == "chunk":
        return {"op": op, "rows": _log_int(rng, 16, 1024), "context": _log_int(rng, 256, 14336), **dims}
    if op == "forest":
        low = _log_int(rng, 32, 512)
        return {"op": op, "prompt": _log_int(rng, 128, 4096), "siblings": rng.randint(2, 8), "low": low,
                "high": _log_int(rng, 2 * low, 4096), **dims}
    if op == "pack":
        low = _log_int(rng, 16, 512)
        return {"op": op, "prompt": _log_int(rng, 64, 4096), "segments": rng.randint(2, 8), "low": low,
                "high": _log_int(rng, 2 * low, 2048), **dims}
    if op == "turn_grad":
        return {"op": op, "rows": _log_int(rng, 256, 9288), "context": _log_int(rng, 64, 8192), **dims}
    if op == "ragged":
        low = _log_int(rng, 16, 512)
        hq, hkv = rng.choice(((16, 8), (32, 8), (24, 4)))
        return {"op": op, "segments": rng.randint(2, 8), "low": low, "high": _log_int(rng, 2 * low, 2048),
                "context": _log_int(rng, 16, 1024), "hq": hq, "hkv": hkv, "dim": rng.choice((32, 64, 64, 64, 96, 192)),
                "dtype": rng.choice(("bf16", "fp16"))}
    if op in ("head", "head_train"):
        train = op == "head_train"
        return {"op": "head", "rows": _log_int(rng, 16, 4096 if train else 11469),
                "hidden": rng.choice((1024, 2048) if train else (1024, 2048, 4096)),
                "vocab": rng.choice((32000, 50257, 151936)), "entropy": rng.random() < 0.5, "train": train,
                "dtype": rng.choice(("bf16", "bf16", "bf16", "fp16"))}
    if op == "head_turn":
        return {"op": op, "rows": _log_int(rng, 8, 2048), "hidden": rng.choice((1024, 2048, 4096)),
                "vocab": rng.choice((32000, 50257, 151936)), "dtype": "bf16"}
    if op == "head_fp32":
        return {"op": "head", "rows": _log_int(rng, 64, 2048), "hidden": rng.choice((128, 512, 1000, 1024)),
                "vocab": rng.choice((1024, 8191, 32000)), "entropy": rng.random() < 0.5, "train": rng.random() < 0.5,
                "dtype": "fp32"}
    if op == "norm":
        width = rng.choice((128, 1024, 2048, 4096, 5120))
        return {"op": op, "rows": _log_int(rng, 16, min(262144, (1 << 26) // width)), "width": width,
                "dtype": rng.choice(("bf16", "bf16", "fp16"))}
    return {"op": op, "rows": _log_int(rng, 64, 16384), "inp": rng.choice((1024, 2048, 4096)),
            "out": rng.choice((1024, 2048, 4096)), "rank": rng.choice((8, 16, 32, 64)), "dtype": "bf16"}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _generators(seed):
    return torch.Generator().manual_seed(seed), torch.Generator(device="cuda").manual_seed(seed)


def _normal(g, *shape, dtype, scale=1.0):
    t = torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32)
    return (t * scale if scale != 1.0 else t).to(dtype)


def _chunk_rows(total):
    return [min(CHUNK, total - i) for i in range(0, total, CHUNK)]


def _sizes(case):
    """Sequence lengths of a case with several sequences.  They are part of the case, the same for every seed."""
    g = torch.Generator().manual_seed(1009 * case.get("segments", case.get("siblings", 0)) + case["low"])
    n = case["segments"] if "segments" in case else case["siblings"]
    return torch.randint(case["low"], case["high"] + 1, (n,), generator=g).tolist()


def prepare(case, seed):
    op, dt = case["op"], DTYPES[case["dtype"]]
    gc, g = _generators(seed)
    s = {"case": case}
    if op in ("turn", "turn_grad", "chunk"):
        hq, hkv, d, t = case["hq"], case["hkv"], case["dim"], case["rows"]
        # the engine keeps the context as retained chunks; the tail of a branch is one tensor with its prefix
        rows = [case["context"] + t] if op == "turn_grad" else [*_chunk_rows(case["context"]), t]
        grad = op != "turn"
        s["q"] = _normal(g, 1, t, hq, d, dtype=dt).transpose(1, 2).requires_grad_(grad)
        s["ks"] = [_normal(g, n, hkv, d, dtype=dt).requires_grad_(grad) for n in rows]
        s["vs"] = [_normal(g, n, hkv, d, dtype=dt).requires_grad_(grad) for n in rows]
        if grad:
            s["dout"] = _normal(g, 1, t, hq, d, dtype=dt).transpose(1, 2)
    elif op == "forest":
        hq, hkv, d = case["hq"], case["hkv"], case["dim"]
        prompt = torch.randint(0, 100000, (case["prompt"],), generator=gc).tolist()
        trajs = []
        for i, n in enumerate(_sizes(case)):
            body = [100000 + i] + torch.randint(0, 100000, (n - 1,), generator=gc).tolist()
            trajs.append(forest.Trajectory([forest.Segment.prompt(prompt), forest.Segment.action(body)],
                                           group_id=0, traj_id=i))
        s["plan"] = forest.compile_plan(forest.build_forest(trajs))
        p = s["plan"].n_physical
        s["q"] = _normal(g, p, hq, d, dtype=dt).requires_grad_()
        s["k"] = _normal(g, p, hkv, d, dtype=dt).requires_grad_()
        s["v"] = _normal(g, p, hkv, d, dtype=dt).requires_grad_()
        s["dout"] = _normal(g, p, hq, d, dtype=dt)
    elif op == "pack":
        hq, hkv, d = case["hq"], case["hkv"], case["dim"]
        lengths = _sizes(case)
        total = sum(lengths)
        s["q"] = _normal(g, 1, total, hq, d, dtype=dt).transpose(1, 2).requires_grad_()
        s["k"] = _normal(g, total, hkv, d, dtype=dt).requires_grad_()
        s["v"] = _normal(g, total, hkv, d, dtype=dt).requires_grad_()
        prompt = tuple(_normal(g, case["prompt"], hkv, d, dtype=dt).requires_grad_() for _ in range(2))
        # every second turn has an earlier turn of its own between the prompt and itself
        own = [tuple(_normal(g, n, hkv, d, dtype=dt).requires_grad_() for _ in range(2)) if i % 2 else None
               for i, n in enumerate(reversed(lengths))]
        s["ancestors"] = [([prompt[0], *([o[0]] if o else [])], [prompt[1], *([o[1]] if o else [])]) for o in own]
        s["leaves"] = [*prompt, *(t for o in own if o for t in o)]
        s["layout"] = attention.pack_layout(lengths, s["ancestors"], "cuda")
        s["inputs"] = s["layout"].inputs(s["ancestors"])
        s["dout"] = _normal(g, 1, total, hq, d, dtype=dt).transpose(1, 2)
    elif op == "ragged":
        hq, hkv, d = case["hq"], case["hkv"], case["dim"]
        lengths = _sizes(case)
        keys = [n + (case["context"] if i % 2 else 0) for i, n in enumerate(lengths)]
        s["qs"] = [_normal(g, 1, n, hq, d, dtype=dt).transpose(1, 2).requires_grad_() for n in lengths]
        s["ks"] = [_normal(g, n, hkv, d, dtype=dt).requires_grad_() for n in keys]
        s["vs"] = [_normal(g, n, hkv, d, dtype=dt).requires_grad_() for n in keys]
        s["douts"] = [_normal(g, 1, n, hq, d, dtype=dt).transpose(1, 2) for n in lengths]
    elif op in ("head", "head_turn"):
        n, d, v = case["rows"], case["hidden"], case["vocab"]
        s["weight"] = _normal(g, v, d, dtype=dt, scale=0.02).requires_grad_(case.get("train", False))
        s["hidden"] = _normal(g, n, d, dtype=dt).requires_grad_()
        if op == "head":
            s["target"] = torch.randint(0, v, (n,), generator=g, device="cuda")
            s["adv"] = torch.randn(n, generator=g, device="cuda")
        else:
            s["boundary"] = _normal(g, d, dtype=dt).requires_grad_()
            s["tokens"] = torch.randint(0, v, (n,), generator=gc).tolist()
            scored = torch.rand(n, generator=torch.Generator().manual_seed(n)) < 0.7
            scored[0] = True
            s["scored"] = scored.tolist()
            s["adv"] = torch.randn(int(scored.sum()), generator=g, device="cuda")
    elif op == "norm":
        s["x"] = _normal(g, case["rows"], case["width"], dtype=dt).requires_grad_()
        s["w"] = torch.linspace(0.4, 3.0, case["width"], device="cuda").to(dt).requires_grad_()
        s["dy"] = _normal(g, case["rows"], case["width"], dtype=dt)
    elif op == "lora":
        n, i, o, r = case["rows"], case["inp"], case["out"], case["rank"]
        s["x"] = _normal(g, n, i, dtype=dt).requires_grad_()
        s["w"] = _normal(g, o, i, dtype=dt, scale=0.02)
        s["a"] = _normal(g, r, i, dtype=torch.float32, scale=0.05).requires_grad_()
        s["b"] = _normal(g, o, r, dtype=torch.float32, scale=0.05).requires_grad_()
        s["dy"] = _normal(g, n, o, dtype=dt)
    else:
        raise ValueError(f"unknown op {op!r}")
    return s


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def _clear(tensors):
    for t in tensors:
        t.grad = None


def run(s):
    case = s["case"]
    op = case["op"]
    if op == "turn":
        with torch.no_grad():
            return {"out": attention.causal_attention(s["q"], s["ks"], s["vs"], case["dim"] ** -0.5)}
    if op in ("turn_grad", "chunk"):
        ks, vs = s["ks"], s["vs"]
        _clear([s["q"], *ks, *vs])
        if op == "chunk":
            out = attention.ChunkedCausalAttention.apply(s["q"], case["dim"] ** -0.5, len(ks), True, "auto", *ks, *vs)
        else:
            out = attention.causal_attention(s["q"], ks, vs, case["dim"] ** -0.5)
        out.backward(s["dout"])
        return {"out": out.detach(), "dq": s["q"].grad, "dk": [k.grad for k in ks], "dv": [v.grad for v in vs]}
    if op == "forest":
        leaves = [s["q"], s["k"], s["v"]]
        _clear(leaves)
        out = attention.forest_attention(s["q"], s["k"], s["v"], s["plan"])
        out.backward(s["dout"])
        return {"out": out.detach(), "grads": [t.grad for t in leaves]}
    if op == "pack":
        leaves = [s["q"], s["k"], s["v"], *s["leaves"]]
        _clear(leaves)
        out = attention.PackedAttention.apply(s["q"], s["k"], s["v"], case["dim"] ** -0.5, s["layout"], *s["inputs"])
        out.backward(s["dout"])
        return {"out": out.detach(), "grads": [t.grad for t in leaves]}
    if op == "ragged":
        leaves = [*s["qs"], *s["ks"], *s["vs"]]
        _clear(leaves)
        outs = attention.ragged_causal_attention(s["qs"], s["ks"], s["vs"], case["dim"] ** -0.5)
        torch.autograd.backward(outs, s["douts"])
        return {"outs": [o.detach() for o in outs], "grads": [t.grad for t in leaves]}
    if op == "head":
        h, w = s["hidden"], s["weight"]
        _clear([h, w])
        if case["entropy"]:
            lp, ent = fused_logprob.fused_logprob_entropy(h, w, s["target"])
        else:
            lp, ent = fused_logprob.fused_logprob(h, w, s["target"]), None
        lp.backward(s["adv"].to(lp.dtype))
        return {"lp": lp.detach(), "ent": None if ent is None else ent.detach(), "dh": h.grad, "dw": w.grad}
    if op == "head_turn":
        _clear([s["hidden"], s["boundary"]])
        lp = fused_logprob.predictor_logprobs(s["boundary"], s["hidden"], s["tokens"], s["scored"], s["weight"])
        lp.backward(s["adv"])
        return {"lp": lp.detach(), "dh": s["hidden"].grad, "db": s["boundary"].grad}
    if op == "norm":
        _clear([s["x"], s["w"]])
        y = rms_norm.FP32RMSNormVJP.apply(s["x"], s["w"], 1e-6)
        y.backward(s["dy"])
        return {"y": y.detach(), "dx": s["x"].grad, "dw": s["w"].grad}
    _clear([s["x"], s["a"], s["b"]])
    y = fused_lora.FusedLoRALinear.apply(s["x"], s["w"], s["a"], s["b"], 2.0)
    y.backward(s["dy"])
    return {"y": y.detach(), "dx": s["x"].grad, "da": s["a"].grad, "db": s["b"].grad}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _segments(case):
    """[(query rows, keys)] of an attention case, and its distinct key rows."""
    op = case["op"]
    if op in ("turn", "turn_grad", "chunk"):
        s = case["context"] + case["rows"]
        return [(case["rows"], s)], s
    lengths = _sizes(case)
    if op == "forest":
        p = case["prompt"]
        return [(p, p), *((n, p + n) for n in lengths)], p + sum(lengths)
    if op == "pack":
        own = [n if i % 2 else 0 for i, n in enumerate(reversed(lengths))]
        return ([(n, case["prompt"] + o + n) for n, o in zip(lengths, own)],
                case["prompt"] + sum(lengths) + sum(own))
    keys = [n + (case["context"] if i % 2 else 0) for i, n in enumerate(lengths)]
    return list(zip(lengths, keys)), sum(keys)


def work(case):
    op = case["op"]
    size = 4 if case["dtype"] == "fp32" else 2
    if op in ("turn", "turn_grad", "chunk", "forest", "pack", "ragged"):
        segs, keys = _segments(case)
        rows = sum(t for t, _ in segs)
        pairs = sum(t * (s - t) + t * (t + 1) // 2 for t, s in segs)
        q, kv = rows * case["hq"] * case["dim"] * size, keys * case["hkv"] * case["dim"] * size
        if op == "turn":  # q, k, v in; out
            return {"bytes": 2 * q + 2 * kv, "flops": 4 * case["dim"] * case["hq"] * pairs}
        # q, k, v, dout in; out, dq, dk, dv
        return {"bytes": 4 * q + 4 * kv, "flops": 14 * case["dim"] * case["hq"] * pairs}
    if op in ("head", "head_turn"):
        n, d, v = case["rows"], case["hidden"], case["vocab"]
        scored = n
        if op == "head_turn":
            picked = torch.rand(n, generator=torch.Generator().manual_seed(n)) < 0.7
            picked[0] = True
            scored = int(picked.sum())
        train = case.get("train", False)
        return {"bytes": size * (2 * n * d + v * d * (2 if train else 1)) + 16 * scored,
                "flops": (8 if train else 6) * scored * v * d}
    if op == "norm":
        return {"bytes": 5 * size * case["rows"] * case["width"], "flops": 12 * case["rows"] * case["width"]}
    n, i, o, r = case["rows"], case["inp"], case["out"], case["rank"]
    return {"bytes": size * (2 * n * i + 2 * n * o + o * i) + 8 * r * (i + o),
            "flops": 4 * n * i * o + 4 * n * r * (i + o)}


def tolerance(case):
    # 16-bit inputs: the outputs, P, dS and dlogits are rounded to the element type (against 64 bits 2.5e-3 in
    # bf16 and 3.2e-4 in fp16); 32 bits: sums over the hidden size and the vocabulary (up to 3.2e-6)
    return {"rel": {"bf16": 1e-2, "fp16": 1.5e-3, "fp32": 1.2e-5}[case["dtype"]]}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------
def _attend(q, k, v, scale, dout=None):
    """One segment, bottom-right causal: q, dout [T, Hq, D], k, v [S, Hkv, D] -> out and, with dout, dq, dk, dv."""
    t, hq, d = q.shape
    s, hkv, _ = k.shape
    group = hq // hkv
    out = torch.empty(t, hq, d, dtype=torch.float64, device=q.device)
    dq = torch.empty_like(out)
    dk = torch.zeros(s, hkv, d, dtype=torch.float64, device=q.device)
    dv = torch.zeros_like(dk)
    block = max(1, (1 << 25) // max(1, s))
    for h in range(hq):
        kh, vh = k[:, h // group].double().contiguous(), v[:, h // group].double().contiguous()
        for r0 in range(0, t, block):
            r1 = min(t, r0 + block)
            seen = s - t + r1  # keys the block's last row sees
            qh = q[r0:r1, h].double().contiguous()
            scores = (qh @ kh[:seen].t().contiguous()) * scale
            last = torch.arange(s - t + r0, s - t + r1, device=q.device)
            scores.masked_fill_(torch.arange(seen, device=q.device)[None, :] > last[:, None], float("-inf"))
            p = torch.softmax(scores, -1)
            del scores
            o = p @ vh[:seen]
            out[r0:r1, h] = o
            if dout is None:
                continue
            g = dout[r0:r1, h].double().contiguous()
            dv[:seen, h // group] += p.t().contiguous() @ g
            ds = p * (g @ vh[:seen].t().contiguous() - (g * o).sum(-1, keepdim=True)) * scale
            dq[r0:r1, h] = ds @ kh[:seen]
            dk[:seen, h // group] += ds.t().contiguous() @ qh
    return out, dq, dk, dv


def _rows(t):
    return t.detach()[0].transpose(0, 1)


def _packed(t):
    return t.transpose(0, 1).unsqueeze(0)


def exact(case, seed):
    s = prepare(case, seed)
    op = case["op"]
    with torch.no_grad():
        if op in ("turn", "turn_grad", "chunk"):
            rows = [k.shape[0] for k in s["ks"]]
            out, dq, dk, dv = _attend(_rows(s["q"]), torch.cat(s["ks"]), torch.cat(s["vs"]), case["dim"] ** -0.5,
                                      _rows(s["dout"]) if "dout" in s else None)
            if op == "turn":
                return {"out": _packed(out)}
            return {"out": _packed(out), "dq": _packed(dq), "dk": list(dk.split(rows)), "dv": list(dv.split(rows))}
        if op == "forest":
            plan = s["plan"]
            grads = [torch.zeros(t.shape, dtype=torch.float64, device="cuda") for t in (s["q"], s["k"], s["v"])]
            out = torch.zeros_like(grads[0])
            for n, (a, b) in enumerate(zip(plan.node_start.tolist(), plan.node_end.tolist())):
                if b <= a:
                    continue
                at = torch.cat([torch.arange(x, y, device="cuda") for x, y in plan.key_ranges[n] if y > x])
                o, dq, dk, dv = _attend(s["q"][a:b], s["k"][at], s["v"][at], case["dim"] ** -0.5, s["dout"][a:b])
                out[a:b], grads[0][a:b] = o, dq
                grads[1][at] += dk
                grads[2][at] += dv
            return {"out": out, "grads": grads}
        if op == "pack":
            q, dout = _rows(s["q"]), _rows(s["dout"])
            leaves = [s["k"], s["v"], *s["leaves"]]
            grad = {id(t): torch.zeros(t.shape, dtype=torch.float64, device="cuda") for t in leaves}
            out = torch.zeros(q.shape, dtype=torch.float64, device="cuda")
            dq = torch.zeros_like(out)
            a = 0
            for n, (ks, vs) in zip(_sizes(case), s["ancestors"]):
                b = a + n
                o, g, dk, dv = _attend(q[a:b], torch.cat([*ks, s["k"][a:b]]), torch.cat([*vs, s["v"][a:b]]),
                                       case["dim"] ** -0.5, dout[a:b])
                out[a:b], dq[a:b] = o, g
                at = 0
                for kc, vc in zip(ks, vs):
                    grad[id(kc)] += dk[at : at + kc.shape[0]]
                    grad[id(vc)] += dv[at : at + vc.shape[0]]
                    at += kc.shape[0]
                grad[id(s["k"])][a:b], grad[id(s["v"])][a:b] = dk[at:], dv[at:]
                a = b
            return {"out": _packed(out), "grads": [_packed(dq), *(grad[id(t)] for t in leaves)]}
        if op == "ragged":
            got = [_attend(_rows(q), k.detach(), v.detach(), case["dim"] ** -0.5, _rows(g))
                   for q, k, v, g in zip(s["qs"], s["ks"], s["vs"], s["douts"])]
            return {"outs": [_packed(x[0]) for x in got],
                    "grads": [*(_packed(x[1]) for x in got), *(x[2] for x in got), *(x[3] for x in got)]}
        if op in ("head", "head_turn"):
            return _exact_head(case, s)
        if op == "norm":
            x, w, dy = s["x"].double(), s["w"].double(), s["dy"].double()
            rstd = torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + 1e-6)
            n, g = x * rstd, dy * w
            return {"y": w * n, "dx": rstd * (g - n * (g * n).mean(-1, keepdim=True)), "dw": (dy * n).sum(0)}
        x, w, dy = s["x"].double(), s["w"].double(), s["dy"].double()
        # the adapters enter the products in the activation dtype
        a, b = (s[n].detach().to(s["x"].dtype).double() for n in ("a", "b"))
        return {"y": x @ w.t().contiguous(), "dx": dy @ w, "da": 2.0 * ((dy @ b).t().contiguous() @ x),
                "db": 2.0 * (dy.t().contiguous() @ (x @ a.t().contiguous()))}


def _exact_head(case, s):
    hidden = s["hidden"].detach()
    if case["op"] == "head_turn":
        at = torch.tensor(s["scored"], device="cuda").nonzero().flatten()
        hidden = torch.cat([s["boundary"].detach()[None], hidden[:-1]])[at]
        target = torch.tensor(s["tokens"], device="cuda")[at]
    else:
        target = s["target"]
    h, w, adv = hidden.double(), s["weight"].detach().double(), s["adv"].double()
    n = h.shape[0]
    lp = torch.empty(n, dtype=torch.float64, device="cuda")
    ent, dh = torch.empty_like(lp), torch.empty_like(h)
    dw = torch.zeros_like(w) if case.get("train") else None
    wt = w.t().contiguous()
    for i in range(0, n, 1024):
        j = min(n, i + 1024)
        logs = torch.log_softmax(h[i:j] @ wt, -1)
        p = logs.exp()
        lp[i:j] = logs.gather(1, target[i:j, None])[:, 0]
        ent[i:j] = -(p * logs).sum(-1)
        dl = -p * adv[i:j, None]
        dl.scatter_add_(1, target[i:j, None], adv[i:j, None])
        dh[i:j] = dl @ w
        if dw is not None:
            dw += dl.t().contiguous() @ h[i:j]
    if case["op"] == "head":
        return {"lp": lp, "ent": ent if case["entropy"] else None, "dh": dh, "dw": dw}
    full = torch.zeros(s["hidden"].shape, dtype=torch.float64, device="cuda")
    full[at[1:] - 1] = dh[1:]
    return {"lp": lp, "dh": full, "db": dh[0]}
