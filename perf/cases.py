"""Performance cases of the attention path.

Each case is one call of the module as an inference server or a training
program makes it, over the sizes the module is used at: single-token decode
against every cache layout, prefill of short and long prompts, packed and
padded, training steps in both precisions, and speculative verification.
``listed()`` are the fixed cases, ``draw()`` gives others of the same ranges.
"""
from __future__ import annotations

import math

import torch

import flash_attn_autograd
import flash_attn_v100 as fa

PAGE = 16  # tokens per page of the paged cache
HALF = torch.float16


def listed():
    return [
        # a short padded prompt on a small model: launch and latency bound
        {"name": "prefill_short", "kind": "prefill", "B": 2, "HQ": 8, "HKV": 8, "N": 256, "D": 64, "causal": True},
        # bidirectional attention over padded sequences with an 80-wide head
        # and a ragged length (an encoder tower)
        {"name": "encode_d80", "kind": "prefill", "B": 8, "HQ": 16, "HKV": 16, "N": 577, "D": 80, "causal": False},
        # one long prompt with grouped KV heads: the largest prefill
        {"name": "prefill_long_gqa", "kind": "prefill", "B": 1, "HQ": 32, "HKV": 8, "N": 8192, "D": 128,
         "causal": True},
        # a server's prefill step: prompts of mixed lengths packed together
        {"name": "prefill_varlen", "kind": "varlen", "B": 16, "H": 32, "lo": 128, "hi": 2048, "D": 128,
         "causal": True, "mix": 0},
        # interactive decode: one sequence, one token
        {"name": "decode_single", "kind": "decode", "B": 1, "HQ": 32, "HKV": 8, "N": 4097, "D": 128,
         "cache_len": 4096},
        # a decode step of a batch whose sequences have reached different lengths
        {"name": "decode_continuous", "kind": "continuous", "B": 64, "HQ": 32, "HKV": 8, "N": 8193, "D": 128,
         "lo": 16, "mix": 0},
        # the same against a paged cache with scattered pages
        {"name": "decode_paged", "kind": "paged", "B": 128, "HQ": 32, "HKV": 8, "hi": 4096, "D": 128, "lo": 64,
         "mix": 0},
        # decode against an INT8 cache with per-token scales
        {"name": "decode_int8_cache", "kind": "int8_cache", "B": 16, "HQ": 32, "HKV": 8, "N": 2049, "D": 128,
         "cache_len": 2048},
        # long-context decode that attends a window and a sink of the cache
        {"name": "decode_window", "kind": "window", "B": 16, "HQ": 32, "HKV": 8, "N": 8193, "D": 128,
         "cache_len": 8000, "window": 2048, "sink": 64},
        # one attention layer of a training step in half precision
        {"name": "train_fp16", "kind": "train", "dtype": "float16", "B": 4, "H": 16, "N": 2048, "D": 128,
         "causal": True},
        # the same in single precision, at a ragged length and narrow heads
        {"name": "train_fp32", "kind": "train", "dtype": "float32", "B": 2, "H": 16, "N": 1000, "D": 64,
         "causal": True},
        # acceptance of drafted tokens over a whole vocabulary
        {"name": "verify_draft", "kind": "verify", "B": 16, "K": 4, "V": 32000},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["prefill", "prefill", "varlen", "decode", "continuous", "paged", "int8_cache", "int8",
                       "window", "train", "train", "verify"])
    hq, hkv = rng.choice([(8, 8), (16, 16), (32, 8), (32, 8), (32, 4), (64, 8), (32, 32)])
    d = rng.choice([64, 80, 96, 128, 128, 128, 256])
    if kind in ("prefill", "varlen"):
        # vector-aligned power-of-two heads run at several times the rate of the others
        budget = 2.5e11 if d in (64, 128) else 4e10
        if kind == "prefill":
            n = _log_int(rng, 64, 8192)
            causal = rng.random() < 0.7
            per_seq = 4.0 * hq * d * n * n * (0.5 if causal else 1.0)
            b = max(1, min(_log_int(rng, 1, 16), int(budget / per_seq)))
            while hq > 8 and per_seq > budget:
                hq, hkv, per_seq = hq // 2, max(1, hkv // 2), per_seq / 2
            if per_seq > budget:
                n = int(n * math.sqrt(budget / per_seq))
            return {"kind": kind, "B": b, "HQ": hq, "HKV": hkv, "N": n, "D": d, "causal": causal}
        hi = _log_int(rng, 256, 2048)
        lo = rng.randint(1, hi // 2)
        per_seq = 2.0 * hq * d * hi * hi
        b = max(1, min(_log_int(rng, 2, 32), int(budget / per_seq)))
        return {"kind": kind, "B": b, "H": hq, "lo": lo, "hi": hi, "D": d, "causal": rng.random() < 0.8,
                "mix": rng.randint(1, 999)}
    if kind in ("decode", "int8_cache", "int8", "window", "continuous", "paged"):
        n = _log_int(rng, 128, 32768)
        # at most about 0.25 GB of attended cache (the listed large ones hold four times that)
        budget = 2.5e8 if d in (64, 128, 256) else 1e8
        b = max(1, min(_log_int(rng, 1, 128), int(budget / (4.0 * hkv * n * d))))
        if kind == "continuous":
            return {"kind": kind, "B": b, "HQ": hq, "HKV": hkv, "N": n, "D": d, "lo": min(16, n // 4),
                    "mix": rng.randint(1, 999)}
        if kind == "paged":
            return {"kind": kind, "B": b, "HQ": hq, "HKV": hkv, "hi": n, "D": d, "lo": max(1, n // 64),
                    "mix": rng.randint(1, 999)}
        case = {"kind": kind, "B": b, "HQ": hq, "HKV": hkv, "N": n, "D": d,
                "cache_len": n - 1 if rng.random() < 0.5 else rng.randint(n // 2, n - 1)}
        if kind == "window":
            case["window"] = rng.randint(max(1, n // 16), n)
            case["sink"] = rng.randint(0, min(64, n // 8))
        return case
    if kind == "train":
        dtype = rng.choice(["float16", "float16", "float32"])
        d = rng.choice([64, 64, 80, 128, 128])
        n = _log_int(rng, 64, 2048)
        h = rng.choice([8, 12, 16, 32])
        budget = (3e10 if d in (64, 128) else 5e9) * (1.0 if dtype == "float16" else 0.25)
        b = max(1, min(_log_int(rng, 1, 8), int(budget / (2.0 * h * d * n * n))))
        return {"kind": kind, "dtype": dtype, "B": b, "H": h, "N": n, "D": d, "causal": rng.random() < 0.8}
    return {"kind": "verify", "B": _log_int(rng, 1, 32), "K": rng.randint(1, 8), "V": _log_int(rng, 4096, 90000)}


def _lengths(case):
    """Sequence lengths of a ragged batch, uniform in [lo, hi] with the longest
    one always there; ``mix`` says which batch composition."""
    g = torch.Generator().manual_seed(case["mix"])
    hi = case["hi"] if "hi" in case else case["N"] - 1
    lens = torch.randint(case["lo"], hi + 1, (case["B"],), generator=g)
    lens[case["B"] // 2] = hi
    return lens


def prepare(case, seed):
    dev = torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(seed)

    def randn(*shape, dtype=HALF):
        return torch.randn(*shape, generator=g, device=dev, dtype=dtype)

    kind, b, d = case["kind"], case["B"], case.get("D")
    st = {"case": case}
    if kind == "prefill":
        st["q"] = randn(b, case["HQ"], case["N"], d)
        st["k"] = randn(b, case["HKV"], case["N"], d)
        st["v"] = randn(b, case["HKV"], case["N"], d)
    elif kind == "varlen":
        lens = _lengths(case)
        cu = torch.zeros(b + 1, dtype=torch.int32)
        cu[1:] = torch.cumsum(lens, 0)
        total = int(cu[-1])
        st["q"], st["k"], st["v"] = (randn(total, case["H"], d) for _ in range(3))
        st["cu"], st["max_seqlen"] = cu.to(dev), int(lens.max())
    elif kind in ("decode", "window", "continuous", "int8"):
        st["q"] = randn(b, case["HQ"], 1, d)
        st["k"] = randn(b, case["HKV"], case["N"], d)
        st["v"] = randn(b, case["HKV"], case["N"], d)
        if kind == "continuous":
            st["lens"] = _lengths(case).to(torch.int32).to(dev)
        if kind == "int8":
            st["q_scale"] = st["q"].float().abs().amax((2, 3)) / 127.0
            k_scale = st["k"].abs().amax((2, 3)).float() / 127.0
            # one scale per head; the kernel reads the first B * HKV values of this tensor
            flat = torch.ones(b * case["HKV"] * case["N"], device=dev)
            flat[:b * case["HKV"]] = k_scale.reshape(-1)
            st["k_scale"] = flat.view(b, case["HKV"], case["N"])
    elif kind == "paged":
        lens = _lengths(case)
        blocks = (case["hi"] + PAGE - 1) // PAGE
        pages = b * blocks
        st["q"] = randn(b, case["HQ"], 1, d)
        st["k"] = randn(pages, case["HKV"], PAGE, d)
        st["v"] = randn(pages, case["HKV"], PAGE, d)
        perm = torch.randperm(pages, generator=torch.Generator().manual_seed(seed))
        st["table"] = perm.to(torch.int32).view(b, blocks).to(dev)
        st["lens"], st["blocks"] = lens.to(torch.int32).to(dev), blocks
    elif kind == "int8_cache":
        st["q"] = randn(b, case["HQ"], 1, d)
        for t in ("k", "v"):
            x = randn(b, case["HKV"], case["N"], d)
            scale = (x.abs().amax(-1).float() / 127.0).half()
            st[t] = torch.clamp(torch.round(x.float() / scale.float()[..., None]), -127, 127).to(torch.int8)
            st[t + "_scale"] = scale
    elif kind == "train":
        dtype = getattr(torch, case["dtype"])
        shape = (b, case["H"], case["N"], d)
        for t in ("q", "k", "v"):
            st[t] = randn(*shape, dtype=dtype).requires_grad_()
        st["dout"] = randn(*shape, dtype=dtype)
    else:  # verify: a draft model's distributions near the target's, its sampled tokens
        k, vocab = case["K"], case["V"]
        logits = 2.5 * randn(b, k + 1, vocab, dtype=torch.float32)
        st["target"] = torch.softmax(logits, -1)
        near = logits[:, :k] + 1.0 * randn(b, k, vocab, dtype=torch.float32)
        st["draft"] = torch.softmax(near, -1)
        st["tokens"] = torch.multinomial(st["draft"].view(b * k, vocab), 1, generator=g).view(b, k)
        st["rand"] = torch.rand(b, k, generator=g, device=dev)
    return st


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "prefill":
        if case["HQ"] == case["HKV"]:
            return fa.forward_fp16(st["q"], st["k"], st["v"], case["causal"])
        return fa.forward_prefill_gqa_fp16(st["q"], st["k"], st["v"], case["causal"])
    if kind == "varlen":
        return fa.forward_varlen_prefill_fp16(st["q"], st["k"], st["v"], st["cu"], st["max_seqlen"], case["causal"])
    if kind == "decode":
        return fa.forward_decode_gqa_fp16(st["q"], st["k"], st["v"], True, case["cache_len"])
    if kind == "window":
        return fa.forward_decode_sliding_window_gqa(st["q"], st["k"], st["v"], True, case["cache_len"],
                                                    case["window"], case["sink"])
    if kind == "continuous":
        return fa.forward_continuous_batching_fp16(st["q"], st["k"], st["v"], st["lens"], True)
    if kind == "paged":
        return fa.forward_paged_decode_gqa_fp16(st["q"], st["k"], st["v"], st["table"], st["lens"], st["blocks"])
    if kind == "int8":
        return fa.forward_decode_int8_gqa(st["q"], st["k"], st["v"], st["q_scale"], st["k_scale"], case["cache_len"])
    if kind == "int8_cache":
        return fa.forward_decode_int8_kv_cache_gqa(st["q"], st["k"], st["v"], st["k_scale"], st["v_scale"],
                                                   case["cache_len"])
    if kind == "train":
        out = flash_attn_autograd.flash_attn(st["q"], st["k"], st["v"], case["causal"])
        dq, dk, dv = torch.autograd.grad(out, (st["q"], st["k"], st["v"]), st["dout"])
        return {"out": out.detach(), "dq": dq, "dk": dk, "dv": dv}
    accepted, tokens = fa.speculative_verify(st["target"], st["draft"], st["tokens"], st["rand"],
                                             case["K"])
    return {"accepted": accepted, "tokens": tokens}


def _window_rows(case):
    """Attended rows of a sliding-window call: the sink, then the window."""
    n, last = case["N"], case["cache_len"]
    start = max(0, min(last + 1, n) - case["window"])
    sink = min(case["sink"], n)
    return sink, max(start, sink), min(last, n - 1) + 1


def work(case):
    kind, b, d = case["kind"], case["B"], case.get("D")
    if kind == "prefill":
        pairs = case["N"] * (case["N"] + 1) / 2 if case["causal"] else case["N"] ** 2
        return {"bytes": 2.0 * b * case["N"] * d * (2 * case["HQ"] + 2 * case["HKV"]),
                "flops": 4.0 * b * case["HQ"] * d * pairs}
    if kind == "varlen":
        lens = _lengths(case).tolist()
        pairs = sum(n * (n + 1) / 2 if case["causal"] else n * n for n in lens)
        return {"bytes": 2.0 * 4 * sum(lens) * case["H"] * d, "flops": 4.0 * case["H"] * d * pairs}
    if kind == "train":
        pairs = case["N"] * (case["N"] + 1) / 2 if case["causal"] else case["N"] ** 2
        size = 2 if case["dtype"] == "float16" else 4
        # forward: q, k, v in, out; backward: dout, q, k, v, out in, dq, dk, dv out.
        # Two products forward, five backward.
        return {"bytes": 12.0 * size * b * case["H"] * case["N"] * d,
                "flops": 14.0 * b * case["H"] * d * pairs}
    if kind == "verify":
        # the row's drafted probabilities, one residual (target and draft) and one bonus row
        return {"bytes": 4.0 * b * 3 * case["V"], "flops": 4.0 * b * case["V"]}
    if kind in ("continuous", "paged"):
        keys = float(_lengths(case).sum()) / b + (kind == "continuous")
    elif kind == "window":
        sink, start, end = _window_rows(case)
        keys = sink + max(0, end - start)
    else:
        keys = case["cache_len"] + 1
    row = 2.0 * (d + 2) if kind == "int8_cache" else 4.0 * d
    return {"bytes": b * case["HKV"] * keys * row + 4.0 * b * case["HQ"] * d,
            "flops": 4.0 * b * case["HQ"] * keys * d}


def tolerance(case):
    kind = case["kind"]
    if kind == "verify":
        return "exact"
    if kind == "train":
        # measured against exact(): 3.1e-4 in half precision, 8e-7 in single
        return {"rel": 1.3e-3} if case["dtype"] == "float16" else {"rel": 4e-6}
    return {"rel": 1.2e-3}  # measured 2.4e-4 to 2.9e-4: half-precision probabilities and output


def _attend(q, k, v, causal=False):
    """softmax(q k^T / sqrt(D)) v of one head in 64 bits."""
    s = q.double() @ k.double().t() / math.sqrt(q.shape[-1])
    if causal:
        n = s.shape[-1]
        s.masked_fill_(torch.ones(n, n, dtype=torch.bool, device=s.device).triu_(1), -math.inf)
    return torch.softmax(s, -1) @ v.double()


def _exact_train(st, case):
    outs = {n: [] for n in ("out", "dq", "dk", "dv")}
    scale = 1.0 / math.sqrt(case["D"])
    mask = None
    if case["causal"]:
        mask = torch.ones(case["N"], case["N"], dtype=torch.bool, device=st["q"].device).triu_(1)
    flat = {t: st[t].detach().flatten(0, 1) for t in ("q", "k", "v", "dout")}
    for i in range(case["B"] * case["H"]):
        q, k, v, do = (flat[t][i].double() for t in ("q", "k", "v", "dout"))
        s = q @ k.t() * scale
        if mask is not None:
            s.masked_fill_(mask, -math.inf)
        p = torch.softmax(s, -1)
        o = p @ v
        ds = p * (do @ v.t() - (do * o).sum(-1, keepdim=True)) * scale
        for name, x in (("out", o), ("dq", ds @ k), ("dk", ds.t() @ q), ("dv", p.t() @ do)):
            outs[name].append(x)
    shape = st["q"].shape
    return {n: torch.stack(x).view(shape) for n, x in outs.items()}


def exact(case, seed):
    kind = case["kind"]
    if kind == "verify":
        return None
    st = prepare(case, seed)
    if kind == "train":
        return _exact_train(st, case)
    if kind == "varlen":
        out = torch.zeros(st["q"].shape, dtype=torch.float64, device=st["q"].device)
        cu = st["cu"].tolist()
        for s, e in zip(cu[:-1], cu[1:]):
            for h in range(case["H"]):
                out[s:e, h] = _attend(st["q"][s:e, h], st["k"][s:e, h], st["v"][s:e, h], case["causal"])
        return out
    q = st["q"]
    out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    group = case["HQ"] // case["HKV"]
    if kind == "prefill":
        for i in range(case["B"]):
            for h in range(case["HQ"]):
                out[i, h] = _attend(q[i, h], st["k"][i, h // group], st["v"][i, h // group], case["causal"])
        return out
    lens = st["lens"].tolist() if "lens" in st else None
    for i in range(case["B"]):
        if kind == "paged":
            ids = st["table"][i, :(lens[i] + PAGE - 1) // PAGE].long()
            k, v = (st[t][ids].transpose(0, 1).reshape(case["HKV"], -1, case["D"])[:, :lens[i]] for t in ("k", "v"))
        elif kind == "window":
            sink, start, end = _window_rows(case)
            rows = torch.cat([torch.arange(sink), torch.arange(start, max(start, end))]).to(q.device)
            k, v = st["k"][i][:, rows], st["v"][i][:, rows]
        else:
            keys = min(case["N"], (lens[i] if lens else case["cache_len"]) + 1)
            k, v = st["k"][i][:, :keys], st["v"][i][:, :keys]
        if kind == "int8_cache":
            k, v = ((st[t][i][:, :keys].float() * st[t + "_scale"][i][:, :keys, None].float()).half()
                    for t in ("k", "v"))
        qi = q[i, :, 0]
        for h in range(case["HKV"]):
            heads = slice(h * group, (h + 1) * group)
            if kind == "int8":
                # the path's own definition: scores from integer codes of q and k
                qs = st["q_scale"][i, heads].double()[:, None]
                ks = st["k_scale"].flatten()[i * case["HKV"] + h].double()
                s = _codes(qi[heads], st["q_scale"][i, heads][:, None]) @ _codes(k[h], ks.float()).t()
                p = torch.softmax(s * qs * ks / math.sqrt(case["D"]), -1)
                out[i, heads, 0] = p @ v[h].double()
            else:
                out[i, heads, 0] = _attend(qi[heads], k[h], v[h])
    return out


def _codes(x, scale):
    """round-half-away(x * (1 / scale)) clamped to +-127, as 64-bit integers' values."""
    y = x.float() * (1.0 / scale.float())
    return torch.clamp(torch.trunc(y + torch.copysign(torch.full_like(y, 0.5), y)), -127, 127).double()
