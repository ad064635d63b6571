"""The attention workloads this framework is timed on, each through a public entry point.

A case is a dict of plain values; its ``kind`` names the entry point:

- ``forward``      ``fastest_flash_attn_forward`` on a whole prompt or batch of sequences
- ``cached``       the same with ``kv_cache=``: new queries over a ``ContinuousKVCache``
- ``paged``        ``fastest_flash_paged_decode``: one token per sequence over a page pool
- ``paged_cache``  ``PagedKVCache``: a prompt is appended, all sequences decode, it is freed
- ``mla_decode``   ``fastest_flash_mla_decode`` over a paged latent cache
- ``mla_module``   ``FastestFlashMLA`` in eval mode on a prompt, projections included
- ``train``        ``fastest_flash_attn_func`` and its gradients

``listed`` holds the fixed cases, ``draw`` makes more of the same ranges.
"""

from __future__ import annotations

import math

import numpy as np
import torch

import fastest_flash_attention_amd as ffa

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
ROPE = 64  # rope dims of the MLA paths


def listed():
    return [
        # One short chat prompt on a small GQA model: launch and latency bound.
        dict(name="prefill_short", kind="forward", B=1, Hq=8, Hkv=2, S=197, D=64, dtype="fp16",
             causal=True, window=0, softcap=0.0, radius=0),
        # A batch of full prompts, multi-head attention.
        dict(name="prefill_mha", kind="forward", B=4, Hq=32, Hkv=32, S=4096, D=128, dtype="bf16",
             causal=True, window=0, softcap=0.0, radius=0),
        # LLaMA-style GQA on long prompts with a sliding window and a score softcap.
        dict(name="prefill_gqa_window_softcap", kind="forward", B=2, Hq=32, Hkv=8, S=8192, D=128,
             dtype="bf16", causal=True, window=4096, softcap=50.0, radius=0),
        # Block-sparse attention: a local band of 64 x 64 tiles over a long, ragged document.
        dict(name="prefill_block_local", kind="forward", B=2, Hq=16, Hkv=16, S=8000, D=128,
             dtype="bf16", causal=True, window=0, softcap=0.0, radius=1024),
        # Chunked prefill: the next chunk of one long prompt over the K/V of the ones before.
        dict(name="chunk_over_cache", kind="cached", B=1, Hq=32, Hkv=8, S=509, Sc=7683,
             max_len=8192, D=128, dtype="bf16", window=0, softcap=0.0),
        # Generation with contiguous caches: one new token per sequence.
        dict(name="token_over_cache", kind="cached", B=8, Hq=32, Hkv=8, S=1, Sc=4095,
             max_len=4608, D=128, dtype="bf16", window=0, softcap=0.0),
        # Serving: a decode step of a large batch with mixed context lengths.
        dict(name="paged_decode", kind="paged", B=64, Hq=32, Hkv=8, D=128, page=16, lo=512,
             hi=32768, dtype="bf16", window=0, softcap=0.0),
        # Serving a few users: a request is admitted into the paged cache and decodes its
        # first token together with the running ones.
        dict(name="paged_admit", kind="paged_cache", running=4, Hq=32, Hkv=8, D=128, page=64,
             lo=300, hi=2000, prompt=777, dtype="fp16"),
        # MLA decode step over the compressed latent cache.
        dict(name="mla_decode", kind="mla_decode", B=32, H=32, latent=512, page=64, lo=4096,
             hi=4096, dtype="bf16"),
        # The MLA module on a batch of prompts, with its projections.
        dict(name="mla_module_prefill", kind="mla_module", B=2, S=4096, hidden=4096, H=32,
             head_dim=128, latent=512, dtype="bf16"),
        # A training step's attention on a GQA model, ragged length.
        dict(name="train_gqa", kind="train", B=2, Hq=32, Hkv=8, S=2011, D=128, dtype="bf16",
             causal=True, window=0, softcap=0.0),
        # Training a small model in fp32.
        dict(name="train_fp32", kind="train", B=2, Hq=8, Hkv=8, S=1024, D=64, dtype="fp32",
             causal=True, window=0, softcap=0.0),
    ]


# ---------------------------------------------------------------------------------
# Drawn cases
# ---------------------------------------------------------------------------------

# The most attention work of a drawn case, in head-dim multiplies of causal (query, key)
# pairs: half of prefill_mha's.
_MAX_FORWARD = 2 * 32 * 4096 * 4097 // 2 * 128


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _heads(rng):
    """(Hq, Hkv) of multi-head, grouped-query and multi-query models."""
    return rng.choice([(8, 8), (12, 12), (16, 16), (32, 32), (8, 2), (32, 8), (24, 8), (28, 4),
                       (40, 8), (8, 1)])


def _options(rng, S):
    return dict(window=_log(rng, 64, 4096) if rng.random() < 0.25 else 0,
                softcap=rng.choice([20.0, 30.0, 50.0]) if rng.random() < 0.2 else 0.0)


def _draw_forward(rng):
    Hq, Hkv = _heads(rng)
    S = _log(rng, 32, 8192)
    D = rng.choice([64, 64, 80, 96, 128, 128, 128, 192, 256])
    room = max(1, int(_MAX_FORWARD // (Hq * S * S // 2 * D)))
    B = rng.randint(1, min(16, room))
    while B * Hq * S * S // 2 * D > _MAX_FORWARD:
        S -= S // 8
    case = dict(kind="forward", B=B, Hq=Hq, Hkv=Hkv, S=S, D=D,
                dtype=rng.choice(["bf16", "bf16", "fp16"]), causal=rng.random() < 0.7,
                radius=0, **_options(rng, S))
    if S >= 512 and rng.random() < 0.2:
        case["radius"] = _log(rng, 64, 2048)
    return case


def _draw_cached(rng):
    Hq, Hkv = _heads(rng)
    D = rng.choice([64, 128, 128, 256])
    token = rng.random() < 0.5
    S = rng.choice([1, 1, 1, 2, 4, 7]) if token else _log(rng, 16, 1024)
    Sc = _log(rng, 64, 16384)
    room = min(32 if token else 4, 2 ** 30 // ((Sc + S) * Hkv * D * 4),
               _MAX_FORWARD // (Hq * S * (Sc + S) * D))
    return dict(kind="cached", B=rng.randint(1, max(1, int(room))), Hq=Hq, Hkv=Hkv, S=S, Sc=Sc,
                max_len=Sc + S + rng.choice([0, 1, 64, 511]), D=D,
                dtype=rng.choice(["bf16", "bf16", "fp16"]), **_options(rng, Sc))


def _draw_paged(rng):
    Hq, Hkv = _heads(rng)
    D = rng.choice([64, 128, 128, 256])
    hi = _log(rng, 64, 32768)
    room = 2 ** 32 // (hi * Hkv * D * 4)
    return dict(kind="paged", B=_log(rng, 1, max(1, min(128, int(room)))), Hq=Hq, Hkv=Hkv, D=D,
                page=rng.choice([16, 16, 32, 64, 128]), lo=max(1, hi // rng.choice([1, 4, 64])),
                hi=hi, dtype=rng.choice(["bf16", "bf16", "fp16"]), **_options(rng, hi))


def _draw_paged_cache(rng):
    Hq, Hkv = _heads(rng)
    hi = _log(rng, 64, 4096)
    return dict(kind="paged_cache", running=rng.randint(0, 8), Hq=Hq, Hkv=Hkv,
                D=rng.choice([64, 128]), page=rng.choice([16, 64]), lo=max(1, hi // 8), hi=hi,
                prompt=_log(rng, 8, 4096), dtype=rng.choice(["bf16", "fp16"]))


def _draw_mla_decode(rng):
    hi = _log(rng, 64, 16384)
    return dict(kind="mla_decode", B=_log(rng, 1, max(1, min(64, 2 ** 19 // hi))),
                H=rng.choice([16, 32, 32, 64, 128]), latent=rng.choice([256, 512, 512]),
                page=rng.choice([16, 64, 64]), lo=max(1, hi // rng.choice([1, 1, 4])), hi=hi,
                dtype=rng.choice(["bf16", "bf16", "fp16"]))


def _draw_mla_module(rng):
    hidden, H = rng.choice([(2048, 16), (4096, 32)])
    S = _log(rng, 24, 4096)
    return dict(kind="mla_module", B=rng.randint(1, 2 if S > 1024 else 4), S=S, hidden=hidden,
                H=H, head_dim=128, latent=rng.choice([256, 512]),
                dtype=rng.choice(["bf16", "bf16", "fp16"]))


def _draw_train(rng):
    Hq, Hkv = _heads(rng)
    dtype = rng.choice(["bf16", "bf16", "fp16", "fp32"])
    fp32 = dtype == "fp32"
    S = _log(rng, 64, 1024 if fp32 else 4096)
    D = rng.choice([64, 128]) if fp32 else rng.choice([64, 96, 128, 128, 192, 256])
    most = _MAX_FORWARD // (20 if fp32 else 2)
    room = max(1, int(most // (Hq * S * S // 2 * D)))
    B = rng.randint(1, min(8, room))
    while B * Hq * S * S // 2 * D > most:
        S -= S // 8
    return dict(kind="train", B=B, Hq=Hq, Hkv=Hkv, S=S, D=D, dtype=dtype,
                causal=rng.random() < 0.75, **_options(rng, S))


def draw(rng):
    return rng.choice([_draw_forward, _draw_forward, _draw_cached, _draw_cached, _draw_paged,
                       _draw_paged_cache, _draw_mla_decode, _draw_mla_module, _draw_train,
                       _draw_train])(rng)


# ---------------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------------


def _rand(gen, shape, dtype):
    return torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32).to(dtype)


def _heads_view(gen, B, H, S, D, dtype):
    """[B, H, S, D] as a projection's output gives it: a view of [B, S, H D]."""
    return _rand(gen, (B, S, H, D), dtype).transpose(1, 2)


def _lengths(rng, n, lo, hi):
    return [int(x) for x in rng.integers(lo, hi + 1, size=n)]


def _tables(rng, lens, page):
    """Block tables over a pool in random page order: (int32 [B, width], pages used)."""
    need = [-(-n // page) for n in lens]
    order = rng.permutation(sum(need))
    bt = np.zeros((len(lens), max(need)), dtype=np.int32)
    at = 0
    for b, n in enumerate(need):
        bt[b, :n] = order[at:at + n]
        at += n
    return torch.from_numpy(bt).cuda(), sum(need)


def _mask(case):
    if not case.get("radius"):
        return None
    return ffa.create_local_block_mask(case["S"], case["S"], 64, 64, case["radius"])


def _opt(case):
    return dict(sliding_window=case["window"] or None, softcap=case["softcap"] or None)


def prepare(case, seed):
    kind = case["kind"]
    dt = DTYPES[case["dtype"]]
    gen = torch.Generator(device="cuda").manual_seed(seed)
    rng = np.random.default_rng(seed)
    st = {"case": case}
    if kind in ("forward", "train"):
        B, Hq, Hkv, S, D = (case[x] for x in ("B", "Hq", "Hkv", "S", "D"))
        st["q"] = _rand(gen, (B, Hq, S, D), dt)
        st["k"] = _rand(gen, (B, Hkv, S, D), dt)
        st["v"] = _rand(gen, (B, Hkv, S, D), dt)
        if kind == "train":
            st["do"] = _rand(gen, (B, Hq, S, D), dt)
            for x in "qkv":
                st[x].requires_grad_()
        else:
            st["mask"] = _mask(case)
    elif kind == "cached":
        B, Hq, Hkv, S, D = (case[x] for x in ("B", "Hq", "Hkv", "S", "D"))
        cache = ffa.ContinuousKVCache(B, case["max_len"], Hkv, D, dtype=dt, device="cuda")
        cache.append(_rand(gen, (B, Hkv, case["Sc"], D), dt), _rand(gen, (B, Hkv, case["Sc"], D), dt))
        st["kv_cache"] = cache.get_cache(B)
        st["q"] = _heads_view(gen, B, Hq, S, D, dt)
        st["k"] = _heads_view(gen, B, Hkv, S, D, dt)
        st["v"] = _heads_view(gen, B, Hkv, S, D, dt)
    elif kind == "paged":
        lens = _lengths(rng, case["B"], case["lo"], case["hi"])
        st["bt"], pages = _tables(rng, lens, case["page"])
        st["lens"] = torch.tensor(lens, dtype=torch.int32, device="cuda")
        st["max_len"] = max(lens)
        shape = (pages, case["Hkv"], case["page"], case["D"])
        st["k"] = _rand(gen, shape, dt)
        st["v"] = _rand(gen, shape, dt)
        st["q"] = _rand(gen, (case["B"], case["Hq"], case["D"]), dt)
    elif kind == "paged_cache":
        H, D, page = case["Hkv"], case["D"], case["page"]
        lens = _lengths(rng, case["running"], case["lo"], case["hi"])
        pages = sum(-(-n // page) for n in lens + [case["prompt"]]) + 8
        cache = ffa.PagedKVCache(pages, page, H, D, dtype=dt, device="cuda")
        for sid, n in enumerate(lens):
            cache.append_tokens(sid, _rand(gen, (H, n, D), dt), _rand(gen, (H, n, D), dt))
        st["cache"] = cache
        st["k"] = _rand(gen, (H, case["prompt"], D), dt)
        st["v"] = _rand(gen, (H, case["prompt"], D), dt)
        st["q"] = _rand(gen, (case["running"] + 1, case["Hq"], D), dt)
    elif kind == "mla_decode":
        lens = _lengths(rng, case["B"], case["lo"], case["hi"])
        st["bt"], pages = _tables(rng, lens, case["page"])
        st["lens"] = torch.tensor(lens, dtype=torch.int32, device="cuda")
        st["max_len"] = max(lens)
        dim = case["latent"] + ROPE
        st["kv"] = _rand(gen, (pages, case["page"], dim), dt)
        st["q"] = _rand(gen, (case["B"], case["H"], dim), dt)
    else:  # mla_module
        with torch.device("cuda"):
            m = ffa.FastestFlashMLA(case["hidden"], case["H"], case["head_dim"], case["latent"],
                                    ROPE).to(dt).eval()
        with torch.no_grad():
            for p in m.parameters():
                p.normal_(0.0, 0.02, generator=gen)
        st["module"] = m
        st["x"] = _rand(gen, (case["B"], case["S"], case["hidden"]), dt)
    return st


# ---------------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------------


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "forward":
        return ffa.fastest_flash_attn_forward(
            state["q"], state["k"], state["v"], causal=case["causal"], num_kv_heads=case["Hkv"],
            block_mask=state["mask"], block_size=64 if case["radius"] else None, return_lse=True,
            **_opt(case))
    if kind == "cached":
        return ffa.fastest_flash_attn_forward(
            state["q"], state["k"], state["v"], causal=True, num_kv_heads=case["Hkv"],
            kv_cache=state["kv_cache"], return_lse=True, **_opt(case))
    if kind == "paged":
        return ffa.fastest_flash_paged_decode(
            state["q"], state["k"], state["v"], state["bt"], state["lens"], return_lse=True,
            max_context_len=state["max_len"], **_opt(case))
    if kind == "paged_cache":
        cache, new = state["cache"], case["running"]
        cache.append_tokens(new, state["k"], state["v"])
        out = cache.decode(state["q"], list(range(new + 1)), return_lse=True)
        cache.free_sequence(new)
        return out
    if kind == "mla_decode":
        return ffa.fastest_flash_mla_decode(
            state["q"], state["kv"], state["bt"], state["lens"], dim_v=case["latent"],
            scale=_mla_scale(), return_lse=True, max_context_len=state["max_len"])
    if kind == "mla_module":
        with torch.no_grad():
            return state["module"](state["x"])
    out = ffa.fastest_flash_attn_func(state["q"], state["k"], state["v"], causal=case["causal"],
                                      num_kv_heads=case["Hkv"], **_opt(case))
    grads = torch.autograd.grad(out, (state["q"], state["k"], state["v"]), state["do"])
    return (out.detach(), *grads)


def _mla_scale():
    return 1.0 / math.sqrt(128 + ROPE)  # the module's: head_dim 128 and the rope dims


# ---------------------------------------------------------------------------------
# Work
# ---------------------------------------------------------------------------------


def _pairs(case):
    """Visible (query, key) pairs per head and the keys any query sees."""
    off = case.get("Sc", 0)
    S = case["S"]
    n = S + off
    row = off + np.arange(S, dtype=np.int64)
    hi = np.minimum(row, n - 1) if case.get("causal", True) else np.full(S, n - 1)
    lo = np.maximum(row - case["window"] + 1, 0) if case["window"] else np.zeros(S, np.int64)
    mask = _mask(case)
    if mask is None:
        return int(np.maximum(hi - lo + 1, 0).sum()), int(n - lo.min())
    kept = mask.numpy()
    j = np.arange(kept.shape[1], dtype=np.int64)
    total = 0
    for i in range(kept.shape[0]):
        a, b = i * 64, min(i * 64 + 64, S)
        over = (np.minimum(hi[a:b, None], j * 64 + 63) - np.maximum(lo[a:b, None], j * 64) + 1)
        total += int((np.maximum(over, 0) * kept[i]).sum())
    return total, n


def work(case):
    kind = case["kind"]
    e = 4 if case["dtype"] == "fp32" else 2
    if kind in ("forward", "cached", "train"):
        pairs, keys = _pairs(case)
        B, Hq, Hkv, S, D = (case[x] for x in ("B", "Hq", "Hkv", "S", "D"))
        qo = B * Hq * S * D * e   # q, or O
        kv = B * Hkv * keys * D * e  # K, or V
        if kind == "train":  # q, dO, O, dQ; K, V, dK, dV; the forward's and five products
            return {"bytes": 4 * qo + 4 * kv, "flops": 14 * D * pairs * B * Hq}
        return {"bytes": 2 * qo + 2 * kv + B * Hq * S * 4, "flops": 4 * D * pairs * B * Hq}
    if kind == "mla_module":
        T = case["B"] * case["S"]
        hid, H, hd, lat = case["hidden"], case["H"], case["head_dim"], case["latent"]
        params = hid * (H * (hd + ROPE) + lat + ROPE) + lat * H * 2 * hd + H * (hd + ROPE) * hid
        pairs = case["S"] * (case["S"] + 1) // 2
        return {"bytes": (2 * T * hid + params) * e,
                "flops": 2 * T * params + 2 * (2 * hd + ROPE) * pairs * case["B"] * H}
    if kind == "paged_cache":  # the running lengths at their mean; the prompt is copied in
        tokens = case["running"] * (case["lo"] + case["hi"]) // 2 + case["prompt"]
        kv = case["Hkv"] * case["D"] * 2 * e
        return {"bytes": (tokens + case["prompt"]) * kv
                + (case["running"] + 1) * case["Hq"] * case["D"] * 2 * e,
                "flops": 4 * tokens * case["Hq"] * case["D"]}
    mean = (case["lo"] + case["hi"]) // 2
    if kind == "mla_decode":
        dim = case["latent"] + ROPE
        return {"bytes": case["B"] * (mean * dim + case["H"] * (dim + case["latent"])) * e,
                "flops": 2 * case["B"] * mean * case["H"] * (dim + case["latent"])}
    if case["window"]:
        mean = min(mean, case["window"])
    kv = mean * case["Hkv"] * case["D"] * 2
    return {"bytes": case["B"] * (kv + 2 * case["Hq"] * case["D"]) * e,
            "flops": 4 * case["B"] * mean * case["Hq"] * case["D"]}


# ---------------------------------------------------------------------------------
# Results in 64 bits
# ---------------------------------------------------------------------------------


def _attend(q, k, v, scale, off, causal, window, softcap, mask=None, do=None):
    """One head in float64: q [S, D] at positions off.., k and v [N, *]. (O, lse), or with
    the output's gradient (O, dq, dk, dv). Rows are taken in blocks."""
    q, k, v = q.double(), k.double(), v.double()
    o, lse, dq = [], [], []
    dk, dv = torch.zeros_like(k), torch.zeros_like(v)
    key = torch.arange(k.size(0), device=k.device)
    kt, vt = k.t().contiguous(), v.t().contiguous()
    for a in range(0, q.size(0), 4096):
        qa = q[a:a + 4096]
        s = (qa @ kt) * scale
        if softcap:
            t = torch.tanh(s / softcap)
            s = softcap * t
        row = off + a + torch.arange(qa.size(0), device=k.device)
        keep = torch.ones_like(s, dtype=torch.bool)
        if causal:
            keep &= key[None, :] <= row[:, None]
        if window:
            keep &= key[None, :] >= row[:, None] - window + 1
        if mask is not None:
            keep &= mask[(row - off) // 64][:, key // 64]
        s = s.masked_fill(~keep, float("-inf"))
        z = torch.logsumexp(s, dim=-1)
        p = torch.exp(s - z[:, None]).masked_fill(~keep, 0.0)
        oa = p @ v
        o.append(oa)
        lse.append(z)
        if do is not None:
            da = do[a:a + 4096].double()
            ds = p * (da @ vt - (da * oa).sum(-1, keepdim=True))
            if softcap:
                ds = ds * (1 - t * t)
            ds = ds * scale
            dq.append(ds @ k)
            dk += ds.t().contiguous() @ qa
            dv += p.t().contiguous() @ da
    if do is None:
        return torch.cat(o), torch.cat(lse)
    return torch.cat(o), torch.cat(dq), dk, dv


def exact(case, seed):
    kind = case["kind"]
    if kind == "mla_module":
        return _exact_module(case, seed)
    st = prepare(case, seed)
    if kind == "mla_decode":
        lat, o, lse = case["latent"], [], []
        for b, n in enumerate(st["lens"].tolist()):
            ids = st["bt"][b, :-(-n // case["page"])].long()
            rows = st["kv"][ids].flatten(0, 1)[:n]
            ob, lb = _attend(st["q"][b], rows, rows[:, :lat], _mla_scale(), n, False, 0, 0.0)
            o.append(ob)
            lse.append(lb)
        return torch.stack(o), torch.stack(lse)
    D, Hq, Hkv = case["D"], case["Hq"], case["Hkv"]
    G, scale = Hq // Hkv, 1.0 / math.sqrt(D)
    if kind in ("paged", "paged_cache"):
        o, lse = [], []
        if kind == "paged":
            seqs = []
            for b, n in enumerate(st["lens"].tolist()):
                ids = st["bt"][b, :-(-n // case["page"])].long()
                seqs.append([st[x][ids].transpose(0, 1).flatten(1, 2)[:, :n] for x in "kv"])
        else:
            seqs = [st["cache"].get_kv(i) for i in range(case["running"])]
            seqs.append((st["k"], st["v"]))
        win, cap = case.get("window", 0), case.get("softcap", 0.0)
        for b, (k, v) in enumerate(seqs):
            # a group's query heads all sit at the last position
            per = [_attend(st["q"][b, h * G:(h + 1) * G], k[h][-win:] if win else k[h],
                           v[h][-win:] if win else v[h], scale, 0, False, 0, cap)
                   for h in range(Hkv)]
            o.append(torch.cat([x for x, _ in per]))
            lse.append(torch.cat([x for _, x in per]))
        return torch.stack(o), torch.stack(lse)
    q, k, v = (st[x].detach() for x in "qkv")
    if kind == "cached":
        k = torch.cat([st["kv_cache"][0], k], dim=2)
        v = torch.cat([st["kv_cache"][1], v], dim=2)
    mask = _mask(case)
    mask = None if mask is None else mask.cuda()
    args = (scale, case.get("Sc", 0), case.get("causal", True), case["window"], case["softcap"])
    B, S = case["B"], case["S"]
    if kind == "train":
        o, dq = (torch.empty(B, Hq, S, D, dtype=torch.float64, device="cuda") for _ in range(2))
        dk, dv = (torch.zeros(B, Hkv, S, D, dtype=torch.float64, device="cuda") for _ in range(2))
        for b in range(B):
            for h in range(Hq):
                o[b, h], dq[b, h], gk, gv = _attend(q[b, h], k[b, h // G], v[b, h // G], *args,
                                                    do=st["do"][b, h])
                dk[b, h // G] += gk
                dv[b, h // G] += gv
        return o, dq, dk, dv
    o = torch.empty(B, Hq, S, D, dtype=torch.float64, device="cuda")
    lse = torch.empty(B, Hq, S, 1, dtype=torch.float64, device="cuda")
    for b in range(B):
        for h in range(Hq):
            o[b, h], lse[b, h, :, 0] = _attend(q[b, h], k[b, h // G], v[b, h // G], *args, mask)
    return o, lse


def _exact_module(case, seed):
    st = prepare(case, seed)
    w = {n: p.detach().double() for n, p in st["module"].named_parameters()}
    x = st["x"].double()
    B, S, H, hd = case["B"], case["S"], case["H"], case["head_dim"]

    def proj(t, name):
        return t @ w[name + ".weight"].t().contiguous()

    # the rotation tables are values of the module's dtype, part of what it defines
    # (positions and frequencies in that dtype); everything after them is exact
    dt = st["x"].dtype
    freq = (1.0 / 10000.0 ** (torch.arange(0, ROPE, 2).float() / ROPE)).cuda().to(dt)
    ang = torch.outer(torch.arange(S, device="cuda", dtype=dt), freq)
    cos, sin = ang.cos().double(), ang.sin().double()

    def rope(t):  # [..., S, ROPE]
        a, b = t[..., :ROPE // 2], t[..., ROPE // 2:]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], dim=-1)

    qn = proj(x, "q_proj").view(B, S, H, hd).transpose(1, 2)
    qr = rope(proj(x, "q_rope_proj").view(B, S, H, ROPE).transpose(1, 2))
    kv = proj(proj(x, "kv_down_proj"), "kv_up_proj").view(B, S, H, 2 * hd).transpose(1, 2)
    kr = rope(proj(x, "k_rope_proj"))
    attn = torch.zeros(B, S, H, hd + ROPE, dtype=torch.float64, device="cuda")
    for b in range(B):
        for h in range(H):
            q = torch.cat([qn[b, h], qr[b, h]], dim=-1)
            k = torch.cat([kv[b, h, :, :hd], kr[b]], dim=-1)
            attn[b, :, h, :hd] = _attend(q, k, kv[b, h, :, hd:], 1.0 / math.sqrt(hd + ROPE), 0,
                                         True, 0, 0.0)[0]
    return proj(attn.flatten(2), "o_proj")


def tolerance(case):
    """About four times the largest error against ``exact`` over listed and drawn cases:
    bf16 2.5e-3 (5e-3 through the module's projections), fp16 an eighth of that (the
    mantissas differ by three bits), fp32 1.5e-6."""
    if case["dtype"] == "fp32":
        return {"rel": 6e-6}
    rel = 2e-2 if case["kind"] == "mla_module" else 1e-2
    return {"rel": rel if case["dtype"] == "bf16" else rel / 8}
