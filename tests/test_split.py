"""Prefill calls whose keys are split over workgroups, and KV caches read in place.

CPU: keeping a cache apart resolves to the concatenated call, for every layout, and
refuses what concatenation refuses. GPU: split calls against the oracle at the edges of
their tiles, ranges and segments."""

from __future__ import annotations

import ctypes
import math

import numpy as np
import pytest
import torch

import fastest_flash_attention_amd as ffa
from fastest_flash_attention_amd.kernels import _lib
from fastest_flash_attention_amd.ops import attention_forward as af
from tests.gpu_util import assert_parity, np32, require_gpu, say, seeded
from oracle import reference_forward as rf

BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32


# ---------------------------------------------------------------------------------
# CPU: the cache's route
# ---------------------------------------------------------------------------------

def _layouts():
    def plain(B, H, S, D, dt):
        return torch.randn(B, H, S, D).to(dt)

    def projection(B, H, S, D, dt):
        return torch.randn(B, S, H * D).to(dt).view(B, S, H, D).transpose(1, 2)

    def prefix(B, H, S, D, dt):  # of a preallocated cache
        return torch.randn(B, H, S + 37, D).to(dt)[:, :, :S]

    def odd_rows(B, H, S, D, dt):
        return torch.randn(B, H, S, D + 4).to(dt)[..., :D]

    def odd_base(B, H, S, D, dt):
        return torch.randn(B * H * S * D + 3).to(dt)[3:].view(B, H, S, D)

    def dims_last(B, H, S, D, dt):
        return torch.randn(B, H, D, S).to(dt).transpose(2, 3)

    def one_head_broadcast(B, H, S, D, dt):
        return torch.randn(B, 1, S, D).to(dt).expand(B, H, S, D)

    return [plain, projection, prefix, odd_rows, odd_base, dims_last, one_head_broadcast]


@pytest.mark.parametrize("cache_of", _layouts(), ids=lambda f: f.__name__)
@pytest.mark.parametrize("new_of", _layouts(), ids=lambda f: f.__name__)
@pytest.mark.parametrize("D,dt", [(64, BF16), (40, F16), (20, BF16), (16, F32)])
def test_cache_in_place_resolves_to_the_concatenated_call(cache_of, new_of, D, dt):
    q = torch.randn(2, 4, 3, D).to(dt)
    k, v = new_of(2, 2, 3, D, dt), new_of(2, 2, 3, D, dt)
    kv = (cache_of(2, 2, 7, D, dt), cache_of(2, 2, 7, D, dt))
    kw = dict(causal=True, num_kv_heads=2, kv_cache=kv, return_lse=True)
    want = af.resolve_forward_args(q, k, v, **kw)
    got = af.resolve_forward_args(q, k, v, cache_in_place=True, **kw)
    assert got.S_kv == want.S_kv == 10 and got.q_offset == want.q_offset == 7
    if got.cache is not None:  # only what the kernels' 16-byte loads can take
        for t in got.cache:
            assert t.stride(3) == 1 and t.data_ptr() % 16 == 0
            assert all(st % 8 == 0 for st in t.stride()[:3])
    af._join_cache(got)
    assert torch.equal(got.k, want.k) and torch.equal(got.v, want.v)


@pytest.mark.parametrize("shape_k,shape_v,dt", [
    ((2, 2, 7, 64), (2, 2, 6, 64), BF16),   # K and V of different lengths
    ((1, 2, 7, 64), (1, 2, 7, 64), BF16),   # batch
    ((2, 3, 7, 64), (2, 3, 7, 64), BF16),   # heads
    ((2, 2, 7, 32), (2, 2, 7, 32), BF16),   # head_dim
])
def test_cache_in_place_refuses_what_concatenation_refuses(shape_k, shape_v, dt):
    q, k = torch.randn(2, 4, 3, 64).to(BF16), torch.randn(2, 2, 3, 64).to(BF16)
    kv = (torch.randn(shape_k).to(dt), torch.randn(shape_v).to(dt))
    kw = dict(num_kv_heads=2, kv_cache=kv)
    with pytest.raises(Exception) as want:
        af.resolve_forward_args(q, k, k, **kw)
    with pytest.raises(type(want.value)):
        af.resolve_forward_args(q, k, k, cache_in_place=True, **kw)


def test_cache_of_another_dtype_is_concatenated():
    q, k = torch.randn(1, 2, 3, 64).to(BF16), torch.randn(1, 2, 3, 64).to(BF16)
    kv = (torch.randn(1, 2, 7, 64), torch.randn(1, 2, 7, 64))
    r = af.resolve_forward_args(q, k, k, kv_cache=kv, cache_in_place=True)
    assert r.cache is None and r.k.dtype == F32  # as torch.cat promotes


def _args(**kw):
    a = _lib.PrefillArgs()
    for name, val in dict(batch=1, heads_q=8, heads_kv=8, seqlen_q=1, seqlen_kv=4096, head_dim=128,
                          causal=1, q_offset=4095, scale=1.0, dtype=_lib.FFA_DTYPE_BF16).items():
        setattr(a, name, kw.pop(name, val))
    for name, val in kw.items():
        setattr(a, name, val)
    return a


def test_workspace_query():
    """0 where the call runs unsplit; else the fp32 partials and their lse."""
    lib = _lib.load()

    def need(**kw):
        return lib.ffa_prefill_workspace_bytes(ctypes.byref(_args(**kw)))

    cached = dict(k_cache=16, v_cache=16, cache_len=4095)
    n = need(**cached)
    assert n > 0 and n % (8 * 129 * 4) == 0
    assert need(dtype=_lib.FFA_DTYPE_FP32, **cached) == 0
    assert need(block_key_mask=16, **cached) == 0
    assert need(head_dim=192, v_head_dim=128, **cached) == 0
    assert need(batch=0, **cached) == 0 and need(seqlen_q=0, **cached) == 0
    assert need(heads_q=7, heads_kv=2, **cached) == 0
    assert need(cache_len=5000, k_cache=16, v_cache=16) == 0
    full = dict(batch=4, heads_q=32, heads_kv=32, q_offset=0)
    assert need(seqlen_q=4096, seqlen_kv=4096, **full) == 0
    assert need(seqlen_q=100, seqlen_kv=100, heads_q=2, heads_kv=2, q_offset=0) == 0
    assert lib.ffa_prefill_workspace_bytes(None) == 0
    for cap in (2 ** 20, 2 ** 28):  # positions up to the ABI's limit: the planner ends
        assert need(seqlen_q=1, seqlen_kv=cap, k_cache=16, v_cache=16, cache_len=cap - 1,
                    q_offset=cap - 1) > 0


def test_cached_call_without_a_workspace_is_refused():
    lib = _lib.load()
    a = _args(k_cache=16, v_cache=16, cache_len=4095, q=16, k=16, v=16, o=16)
    for name in ("q_stride", "k_stride", "v_stride", "o_stride", "k_cache_stride", "v_cache_stride"):
        getattr(a, name)[:] = [128, 128, 128, 1]
    assert lib.ffa_prefill_fwd(ctypes.byref(a), None) == -6
    a.k_cache_stride[2] = 100
    assert lib.ffa_prefill_fwd(ctypes.byref(a), None) == -4
    a.cache_len = 4097
    assert lib.ffa_prefill_fwd(ctypes.byref(a), None) == -1


# ---------------------------------------------------------------------------------
# GPU
# ---------------------------------------------------------------------------------

CACHED = [
    # B, Hq, Hkv, Sq, Sc, D, dtype, window, softcap
    (1, 2, 2, 1, 1, 64, BF16, None, None),
    (2, 8, 2, 1, 63, 128, BF16, None, None),
    (2, 8, 2, 1, 64, 128, F16, None, None),
    (1, 4, 1, 1, 65, 72, BF16, None, None),
    (3, 8, 2, 1, 255, 128, BF16, None, 30.0),
    (1, 8, 8, 1, 256, 64, F16, None, None),
    (2, 6, 2, 2, 257, 256, BF16, None, None),
    (1, 8, 2, 1, 1500, 128, BF16, 100, None),    # the window starts inside the cache
    (1, 8, 2, 5, 1500, 128, BF16, 3, None),      # and inside the call's own keys
    (1, 28, 4, 7, 700, 128, F16, None, None),    # packed rows, not a tile's multiple
    (1, 8, 2, 32, 700, 64, BF16, None, None),    # packed rows filling one tile
    (1, 8, 2, 33, 700, 64, BF16, 300, 20.0),
    (1, 8, 2, 127, 300, 128, BF16, None, None),  # packing saves no tile
    (1, 4, 4, 128, 300, 128, F16, None, None),
    (1, 4, 4, 129, 300, 128, BF16, 150, None),
    (1, 4, 2, 300, 90, 128, BF16, None, None),   # more queries than cached keys
    (1, 4, 2, 100, 600, 192, BF16, None, None),
    (1, 2, 2, 70, 333, 256, F16, 200, 50.0),
    (1, 64, 1, 3, 400, 128, BF16, None, None),
    (40, 16, 16, 1, 130, 64, BF16, None, None),  # more workgroups than slots
]


@pytest.mark.gpu
@pytest.mark.parametrize("B,Hq,Hkv,Sq,Sc,D,dt,window,softcap", CACHED)
def test_cached_call(B, Hq, Hkv, Sq, Sc, D, dt, window, softcap):
    require_gpu()
    say(f"split cached B{B} {Hq}/{Hkv} Sq{Sq} Sc{Sc} D{D} {dt} w{window} cap{softcap}")
    q = seeded((B, Sq, Hq, D), dt, 1).transpose(1, 2)
    k, v = (seeded((B, Sq, Hkv, D), dt, s).transpose(1, 2) for s in (2, 3))
    kc, vc = (seeded((B, Hkv, Sc, D), dt, s) for s in (4, 5))
    # the cache as a prefix view of a larger buffer whose other rows must not be read
    big = [torch.full((B, Hkv, Sc + 70, D), float("nan"), dtype=dt, device="cuda") for _ in "kv"]
    big[0][:, :, :Sc] = kc.cuda()
    big[1][:, :, :Sc] = vc.cuda()
    kw = dict(causal=True, num_kv_heads=Hkv, sliding_window=window, softcap=softcap)
    args = (q.cuda(), k.cuda(), v.cuda())
    cache = (big[0][:, :, :Sc], big[1][:, :, :Sc])
    assert af.prepare_prefill(*args, kv_cache=cache, **kw).args.k_cache  # read in place
    o, lse = ffa.fastest_flash_attn_forward(*args, kv_cache=cache, return_lse=True, **kw)
    ro, rl = rf.forward(np32(q), np32(k), np32(v), kv_cache=(np32(kc), np32(vc)), return_lse=True,
                        **kw)
    assert_parity(o, ro, lse, rl, "cached")


OWN = [
    # B, Hq, Hkv, Sq, Skv, D, dtype, causal, window, softcap, scale
    (1, 2, 2, 2048, 2048, 64, BF16, True, None, None, None),
    (1, 2, 1, 2049, 2049, 128, F16, True, None, None, None),
    (1, 1, 1, 2500, 2500, 128, BF16, True, 2100, 30.0, None),
    (2, 4, 1, 17, 3001, 128, BF16, False, None, None, -0.4),
    (1, 2, 2, 130, 2111, 256, BF16, False, None, None, None),
    (1, 2, 2, 2300, 2300, 192, F16, True, None, None, 0.5),
    (1, 8, 2, 40, 2050, 64, BF16, False, None, 20.0, 3.0),
]


@pytest.mark.gpu
@pytest.mark.parametrize("B,Hq,Hkv,Sq,Skv,D,dt,causal,window,softcap,scale", OWN)
@pytest.mark.parametrize("mask", [False, True])
def test_own_keys(B, Hq, Hkv, Sq, Skv, D, dt, causal, window, softcap, scale, mask):
    require_gpu()
    say(f"split own B{B} {Hq}/{Hkv} Sq{Sq} Skv{Skv} D{D} {dt} causal{causal} mask{mask}")
    q = seeded((B, Hq, Sq, D), dt, 1)
    k, v = (seeded((B, Hkv, Skv, D), dt, s) for s in (2, 3))
    kw = dict(causal=causal, num_kv_heads=Hkv, sliding_window=window, softcap=softcap, scale=scale,
              block_size=64)
    if mask:  # every third key tile dropped, and one query tile that sees nothing
        bm = torch.ones(math.ceil(Sq / 64), math.ceil(Skv / 64), dtype=torch.bool)
        bm[:, ::3] = False
        bm[-1] = False
        kw["block_mask"] = bm
    args = (q.cuda(), k.cuda(), v.cuda())
    assert af.prepare_prefill(*args, **kw).args.workspace  # split
    o, lse = ffa.fastest_flash_attn_forward(*args, return_lse=True, **kw)
    if mask:
        kw["block_mask"] = bm.numpy()
    ro, rl = rf.forward(np32(q), np32(k), np32(v), return_lse=True, **kw)
    assert_parity(o, ro, lse, rl, "own keys")


@pytest.mark.gpu
def test_rows_without_a_visible_key():
    """Each range leaves such rows -inf; the merge gives them O = 0 and the reference's lse
    sentinel, and the one-pass floor to rows whose scores are far below it."""
    require_gpu()
    B, H, S, Skv, D = 1, 2, 40, 2200, 64
    q = torch.ones(B, H, S, D, dtype=BF16)
    k = torch.full((B, H, Skv, D), -1.0).to(BF16)
    v = seeded((B, H, Skv, D), BF16, 3)
    for two_pass in (False, True):
        kw = dict(scale=1.6, block_size=64, two_pass=two_pass)  # every score is -102.4
        o, lse = ffa.fastest_flash_attn_forward(q.cuda(), k.cuda(), v.cuda(), return_lse=True, **kw)
        ro, rl = rf.forward(np32(q), np32(k), np32(v), return_lse=True, **kw)
        assert_parity(o, ro, lse, rl, f"floor two_pass={two_pass}")
    bm = torch.zeros(1, math.ceil(Skv / 64), dtype=torch.bool)
    o, lse = ffa.fastest_flash_attn_forward(q.cuda(), k.cuda(), v.cuda(), block_mask=bm,
                                            block_size=64, return_lse=True)
    assert not o.any() and torch.isneginf(lse).all()


@pytest.mark.gpu
@pytest.mark.parametrize("D,softcap", [(64, None), (128, None), (192, None), (128, 20.0)])
@pytest.mark.parametrize("cached", [False, True])
def test_not_a_number_reaches_the_output(D, softcap, cached):
    """A NaN query or key makes the rows that see it NaN, whichever range it lies in, and no
    other row: a range with a NaN sum is not one without a visible key."""
    require_gpu()
    say(f"split nan D{D} cap{softcap} cached{cached}")
    B, Hq, Hkv, Sq, Skv = 1, 4, 2, 40, 2200
    q = seeded((B, Hq, Sq, D), BF16, 1)
    k, v = (seeded((B, Hkv, Skv, D), BF16, s) for s in (2, 3))
    kw = dict(causal=False, num_kv_heads=Hkv, softcap=softcap)

    def call(q, k):
        if not cached:
            assert af.prepare_prefill(q.cuda(), k.cuda(), v.cuda(), **kw).args.workspace
            return ffa.fastest_flash_attn_forward(q.cuda(), k.cuda(), v.cuda(), **kw)[0].cpu()
        cache = tuple(t[:, :, :-Sq].cuda() for t in (k, v))
        own = tuple(t[:, :, -Sq:].cuda() for t in (k, v))
        assert af.prepare_prefill(q.cuda(), *own, kv_cache=cache, **kw).args.k_cache
        return ffa.fastest_flash_attn_forward(q.cuda(), *own, kv_cache=cache, **kw)[0].cpu()

    clean = call(q, k)
    assert not clean.isnan().any()
    bad_q = q.clone()
    bad_q[0, 3, 7, 5] = float("nan")
    out = call(bad_q, k)
    rows = torch.zeros(B, Hq, Sq, dtype=torch.bool)
    rows[0, 3, 7] = True
    assert out[rows].isnan().all() and not out[~rows].isnan().any()
    # (the rows of a wave move their running maxima together, so P may round to bf16
    # elsewhere: each p by 2^-8 of itself at most, O by 2^-8 max |v|, and as much when stored)
    assert (out[~rows].float() - clean[~rows].float()).abs().max() <= 2 ** -7 * v.float().abs().max()
    for at in (0, 1000, Skv - 1):  # the first range, one inside, the last key
        bad_k = k.clone()
        bad_k[0, 1, at, D - 1] = float("nan")
        out = call(q, bad_k)
        assert out[:, 2:].isnan().all() and torch.equal(out[:, :2], clean[:, :2])


@pytest.mark.gpu
def test_block_mask_sweep_longer_than_the_tile_list():
    """A workgroup whose sweep has more key tiles than its live-tile list holds (2048) visits
    every tile; too many workgroups here for the keys to be split."""
    require_gpu()
    Hq, Sq, Skv, D = 160, 128, 2048 * 64 + 200, 64
    q = seeded((1, Hq, Sq, D), BF16, 51).cuda()
    k, v = (seeded((1, 1, Skv, D), BF16, s).cuda() for s in (52, 53))
    full = torch.ones(2, math.ceil(Skv / 64), dtype=torch.bool)
    kw = dict(block_size=64, num_kv_heads=1)
    assert not af.prepare_prefill(q, k, v, block_mask=full, **kw).args.workspace
    say(f"mask sweep Skv{Skv}")
    dense, dl = ffa.fastest_flash_attn_forward(q, k, v, return_lse=True, **kw)
    masked, ml = ffa.fastest_flash_attn_forward(q, k, v, block_mask=full, return_lse=True, **kw)
    assert torch.equal(dense, masked) and torch.equal(dl, ml)


@pytest.mark.gpu
def test_split_calls_under_capture_and_on_two_streams():
    require_gpu()
    dt, D, Sc = BF16, 128, 900
    q = seeded((2, 8, 1, D), dt, 1).cuda()
    k, v = (seeded((2, 2, 1, D), dt, s).cuda() for s in (2, 3))
    cache = tuple(seeded((2, 2, Sc, D), dt, s).cuda() for s in (4, 5))

    def run():
        return ffa.fastest_flash_attn_forward(q, k, v, causal=True, num_kv_heads=2, kv_cache=cache,
                                              return_lse=True)

    run()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        go, gl = run()
    for seed in (11, 12, 13):
        q.copy_(seeded((2, 8, 1, D), dt, seed))
        cache[0].copy_(seeded((2, 2, Sc, D), dt, seed + 50))
        o, lse = run()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(go, o) and torch.equal(gl, lse), seed
    streams = [torch.cuda.Stream() for _ in range(2)]
    outs = []
    for s in streams:
        s.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(s):
            outs.append([run() for _ in range(5)])
    torch.cuda.synchronize()
    for per in outs:
        for oo, ll in per:
            assert torch.equal(oo, o) and torch.equal(ll, lse)


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["band", "runs", "causal"])
@pytest.mark.parametrize("D,softcap", [(128, None), (64, 20.0), (32, None), (64, None), (192, None),
                                       (192, 20.0), (256, None), (256, 20.0)])
def test_block_mask_runs(name, D, softcap):
    """Runs of whole, consecutive tiles in the live-tile list take the fast steps: runs that
    start at odd positions, end inside and cross the 64 positions looked at together (128 of
    32 keys from head_dim 192 on)."""
    require_gpu()
    S, Hq, n = 4400, 4, 69  # 140 workgroups: not split
    bm = torch.zeros(n, n, dtype=torch.bool)
    i, j = torch.arange(n)[:, None], torch.arange(n)[None, :]
    if name == "band":
        bm |= (j == 0) | ((i - j).abs() <= 9)
    elif name == "runs":  # 3, then 5, then the rest with holes
        bm |= (j < 3) | ((j >= 5) & (j < 10)) | ((j > 11) & (j % 13 != 0))
    else:
        bm |= j <= i
        bm[:, 66] = False
    say(f"mask runs {name} D{D} cap{softcap}")
    q = seeded((1, Hq, S, D), BF16, 1)
    k, v = (seeded((1, 1, S, D), BF16, s) for s in (2, 3))
    kw = dict(causal=name != "runs", num_kv_heads=1, softcap=softcap, block_size=64)
    args = (q.cuda(), k.cuda(), v.cuda())
    assert not af.prepare_prefill(*args, block_mask=bm, **kw).args.workspace
    o, lse = ffa.fastest_flash_attn_forward(*args, block_mask=bm, return_lse=True, **kw)
    rows = np.r_[0:70, 1000:1040, 2170:2240, 4300:4400]  # in whole 64-row tiles of the mask
    tiles = sorted({r // 64 for r in rows})
    for t in tiles:  # one query tile of the mask at a time, at its offset
        a, b = t * 64, min(t * 64 + 64, S)
        off = a
        sub = bm[t:t + 1].numpy()
        ro, rl = rf.flash_attn_cpu_forward(
            np32(q[:, :, a:b]), np.repeat(np32(k), Hq, 1), np.repeat(np32(v), Hq, 1),
            scale=1 / math.sqrt(D), causal=kw["causal"], block_q=64, block_kv=64, block_mask=sub,
            softcap=softcap, sliding_window=None, two_pass=False, compute_dtype=None, q_offset=off,
            return_lse=True)
        assert_parity(o[:, :, a:b], ro, lse[:, :, a:b], rl, f"{name} tile {t}")


@pytest.mark.gpu
@pytest.mark.parametrize("D,softcap", [(64, None), (128, 20.0), (128, None), (192, None), (192, 20.0),
                                       (256, None), (256, 20.0)])
@pytest.mark.parametrize("causal", [False, True])
def test_split_block_mask_runs(D, softcap, causal):
    """The same in split calls, whose ranges have lists of their own: whole tiles on both sides
    of a range's end, holes inside ranges, and a run up to the ragged last tile."""
    require_gpu()
    Hq, Sq, Skv = (2, 2500, 2500) if causal else (4, 300, 9017)
    say(f"split mask runs D{D} cap{softcap} causal{causal}")
    q = seeded((1, Hq, Sq, D), BF16, 1)
    k, v = (seeded((1, 1, Skv, D), BF16, s) for s in (2, 3))
    bm = torch.ones(math.ceil(Sq / 64), math.ceil(Skv / 64), dtype=torch.bool)
    bm[:, 13] = bm[:, 30:32] = False
    bm[1::2, 21] = False
    kw = dict(causal=causal, num_kv_heads=1, softcap=softcap, block_size=64)
    args = (q.cuda(), k.cuda(), v.cuda())
    assert af.prepare_prefill(*args, block_mask=bm, **kw).args.workspace  # split
    o, lse = ffa.fastest_flash_attn_forward(*args, block_mask=bm, return_lse=True, **kw)
    ro, rl = rf.forward(np32(q), np32(k), np32(v), block_mask=bm.numpy(), return_lse=True, **kw)
    assert_parity(o, ro, lse, rl, "split mask runs")


def _broadcast(t, dim):
    """t's first entry along dim, repeated without a copy, and the same values in memory."""
    one = t.narrow(dim, 0, 1)
    wide = one.expand(t.shape)
    return (one if dim == 0 else wide), wide.contiguous()


@pytest.mark.gpu
@pytest.mark.parametrize("dim", [0, 1], ids=["batch", "heads"])
@pytest.mark.parametrize("Sq,Sc", [(1, 900), (5, 700), (130, 333), (40, 0)])
def test_broadcast_keys_are_read_in_place(dim, Sq, Sc):
    """One batch entry of k, v and the cache under a larger batch of queries, and one head
    expanded to all: read through zero strides, the same bits as from memory."""
    require_gpu()
    B, Hq, Hkv, D = 3, 8, 4, 128
    say(f"split broadcast dim{dim} Sq{Sq} Sc{Sc}")
    q = seeded((B, Hq, Sq, D), BF16, 1).cuda()
    own = Sq if Sc else 2300
    pairs = [_broadcast(seeded((B, Hkv, n, D), BF16, s).cuda(), dim)
             for n, s in ((own, 2), (own, 3), (max(Sc, 1), 4), (max(Sc, 1), 5))]
    outs = []
    for form in (0, 1):
        k, v, kc, vc = (p[form] for p in pairs)
        kw = dict(causal=bool(Sc), num_kv_heads=Hkv, kv_cache=(kc, vc) if Sc else None)
        args = af.prepare_prefill(q, k, v, **kw).args
        assert args.workspace and bool(args.k_cache) == bool(Sc)  # split, the cache in place
        outs.append(ffa.fastest_flash_attn_forward(q, k, v, return_lse=True, **kw))
    assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])
    ro, rl = rf.forward(np32(q), np32(k), np32(v), return_lse=True, causal=bool(Sc),
                        num_kv_heads=Hkv, kv_cache=(np32(kc), np32(vc)) if Sc else None)
    assert_parity(outs[0][0], ro, outs[0][1], rl, "broadcast")
