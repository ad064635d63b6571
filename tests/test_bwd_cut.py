"""Backward calls whose dK/dV sweeps are cut into parts (few, uneven workgroups)."""

from __future__ import annotations

import ctypes
import math

import numpy as np
import pytest
import torch

import fastest_flash_attention_amd as ffa
from fastest_flash_attention_amd.kernels import _lib
from oracle import reference_backward as rb
from tests.gpu_util import np32, require_gpu, say, seeded
from tests.test_gpu_backward import _check, _oracle_forward

BF16, F16 = torch.bfloat16, torch.float16


def _args(B, Hq, Hkv, Sq, Skv, D, Dv=0, q_offset=0, causal=1, window=0, dtype=0):
    a = _lib.AttnBwdArgs()
    a.batch, a.heads_q, a.heads_kv, a.seqlen_q, a.seqlen_kv, a.head_dim = B, Hq, Hkv, Sq, Skv, D
    a.v_head_dim, a.q_offset, a.causal, a.window, a.dtype = Dv, q_offset, causal, window, dtype
    return a


def test_workspace_query():
    """The statistics alone where no sweep is cut, else whole fp32 partial tiles with them."""
    lib = _lib.load()

    def extra(*args, **kw):
        a = _args(*args, **kw)
        base = lib.ffa_attn_bwd_workspace_bytes(a.batch, a.heads_q, a.seqlen_q)
        return lib.ffa_attn_bwd_split_workspace_bytes(ctypes.byref(a)) - base

    n = extra(2, 32, 8, 2011, 2011, 128)
    assert n > 0 and n % (2 * 8 * 128 * 256 * 4) == 0
    assert extra(2, 32, 8, 2011, 2011, 192, Dv=128) % (128 * 320 * 4) == 0
    for plain in ((4, 32, 32, 8192, 8192, 128), (1, 2, 2, 100, 100, 64), (1, 8, 2, 2048, 2048, 256)):
        assert extra(*plain) == 0, plain
    assert extra(2, 32, 8, 2011, 2011, 128, dtype=2) == 0
    assert extra(1, 8, 2, 2000, 0, 128) == 0
    assert lib.ffa_attn_bwd_split_workspace_bytes(None) == 0
    assert lib.ffa_attn_bwd_split_workspace_bytes(ctypes.byref(_args(1, 7, 2, 9, 9, 64))) == 0


@pytest.mark.parametrize("B,Hq,Hkv,Sq,Skv,D,off,causal,window,tiles", [
    # key tiles that see rows: a window's ten or so, the first sixteen of a prefix
    (1, 32, 8, 512, 16000, 128, 15488, 1, 1024, 12),
    (1, 8, 1, 2048, 65536, 128, 0, 1, 0, 16),
    (1, 32, 1, 512, 130000, 128, 129488, 1, 1024, 13),
    (1, 64, 2, 324, 63064, 192, 0, 1, 127, 3),
    (3, 32, 1, 525, 32016, 192, 12526, 1, 102, 6),
])
def test_workspace_of_few_live_key_tiles(B, Hq, Hkv, Sq, Skv, D, off, causal, window, tiles):
    """Partial tiles for the key tiles whose sweep is cut, at most sixteen each, and never more
    than 4/3 of the workgroups that run at once."""
    lib = _lib.load()
    a = _args(B, Hq, Hkv, Sq, Skv, D, 0, off, causal, window)
    extra = (lib.ffa_attn_bwd_split_workspace_bytes(ctypes.byref(a))
             - lib.ffa_attn_bwd_workspace_bytes(B, Hq, Sq))
    n, rest = divmod(extra, 128 * 2 * D * 4)
    assert rest == 0 and 0 < n <= min(B * Hkv * tiles * 16, (512 if D <= 128 else 256) * 4 // 3)


CASES = [
    # B, Hq, Hkv, Sq, Skv, D, Dv, q_offset, causal, window, softcap, dtype
    (1, 8, 1, 513, 513, 64, 64, 0, True, None, None, BF16),
    (2, 8, 2, 1000, 1000, 128, 128, 0, True, None, None, BF16),
    (1, 6, 1, 700, 700, 96, 96, 0, True, 333, 30.0, F16),
    (1, 28, 4, 385, 385, 128, 128, 0, True, None, 20.0, BF16),
    (1, 16, 1, 300, 1025, 128, 128, 725, True, None, None, BF16),
    (1, 16, 1, 640, 129, 64, 64, 0, False, None, None, BF16),   # a part's last key tile of one row
    (1, 8, 1, 800, 800, 192, 192, 0, True, None, None, BF16),
    (1, 4, 1, 900, 900, 192, 128, 0, True, None, None, BF16),   # V narrower than head_dim
    (1, 4, 1, 900, 900, 176, 72, 0, True, 500, None, F16),
    # cut key tiles that start late and end early (two KV heads: their partials are adjacent)
    (2, 16, 2, 260, 2500, 128, 128, 1900, True, 300, None, BF16),
    (1, 16, 2, 500, 3000, 64, 64, 0, True, None, 20.0, F16),
]


@pytest.mark.gpu
@pytest.mark.parametrize("B,Hq,Hkv,Sq,Skv,D,Dv,off,causal,window,softcap,dt", CASES)
def test_cut_sweeps(B, Hq, Hkv, Sq, Skv, D, Dv, off, causal, window, softcap, dt, monkeypatch):
    require_gpu()
    say(f"bwd cut B{B} {Hq}/{Hkv} Sq{Sq} Skv{Skv} D{D}/{Dv} off{off} w{window} cap{softcap} {dt}")
    lib = _lib.load()
    a = _args(B, Hq, Hkv, Sq, Skv, D, Dv if Dv < D else 0, off, int(causal), window or 0,
              _lib.dtype_code(dt))
    assert (lib.ffa_attn_bwd_split_workspace_bytes(ctypes.byref(a))
            > lib.ffa_attn_bwd_workspace_bytes(B, Hq, Sq))
    q, do = seeded((B, Hq, Sq, D), dt, 1), seeded((B, Hq, Sq, D), dt, 2)
    k, v = seeded((B, Hkv, Skv, D), dt, 3), seeded((B, Hkv, Skv, Dv), dt, 4)
    kw = dict(causal=causal, sliding_window=window, softcap=softcap, scale=1 / math.sqrt(D))
    # O and LSE of the same problem in float64
    s = torch.einsum("bhqd,bhkd->bhqk", q.double(), k.double().repeat_interleave(Hq // Hkv, 1))
    s = s * kw["scale"]
    s = softcap * torch.tanh(s / softcap) if softcap else s
    row, key = off + torch.arange(Sq)[:, None], torch.arange(Skv)[None, :]
    keep = torch.ones(Sq, Skv, dtype=torch.bool)
    keep &= (key <= row) if causal else True
    keep &= (key >= row - window + 1) if window else True
    s = s.masked_fill(~keep, float("-inf"))
    lse = torch.logsumexp(s, -1, keepdim=True)
    vp = torch.nn.functional.pad(v, (0, D - Dv))
    o = torch.einsum("bhqk,bhkd->bhqd", torch.exp(s - lse),
                     vp.double().repeat_interleave(Hq // Hkv, 1)).to(dt)
    lse = lse.float()
    args = [t.cuda() for t in (do, q, k, v, o, lse)]
    got = ffa.fastest_flash_attn_backward(*args, q_offset=off, **kw)
    again = ffa.fastest_flash_attn_backward(*args, q_offset=off, **kw)
    assert all(torch.equal(x, y) for x, y in zip(got, again))  # no order left to chance
    monkeypatch.setattr(lib, "ffa_attn_bwd_split_workspace_bytes", lambda _: 0)
    whole = ffa.fastest_flash_attn_backward(*args, q_offset=off, **kw)
    assert torch.equal(got[0], whole[0])
    for name, g, w in zip(("dk", "dv"), got[1:], whole[1:]):
        # the same fp32 terms in another order, then one rounding to 16 bits each
        eps = 2 ** -7 if dt == BF16 else 2 ** -10
        tol = eps * w.float().abs() + 1e-5 * w.float().abs().max()
        assert ((g.float() - w.float()).abs() <= tol).all(), name
    ref = rb.backward(np32(do), np32(q), np32(k), np32(vp), np32(o), np32(lse), q_offset=off, **kw)
    for name, g, r in zip(("dq", "dk", "dv"), got, ref):
        _check(g, np.asarray(r)[..., :g.size(-1)], dt, name)


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,S", [(3, 8, 512), (5, 7, 350), (4, 8, 401), (8, 8, 288)])
@pytest.mark.parametrize("causal", [True, False])
def test_fp32_workgroups_per_cu(B, H, S, causal):
    """fp32 dK/dV at head_dim 64 around its switch to two workgroups per CU (384 blocks of 32
    keys), inside the paired range (385 to 512) and past it."""
    require_gpu()
    dt = torch.float32
    say(f"fp32 dkdv blocks {B * H * math.ceil(S / 32)} causal{causal}")
    q, k, v, do = (seeded((B, H, S, 64), dt, i) for i in range(4))
    kw = dict(causal=causal, scale=0.125)
    o, lse = _oracle_forward(q, k, v, window=None, softcap=None, q_offset=0, **kw)
    args = [torch.from_numpy(np.ascontiguousarray(x)).cuda() if isinstance(x, np.ndarray) else x.cuda()
            for x in (do, q, k, v, o, lse)]
    got = ffa.fastest_flash_attn_backward(*args, **kw)
    ref = rb.backward(np32(do), np32(q), np32(k), np32(v), o, lse, **kw)
    for name, g, r in zip(("dq", "dk", "dv"), got, ref):
        _check(g, r, dt, name)
