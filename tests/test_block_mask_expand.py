"""The block-mask expansion kernel against its elementwise statement on the CPU."""

from __future__ import annotations

import ctypes
import math

import pytest
import torch

from fastest_flash_attention_amd.kernels import _lib
from fastest_flash_attention_amd.ops.attention_forward import (
    _expand_block_mask,
    resolve_forward_args,
)
from tests.gpu_util import require_gpu, say


def test_abi_checks():
    lib = _lib.load()

    def rc(**kw):
        a = _lib.BlockMaskArgs()
        base = dict(mask=1, key_mask=8, visited=4, mask_stride=1, words=1, seqlen_q=1, seqlen_kv=64,
                    block_q=64, block_kv=64)
        for name, val in {**base, **kw}.items():
            setattr(a, name, val)
        return lib.ffa_block_mask_expand(ctypes.byref(a), None)

    assert lib.ffa_block_mask_expand(None, None) == -1
    for bad in (dict(words=0), dict(seqlen_kv=65), dict(block_q=0), dict(block_kv=0), dict(mask=None),
                dict(key_mask=None), dict(visited=None), dict(seqlen_q=-1), dict(mask_stride=-1)):
        assert rc(**bad) == -1, bad
    assert rc(key_mask=12) == -4
    assert rc(block_q=1 << 30) == -9
    assert rc(seqlen_q=0, key_mask=None) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("S_q,S_kv,bs", [(1, 1, 1), (37, 130, 7), (200, 200, 16), (200, 333, 48),
                                         (130, 64, 64), (257, 2049, 64), (100, 20000, 64),
                                         (300, 700, 100), (129, 513, 128), (50, 60, 1 << 20),
                                         (40, 0, 16)])
@pytest.mark.parametrize("causal,window", [(False, None), (True, None), (True, 90), (False, 1 << 40)])
def test_same_as_the_elementwise_form(S_q, S_kv, bs, causal, window):
    require_gpu()
    say(f"mask expand Sq{S_q} Skv{S_kv} bs{bs} causal{causal} w{window}")
    g = torch.Generator().manual_seed(S_q * 7 + S_kv)
    q, k = torch.zeros(1, 1, S_q, 8), torch.zeros(1, 1, S_kv, 8)
    n_br, n_bc = math.ceil(S_q / bs), math.ceil(S_kv / bs)
    bm = torch.rand(n_br + 1, n_bc + 2, generator=g) < 0.5  # a mask may cover more
    r = resolve_forward_args(q, k, k, causal=causal, sliding_window=window, block_size=bs,
                             block_mask=bm)
    want, words, wv = _expand_block_mask(bm, r, torch.device("cpu"))
    device = torch.device("cuda", torch.cuda.current_device())
    for form in (bm, bm.cuda(), bm.t().contiguous().t().cuda(), bm.to(torch.float32), bm.numpy()):
        got, gw, gv = _expand_block_mask(form, r, device)
        assert gw == words and torch.equal(got.cpu(), want) and torch.equal(gv.cpu(), wv)


@pytest.mark.gpu
@pytest.mark.parametrize("S_kv,bkv,words", [(130, 100, 4), (64, 48, 3), (130, 64, 5), (65, 200, 300)])
def test_words_past_the_last_key_are_clear(S_kv, bkv, words):
    """The C entry takes more words than the keys need; the last tile, which may end in one of
    them, sets no bit there."""
    require_gpu()
    say(f"mask words Skv{S_kv} bkv{bkv} words{words}")
    n_bc = math.ceil(S_kv / bkv)
    mask = torch.ones(2, n_bc, dtype=torch.bool, device="cuda")
    bits = torch.full((2, words), -1, dtype=torch.int64, device="cuda")
    visited = torch.empty(2, dtype=torch.int32, device="cuda")
    a = _lib.BlockMaskArgs()
    a.mask, a.key_mask, a.visited = mask.data_ptr(), bits.data_ptr(), visited.data_ptr()
    a.mask_stride, a.words, a.seqlen_q, a.seqlen_kv = n_bc, words, 20, S_kv
    a.block_q, a.block_kv = 16, bkv
    _lib.launch(_lib.load().ffa_block_mask_expand, a, mask.device)
    keys = torch.arange(words * 64).view(words, 64) < S_kv
    want = (keys.to(torch.int64) << torch.arange(64)).sum(-1)
    assert torch.equal(bits.cpu(), want.expand(2, -1)) and visited.tolist() == [n_bc, n_bc]


@pytest.mark.gpu
def test_a_pinned_mask_may_change_after_the_call():
    require_gpu()
    big = torch.randn(4096, 4096, device="cuda")
    device = big.device
    q = torch.zeros(1, 1, 640, 8)
    bm = torch.ones(10, 10, dtype=torch.bool).pin_memory()
    r = resolve_forward_args(q, q, q, block_size=64, block_mask=bm)
    want, _, wv = _expand_block_mask(bm, r, torch.device("cpu"))
    for _ in range(30):  # work queued ahead of the copy
        big = big @ big * 1e-4
    got, _, gv = _expand_block_mask(bm, r, device)
    bm.zero_()
    assert torch.equal(got.cpu(), want) and torch.equal(gv.cpu(), wv)
