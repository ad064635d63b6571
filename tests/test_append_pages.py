"""Appends whose page ids travel with the launch, and block tables sent in one copy."""

from __future__ import annotations

import ctypes

import pytest
import torch

import fastest_flash_attention_amd as ffa
from fastest_flash_attention_amd.kernels import _lib
from fastest_flash_attention_amd.ops.kv_cache import device_tables
from tests.gpu_util import require_gpu, say

BF16 = torch.bfloat16


def test_abi_checks():
    lib = _lib.load()
    ids = (ctypes.c_int32 * 500)(*range(500))

    def rc(**kw):
        a = _lib.PagedAppendArgs()
        base = dict(k_pages=16, v_pages=16, k_new=16, v_new=16, num_pages=9, heads_kv=1, page_size=4,
                    head_dim=8, start=3, n_tokens=6, elem_bytes=2, n_host_pages=3,
                    host_pages=ctypes.addressof(ids))
        for name, val in {**base, **kw}.items():
            setattr(a, name, val)
        return lib.ffa_paged_append(ctypes.byref(a), None)

    assert rc(host_pages=None) == -1                      # no table of either kind
    assert rc(n_host_pages=2) == -1                       # token 8 lies in a third page
    assert rc(n_host_pages=_lib.FFA_APPEND_HOST_PAGES + 1) == -1
    assert rc(n_tokens=0, n_host_pages=0) == 0


def test_device_tables_on_the_host():
    bt, lens = device_tables([[3, 1], [], [7, 8, 9]], [5, 0, 12], torch.device("cpu"))
    assert bt.dtype == lens.dtype == torch.int32 and bt.is_contiguous()
    assert bt.tolist() == [[3, 1, 0], [0, 0, 0], [7, 8, 9]] and lens.tolist() == [5, 0, 12]
    bt, lens = device_tables([], [], torch.device("cpu"))
    assert tuple(bt.shape) == (0, 1) and tuple(lens.shape) == (0,)
    bt, lens = device_tables([[]], [0], torch.device("cpu"))
    assert bt.tolist() == [[0]] and lens.tolist() == [0]


@pytest.mark.gpu
@pytest.mark.parametrize("D,dt", [(64, BF16), (6, BF16), (5, torch.float16), (3, torch.float32)])
@pytest.mark.parametrize("page", [1, 4, 48])
def test_append_matches_the_host_pool(D, dt, page):
    """Chunks of 1 token up to more pages than a launch carries, at every offset in a page."""
    require_gpu()
    say(f"append pages D{D} {dt} page{page}")
    n_pages = 1100 if page < 48 else 40
    pools = [ffa.PagedKVCache(n_pages, page, 2, D, dtype=dt, device=d) for d in ("cpu", "cuda")]
    for p in pools:
        p.free_pages = p.free_pages[::-1]
    g = torch.Generator().manual_seed(1)
    for n in (1, 3, 16 * page, 16 * page + 1, 1, 480 * page, 481 * page, 2):
        if sum(p.num_free_pages for p in pools) // 2 * page < n + page:
            continue
        k, v = (torch.randn(2, n, D, generator=g).to(dt) for _ in "kv")
        assert pools[0].append_tokens(7, k, v) == pools[1].append_tokens(7, k.cuda(), v.cuda())
    assert torch.equal(pools[0].k_pages, pools[1].k_pages.cpu())
    assert torch.equal(pools[0].v_pages, pools[1].v_pages.cpu())
    for a, b in zip(pools[0].get_kv(7), pools[1].get_kv(7)):
        assert torch.equal(a, b.cpu())


@pytest.mark.gpu
def test_tables_are_not_overwritten_while_in_flight():
    """Tables of many steps queued behind device work keep their own values."""
    require_gpu()
    big = torch.randn(4096, 4096, device="cuda")
    got = []
    for i in range(40):
        big = big @ big * 1e-4
        got.append(device_tables([[i] * (1 + i % 7), [i + 1]], [i, 2 * i], big.device))
    for i, (bt, lens) in enumerate(got):
        assert bt[0].tolist() == [i] * (1 + i % 7) and bt[1, 0].item() == i + 1
        assert lens.tolist() == [i, 2 * i]
