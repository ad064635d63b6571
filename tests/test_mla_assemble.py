"""The MLA module's fused query / key assembly and its token-major attention output."""

from __future__ import annotations

import ctypes

import pytest
import torch

import fastest_flash_attention_amd as ffa
from fastest_flash_attention_amd.kernels import _lib
from fastest_flash_attention_amd.modules import flash_mla
from fastest_flash_attention_amd.ops.attention_forward import forward_token_major
from fastest_flash_attention_amd.ops.mla_decode import mla_assemble, mla_assembles
from tests.gpu_util import require_gpu, say, seeded

BF16, F16 = torch.bfloat16, torch.float16


def test_abi_checks():
    lib = _lib.load()

    def rc(**kw):
        a = _lib.MlaAssembleArgs()
        base = dict(batch=1, heads=2, seqlen=3, head_dim=64, rope_dim=16, dtype=0, table_dtype=2,
                    q_nope_stride=128, q_rope_stride=32, kv_stride=256, k_rope_stride=16)
        for name in ("q_nope", "q_rope", "kv", "k_rope", "cos", "sin", "q", "k"):
            base[name] = 16
        for name, val in {**base, **kw}.items():
            setattr(a, name, val)
        return lib.ffa_mla_assemble(ctypes.byref(a), None)

    assert lib.ffa_mla_assemble(None, None) == -1
    assert rc(dtype=2) == -2 and rc(table_dtype=1) == -2
    assert rc(batch=-1) == -1 and rc(heads=0) == -1 and rc(cos=None) == -1 and rc(kv_stride=-8) == -1
    assert rc(head_dim=60) == -4 and rc(rope_dim=24) == -4 and rc(q=24) == -4 and rc(kv_stride=12) == -4
    assert rc(batch=0, q=None) == 0 and rc(seqlen=0) == 0


def test_cpu_and_differentiable_inputs_take_the_general_path():
    t = torch.zeros(1, 2, 64, dtype=BF16)
    assert not mla_assembles(t, t, t, t, 64, 16)          # not on a ROCm device
    m = ffa.FastestFlashMLA(64, 2, head_dim=16, latent_dim=32, rope_dim=16).to(BF16).eval()
    q, k, v = m.project_qkv(torch.randn(1, 5, 64).to(BF16))
    assert q.requires_grad and k.requires_grad and v.requires_grad


def replace_instance(m, forward, monkeypatch):
    m.forward = lambda *args: forward(m, *args)


def replace_class(m, forward, monkeypatch):
    monkeypatch.setattr(type(m), "forward", lambda self, *args: forward(self, *args))


def replace_compiled(m, forward, monkeypatch):
    m._compiled_call_impl = lambda *args: forward(m, *args)


@pytest.mark.parametrize("replace", [replace_instance, replace_class, replace_compiled])
@pytest.mark.parametrize("name", ["o_proj", "rope"])
def test_a_replaced_forward_is_called(name, replace, monkeypatch):
    """A submodule whose forward was set from outside (by a wrapper that offloads, adapts or
    quantises it) is called, also where the work of a plain one is done without the call: the
    projection from 4096 rows on, the rotary module without gradients."""
    m = ffa.FastestFlashMLA(64, 2, head_dim=128, latent_dim=32, rope_dim=64).to(BF16).eval()
    seen, fused = [], []
    monkeypatch.setattr(flash_mla, "mla_assembles", lambda *args: True)

    def assemble(q_nope, q_rope, kv, k_rope, cos, sin, heads, head_dim, rope_dim):
        fused.append("rope")
        return (q_nope.new_zeros(1, heads, q_nope.size(1), head_dim + rope_dim),) * 2

    def attend(q, k, v, drop_zero_dims=False, **kw):
        fused.extend(["o_proj"] if drop_zero_dims else [])
        return q.new_zeros(1, q.size(2), 2, 128 if drop_zero_dims else 192), None

    monkeypatch.setattr(flash_mla, "mla_assemble", assemble)
    monkeypatch.setattr(flash_mla, "forward_token_major", attend)
    x = torch.zeros(1, 4096, 64, dtype=BF16)
    with torch.no_grad():
        m(x)
        assert fused == ["rope", "o_proj"]  # a plain module
        sub = getattr(m, name)
        original = type(sub).forward
        replace(sub, lambda mod, *args: (seen.append(mod), original(mod, *args))[1], monkeypatch)
        m(x)
    assert any(mod is sub for mod in seen) and fused.count(name) == 1


def general(m, x):
    """project_qkv with the elementwise operations (the path of differentiable inputs)."""
    with torch.enable_grad():
        return [t.detach() for t in m.project_qkv(x, pad_v=False)]


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [BF16, F16])
@pytest.mark.parametrize("rope32", [False, True])
@pytest.mark.parametrize("B,S,H,hd,R", [(1, 1, 1, 128, 64), (2, 77, 3, 128, 64), (1, 300, 2, 8, 16),
                                        (3, 33, 5, 72, 48), (1, 5000, 1, 64, 32)])
def test_same_bits_as_the_elementwise_operations(dt, rope32, B, S, H, hd, R):
    require_gpu()
    say(f"mla assemble B{B} S{S} H{H} hd{hd} R{R} {dt} rope32={rope32}")
    torch.manual_seed(0)
    m = ffa.FastestFlashMLA(96, H, head_dim=hd, latent_dim=64, rope_dim=R).cuda().to(dt).eval()
    if rope32:
        m.rope = flash_mla.RotaryEmbedding(R).cuda()
    x = seeded((B, S, 96), dt, 5).cuda()
    want = general(m, x)
    with torch.no_grad():
        raw = (m.q_proj(x), m.q_rope_proj(x), m.kv_up_proj(m.kv_down_proj(x)), m.k_rope_proj(x))
        assert mla_assembles(*raw, hd, R)
        got = m.project_qkv(x, pad_v=False)
    for g, w in zip(got, want):
        assert g.shape == w.shape and torch.equal(g, w)


@pytest.mark.gpu
def test_infinities_and_signed_zeros_pass_through():
    require_gpu()
    dt, B, S, H, hd, R = F16, 1, 4, 2, 8, 16
    raw = [seeded((B, S, n), dt, i).cuda() for i, n in enumerate((H * hd, H * R, H * 2 * hd, R))]
    for t in raw:
        t.view(-1)[0], t.view(-1)[1], t.view(-1)[2] = float("inf"), float("nan"), -0.0
    rope = flash_mla.RotaryEmbedding(R).cuda()
    q, k = mla_assemble(*raw, *rope.tables(raw[0]), H, hd, R)
    qw = torch.cat([raw[0].view(B, S, H, hd).transpose(1, 2),
                    rope(raw[1].view(B, S, H, R).transpose(1, 2))], dim=-1)
    kw = torch.cat([raw[2].view(B, S, H, 2 * hd).transpose(1, 2)[..., :hd],
                    rope(raw[3].unsqueeze(1).expand(-1, H, -1, -1))], dim=-1)
    assert torch.equal(q.nan_to_num(7.0), qw.nan_to_num(7.0))
    assert torch.equal(k.nan_to_num(7.0), kw.nan_to_num(7.0))


@pytest.mark.gpu
@pytest.mark.parametrize("S", [1, 130, 4097])
@pytest.mark.parametrize("D,Dv,H", [(192, 128, 3), (136, 8, 2), (192, 192, 2), (64, 64, 2), (20, 20, 2)])
def test_token_major_output(S, D, Dv, H):
    require_gpu()
    say(f"token major S{S} D{D} Dv{Dv}")
    q, k, v = (seeded((1, H, S, d), BF16, i).cuda() for i, d in enumerate((D, D, Dv)))
    want, lw = ffa.fastest_flash_attn_forward(q, k, v, causal=True, return_lse=True)
    want = want.transpose(1, 2)
    got, lg = forward_token_major(q, k, v, causal=True, return_lse=True)
    assert got.is_contiguous() and torch.equal(got, want) and torch.equal(lg, lw)
    got, _ = forward_token_major(q, k, v, causal=True, drop_zero_dims=True)
    assert torch.equal(got, want[..., :got.size(-1)]) and not want[..., got.size(-1):].any()


@pytest.mark.gpu
@pytest.mark.parametrize("B,S", [(1, 4095), (1, 4096), (2, 2100)])
def test_o_proj_without_the_zero_columns(B, S):
    """From 4096 rows on the output projection skips the columns that meet V's padding: the
    same sums (in another order) as the whole product; a hooked projection is called as it
    is."""
    require_gpu()
    say(f"o_proj B{B} S{S}")
    torch.manual_seed(1)
    m = ffa.FastestFlashMLA(128, 2, head_dim=128, latent_dim=64, rope_dim=64).cuda().to(BF16).eval()
    x = seeded((B, S, 128), BF16, 3).cuda()
    calls = []
    with torch.no_grad():
        got = m(x)
        hook = m.o_proj.register_forward_pre_hook(lambda mod, args: calls.append(args[0].shape))
        whole = m(x)
        hook.remove()
    assert calls == [(B, S, 2 * 192)]
    # bf16 outputs of one fp32 sum: at most a rounding of the last bit apart
    assert (got - whole).abs().max() <= 2 ** -7 * whole.abs().max()


def test_rope_tables_abi_checks():
    lib = _lib.load()

    def rc(**kw):
        a = _lib.RopeTablesArgs()
        base = dict(inv_freq=16, cos=16, sin=16, seqlen=3, half=4, dtype=0, table_dtype=0)
        for name, val in {**base, **kw}.items():
            setattr(a, name, val)
        return lib.ffa_rope_tables(ctypes.byref(a), None)

    assert lib.ffa_rope_tables(None, None) == -1
    assert rc(dtype=2) == -2 and rc(table_dtype=1) == -2
    assert rc(seqlen=-1) == -1 and rc(half=0) == -1 and rc(sin=None) == -1
    assert rc(cos=17) == -4 and rc(table_dtype=2, sin=18) == -4
    assert rc(seqlen=0, cos=None) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [BF16, F16])
@pytest.mark.parametrize("table", [torch.float32, None])
@pytest.mark.parametrize("S,R", [(1, 16), (77, 48), (4096, 64), (70000, 32)])
def test_rope_tables_are_the_elementwise_ones(dt, table, S, R):
    """Positions past fp16's range become infinities, and their tables NaN, in both."""
    require_gpu()
    say(f"rope tables S{S} R{R} {dt} {table}")
    rope = flash_mla.RotaryEmbedding(R).cuda().to(table or dt)
    x = torch.empty(1, S, 8, dtype=dt, device="cuda")
    freqs = torch.outer(torch.arange(S, device="cuda", dtype=dt), rope.inv_freq)
    for got, want in zip(rope.tables(x), (freqs.cos(), freqs.sin())):
        assert got.dtype == want.dtype and got.is_contiguous()
        assert torch.equal(got.isnan(), want.isnan())
        assert torch.equal(got.nan_to_num(7.0), want.nan_to_num(7.0))


@pytest.mark.gpu
def test_rotary_of_another_width_keeps_the_general_path():
    """A replaced rotary module whose tables have another width is not read by the kernel."""
    require_gpu()
    torch.manual_seed(0)
    m = ffa.FastestFlashMLA(64, 2, head_dim=16, latent_dim=32, rope_dim=32).cuda().to(BF16).eval()
    m.rope = flash_mla.RotaryEmbedding(16).cuda().to(BF16)
    x = seeded((1, 40, 64), BF16, 2).cuda()
    with torch.no_grad():
        with pytest.raises(ValueError):
            mla_assemble(m.q_proj(x), m.q_rope_proj(x), m.kv_up_proj(m.kv_down_proj(x)),
                         m.k_rope_proj(x), *m.rope.tables(x), 2, 16, 32)
        got = m.project_qkv(x, pad_v=False)
    for g, w in zip(got, general(m, x)):
        assert torch.equal(g, w)


@pytest.mark.gpu
def test_autocast_builds_the_tables_in_the_projections_dtype():
    """fp32 input and weights under autocast: bf16 projections, whose positions past 256 round
    as the elementwise operations round them."""
    require_gpu()
    torch.manual_seed(0)
    m = ffa.FastestFlashMLA(96, 2, head_dim=128, latent_dim=64, rope_dim=64).cuda().eval()
    x = seeded((2, 700, 96), torch.float32, 5).cuda()
    with torch.autocast("cuda", dtype=BF16):
        want = general(m, x)
        with torch.no_grad():
            got = m.project_qkv(x, pad_v=False)
    for g, w in zip(got, want):
        assert g.dtype == w.dtype == BF16 and torch.equal(g, w)


@pytest.mark.gpu
def test_double_or_learned_frequencies_keep_the_general_path():
    """The kernel takes tables of the projections' dtype or fp32, and gives no gradient."""
    require_gpu()
    torch.manual_seed(0)
    m = ffa.FastestFlashMLA(64, 2, head_dim=16, latent_dim=32, rope_dim=16).cuda().to(BF16).eval()
    m.requires_grad_(False)
    x = seeded((1, 40, 64), BF16, 2).cuda()
    m.rope = flash_mla.RotaryEmbedding(16).cuda().double()
    want_q = torch.cat([m.q_proj(x).view(1, 40, 2, 16).transpose(1, 2),
                        m.rope(m.q_rope_proj(x).view(1, 40, 2, 16).transpose(1, 2))], dim=-1)
    assert torch.equal(m.project_qkv(x, pad_v=False)[0], want_q)
    m.rope = flash_mla.RotaryEmbedding(16).cuda()
    m.rope.inv_freq.requires_grad_()
    q, k, v = m.project_qkv(x, pad_v=False)
    assert q.requires_grad and k.requires_grad and not v.requires_grad
