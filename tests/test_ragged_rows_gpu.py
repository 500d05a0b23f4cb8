"""Row counts that are no multiple of 256: the q|k|v epilogue's fp32 pre-norm columns (which the separate
projection and norm kernels keep there too) and the attention backward that reads them."""
import pytest
import torch

from uno_amd import kernels as K
from uno_amd import layers as Lyr
from uno_amd.model import UnoQwen3Config, UnoQwen3ForCausalLM, bd_prepare
from uno_amd.training.config import LoraSettings
from uno_amd.training.lora import create_lora_model

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return ((a.float() - b.float()).norm() / b.float().norm().clamp_min(1e-30)).item()


def _context(dev, B, L, d, theta=1e6):
    g = torch.Generator().manual_seed(B + L)
    ids = torch.randint(0, 500, (B, L), generator=g).to(dev)
    pos = torch.arange(L)[None].repeat(B, 1).to(dev)
    prompt = torch.zeros(B, L, dtype=torch.bool, device=dev)
    prompt[:, :9] = True
    mask = bd_prepare(ids, pos, prompt, block_size=8, mask_token_id=511)[2]
    inv = (1.0 / (theta ** (torch.arange(0, d, 2, dtype=torch.int64).float() / d))).to(dev)
    sc = Lyr.StreamContext(mask.pos_stream, inv, mask.iv_noisy, mask.iv_clean, [], [])
    sc.rope_cos, sc.rope_sin = K.rope_table(L, inv)
    return sc


@pytest.mark.parametrize("B,L,dtype", [(3, 131, torch.float32), (1, 255, torch.float32), (1, 257, torch.float32),
                                       (2, 256, torch.bfloat16)])
@pytest.mark.parametrize("norm", [True, False])
def test_layer_keeps_the_projection_in_fp32(dev, B, L, dtype, norm):
    """The pre-norm q/k columns a bf16 layer keeps for its backward: at ragged row counts bit for bit
    the fp32 projection output's, at whole tiles their bf16 rounding."""
    cfg = UnoQwen3Config(vocab_size=512, hidden_size=256, intermediate_size=512, num_hidden_layers=1,
                         num_attention_heads=4, num_key_value_heads=2, head_dim=128, qk_norm=norm, block_size=8)
    model = UnoQwen3ForCausalLM(cfg, device=dev, dtype=torch.bfloat16)
    model.random_init(1)
    lm, _ = create_lora_model(model, LoraSettings("all", 32, 64, 0.0))
    g, lora, lw = model.model.geo, model.model._uno_lora, model.model.layers[0].weights()
    sc = _context(dev, B, L, g.d)
    torch.manual_seed(L)
    h0 = torch.randn(B * L, g.H, device=dev).bfloat16()
    _, k, v = Lyr.clean_layer(h0, lw, g, sc)
    sc.clean_k.append(k)
    sc.clean_v.append(v)
    _, bufs = Lyr.noisy_layer_forward(h0, lw, lora, 0, g, sc)
    pre, end = bufs[4], g.q + g.kv
    x1, _ = K.rmsnorm_fwd(h0, lw.ln_in, g.eps)
    full = K.gemm_nt(x1, lw.w_qkv, a2=K.gemm_nt(x1, lora.a_c(0, "qkv")), b2=lora.sb_c(0, "qkv"),
                     segments=[(g.q, 0), (end, 32), (end + g.kv, 64)], out_dtype=torch.float32)
    assert pre.dtype == dtype and tuple(pre.shape) == (B * L, end)
    assert torch.equal(pre, full[:, :end].to(dtype))


@pytest.mark.parametrize("D,Hq,Hkv,norm", [(128, 8, 2, True), (128, 4, 4, False), (64, 4, 2, True)])
def test_attention_backward_reads_fp32_pre_norm_columns(dev, D, Hq, Hkv, norm):
    """The q/k-norm + RoPE backward in the dQ and dK/dV epilogues from fp32 pre-norm columns against the
    two-kernel path from the same columns: dV bit-identical, the q and k blocks within a bf16 step."""
    torch.manual_seed(17)
    B, L, bf = 3, 101, torch.bfloat16
    M, e = B * L, (Hq + Hkv) * D
    sc = _context(dev, B, L, D)
    q, do = (torch.randn(M, Hq * D, device=dev).to(bf) for _ in range(2))
    kc, vc, kn, vn = (torch.randn(M, Hkv * D, device=dev).to(bf) for _ in range(4))
    o, lse = K.attn_fwd(q, kc, vc, sc.iv_noisy, Hq, Hkv, D, k2=kn, v2=vn)
    pre = torch.randn(M, e, device=dev)
    wq, wk = ((1 + 0.1 * torch.randn(D, device=dev)).to(bf) if norm else None for _ in range(2))
    rstd = torch.rsqrt(pre.view(M, Hq + Hkv, D).pow(2).mean(-1) + 1e-6).contiguous()
    fused, ref = (torch.zeros(M, e + Hkv * D, device=dev, dtype=bf) for _ in range(2))
    K.attn_bwd_qknorm(q, kc, vc, sc.iv_noisy, o, lse, do, Hq, Hkv, D, kn, vn, pre, rstd, wq, wk, sc.pos, sc.rope_cos,
                      sc.rope_sin, fused)
    dk = torch.empty(M, Hkv * D, device=dev)
    dq = K.attn_bwd(q, kc, vc, sc.iv_noisy, o, lse, do, Hq, Hkv, D, k2=kn, v2=vn, ivk=sc.iv_noisy, dk=dk, dv=ref[:, e:],
                    grad_dtype=torch.float32)
    K.qknorm_rope_bwd(dq, dk, pre, Hq, Hkv, D, wq, wk, sc.pos, sc.inv_freq, rstd, ref)
    assert torch.equal(fused[:, e:], ref[:, e:])
    diff, mag = (fused[:, :e].float() - ref[:, :e].float()).abs(), ref[:, :e].float().abs()
    assert _rel(fused[:, :e], ref[:, :e]) < 2e-3
    assert bool((diff <= mag.clamp_min(mag.max() * 2 ** -8) * 2 ** -7).all())


def test_fused_products_refuse_mismatched_operands(dev):
    """What the separate products refuse, the fused ones refuse too: dtypes and sizes of weights, norm
    weights, extension operands and outputs."""
    bf, M, H, F, nq, nk, r = torch.bfloat16, 70, 128, 256, 4, 2, 32
    n = 128 * (nq + 2 * nk)
    z = lambda *s, dtype=bf: torch.zeros(*s, device=dev, dtype=dtype)
    x, wqkv, wn = z(M, H), z(n, H), z(128)
    pos = torch.zeros(M, device=dev, dtype=torch.int64)
    cos, sin = K.rope_table(4, torch.ones(64, device=dev))
    qkv = lambda x=x, w=wqkv, wq=wn, **kw: K.gemm_nt_qkv_rope(x, w, nq, nk, wq, wn, pos, cos, sin, 1e-6, any_rows=True, **kw)
    qkv()
    ext = lambda a, b: dict(a2=a, b2=b, segments=[(128 * nq, 0), (128 * (nq + nk), r), (n, 2 * r)])
    qkv(**ext(z(M, 3 * r), z(n, r)))
    for bad in (lambda: qkv(w=wqkv.float()), lambda: qkv(wq=wn.float()), lambda: qkv(wq=z(64)),
                lambda: qkv(**ext(z(M, 3 * r, dtype=torch.float32), z(n, r))),
                lambda: qkv(**ext(z(M, 3 * r), z(n, r, dtype=torch.float32))),
                lambda: qkv(**ext(z(M - 1, 3 * r), z(n, r))), lambda: qkv(**ext(z(M, 3 * r), z(n - 8, r)))):
        with pytest.raises(RuntimeError, match="gemm_nt_qkv_rope"):
            bad()
    w, h, b2 = z(2 * F, H), z(M, 2 * r), z(2 * F, 2 * r)
    up = lambda **kw: K.gemm_nt_swiglu(x, w, any_rows=True, plain_rows=True, **kw)
    up(a2=h, b2_interleaved=b2)
    for kw in (dict(a2=h.float(), b2_interleaved=b2), dict(a2=h, b2_interleaved=b2.float()), dict(out=z(M, F - 8)),
               dict(out=z(M, F, dtype=torch.float32))):
        with pytest.raises(RuntimeError, match="gemm_nt_swiglu"):
            up(**kw)
    gu, wd, h, b2 = z(M, 2 * F), z(F, H), z(M, r), z(F, r)
    down = lambda b=wd, a2=h, b2=b2, gu=gu, **kw: K.gemm_nt_swiglu_bwd(x, b, a2, b2, gu, any_rows=True, **kw)
    down()
    for kw in (dict(b=wd.float()), dict(a2=h.float()), dict(b2=b2.float()), dict(gu=gu.float()), dict(dgu=z(M, F))):
        with pytest.raises(RuntimeError, match="gemm_nt_swiglu_bwd"):
            down(**kw)
