"""The fp32 products and attention (parity mode) against 64-bit torch results at tile edges, remainders
and unaligned operands.

Tolerance: every result is an fp32 sum of K exact-product terms in some order, whose 2-norm error is
below K 2^-24 of the sum of magnitudes and in practice near sqrt(K) 2^-24; 2e-6 covers K = 4096 with
operands of either sign, and softmax adds a few ulp of exp2."""
import pytest
import torch

from uno_amd import kernels as K

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return ((a.double() - b).norm() / b.norm().clamp_min(1e-300)).item()


@pytest.mark.parametrize("M,N,Kd", [(1, 1, 1), (33, 8, 16), (512, 256, 256), (31, 65, 37), (230, 256, 4096), (64, 96, 1028),
                                    # 64x64 tiles for a short K over many outputs; 32x32 ones from K = 256 there
                                    (700, 2100, 8), (1001, 1300, 33), (1001, 1300, 256)])
@pytest.mark.parametrize("offset", [0, 1])
def test_nt_f32(dev, M, N, Kd, offset):
    """offset 1: operands that start 4 bytes past 16-byte alignment (element loads)."""
    print(f"[f32 nt] {M}x{N}x{Kd} offset {offset}", flush=True)
    torch.manual_seed(M + N + Kd)
    take = lambda r, c: torch.randn(r * c + 1, device=dev)[offset:offset + r * c].view(r, c)  # noqa: E731
    a, b, res = take(M, Kd), take(N, Kd), take(M, N)
    gate = torch.rand(M, device=dev) > 0.3
    out = K.gemm_nt(a, b, residual=res, gate=gate)
    ref = (a.double() @ b.double().T) * gate[:, None] + res.double()
    assert _rel(out, ref) < 2e-6
    assert torch.equal(out, K.gemm_nt(a, b, residual=res, gate=gate))


@pytest.mark.parametrize("r", [3, 8, 16, 40])
def test_nt_f32_segments(dev, r):
    """LoRA extension with three column segments; r = 3 takes element loads."""
    torch.manual_seed(r)
    M, Kd, segs = 77, 256, [(128, 0), (192, r), (256, 2 * r)]
    a, b = torch.randn(M, Kd, device=dev), torch.randn(256, Kd, device=dev)
    a2, b2 = torch.randn(M, 3 * r, device=dev), torch.randn(256, r, device=dev)
    ref, lo = a.double() @ b.double().T, 0
    for end, col in segs:
        ref[:, lo:end] += a2[:, col:col + r].double() @ b2[lo:end].double().T
        lo = end
    assert _rel(K.gemm_nt(a, b, a2=a2, b2=b2, segments=segs), ref) < 2e-6


@pytest.mark.parametrize("Mr,P,Q", [(512, 256, 8), (512, 8, 256), (1, 1, 1), (257, 65, 24), (700, 17, 70), (64, 100, 100),
                                    # both sides of the line to 64x64 tiles (320 of them, 36 (rows - 10), 64 rows)
                                    (1, 1000, 1290), (1, 1000, 1270), (33, 2040, 1700), (33, 2040, 1600), (64, 3840, 2100),
                                    (65, 3840, 2100)])
@pytest.mark.parametrize("offset", [0, 1])
def test_tn_f32(dev, Mr, P, Q, offset):
    print(f"[f32 tn] {Mr} {P}x{Q} offset {offset}", flush=True)
    torch.manual_seed(Mr + P)
    take = lambda r, c: torch.randn(r * c + 1, device=dev)[offset:offset + r * c].view(r, c)  # noqa: E731
    a, b = take(Mr, P), take(Mr, Q)
    out = torch.randn(P, Q, device=dev)
    ref = 0.5 * (a.double().T @ b.double()) + out.double()
    K.gemm_tn(a, b, out=out, alpha=0.5, beta=1.0)
    assert _rel(out, ref) < 2e-6


@pytest.mark.parametrize("D,Hq,Hkv", [(64, 4, 2), (128, 2, 2), (32, 2, 1)])
def test_attention_f32_rows(dev, D, Hq, Hkv):
    """Row intervals of 0 to 200 keys of the first source (over three rounds of 64) and 0 to 70 of the
    second, forward and dQ; head dim 32 stays on the one-key-at-a-time kernels."""
    print(f"[f32 attention] D={D}", flush=True)
    torch.manual_seed(D)
    M, Mk = 67, 200
    q, do = torch.randn(M, Hq * D, device=dev), torch.randn(M, Hq * D, device=dev)
    k1, v1 = torch.randn(Mk, Hkv * D, device=dev), torch.randn(Mk, Hkv * D, device=dev)
    k2, v2 = torch.randn(M, Hkv * D, device=dev), torch.randn(M, Hkv * D, device=dev)
    iv = torch.zeros(M, 8, dtype=torch.int32, device=dev)
    iv[:, 1] = torch.arange(M, device=dev) * 3
    iv[:, 0] = torch.minimum(torch.arange(M, device=dev), iv[:, 1])
    iv[:, 3] = torch.where(torch.arange(M, device=dev) % 3 == 1, M, 0)
    iv[0, 1], iv[0, 3] = 0, 0                                # a row without keys
    iv[5, 0], iv[5, 1] = 0, Mk
    iv[:, 5] = 0                                             # key side unused
    o, lse = K.attn_fwd(q, k1, v1, iv, Hq, Hkv, D, k2=k2, v2=v2)
    qd = q.double().view(M, Hq, D).requires_grad_(True)
    kk = torch.cat((k1, k2)).double().view(-1, Hkv, D).repeat_interleave(Hq // Hkv, 1)
    vv = torch.cat((v1, v2)).double().view(-1, Hkv, D).repeat_interleave(Hq // Hkv, 1)
    j = torch.arange(Mk + M, device=dev)[None, :]
    mask = ((j >= iv[:, :1]) & (j < iv[:, 1:2]) & (j < Mk)) | ((j - Mk >= iv[:, 2:3]) & (j - Mk < iv[:, 3:4]) & (j >= Mk))
    s = torch.einsum("mhd,khd->hmk", qd, kk) * D ** -0.5
    s = s.masked_fill(~mask, float("-inf"))
    p = torch.where(mask.any(1)[None, :, None], torch.softmax(s, -1), torch.zeros((), dtype=s.dtype, device=dev))
    ref = torch.einsum("hmk,khd->mhd", p.nan_to_num(0.0), vv)
    assert _rel(o.view(M, Hq, D), ref) < 2e-6
    seen = mask.any(1)
    (ref[seen] * do.double().view(M, Hq, D)[seen]).sum().backward()
    dq = K.attn_bwd(q, k1, v1, iv, o, lse, do, Hq, Hkv, D, k2=k2, v2=v2)
    dq = dq[0] if isinstance(dq, tuple) else dq
    want = qd.grad.nan_to_num(0.0)
    assert _rel(dq.view(M, Hq, D)[seen], want[seen]) < 4e-6
    assert bool((dq[0] == 0).all())
