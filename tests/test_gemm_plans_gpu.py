"""The tiles and K ranges unok_gemm_nt_ws chooses between (256x256, 128x256, 128x128, 64 rows x all
columns; one or several ranges) against fp32 torch products of the same operands, at tile edges and
remainders, with strided operands, LoRA segments, row gate, residual and both output types.

Tolerances: a bf16 result is one rounding (2^-9 relative) of an fp32 sum, so its 2-norm error is below
2^-9 of the result's plus what cancels against a residual; fp32 sums of at most 2^13 products of unit
variance keep 1e-5."""
import pytest
import torch

from uno_amd import _native as N
from uno_amd import kernels as K

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return ((a.float() - b.float()).norm() / b.float().norm().clamp_min(1e-30)).item()


def _call(plan, a, b, a2, b2, segs, out, res, gate, alpha, ranges):
    M, Kd = a.shape
    Nn = b.shape[0]
    ws = torch.full((ranges * M * Nn,), float("nan"), device=a.device) if ranges > 1 else None
    N.call("unok_gemm_nt_ws", N.BF16, N.dtype_code(out.dtype), M, Nn, Kd, N.ptr(a), a.stride(0), N.ptr(b), b.stride(0),
           N.ptr(a2), a2.stride(0) if a2 is not None else 0, N.ptr(b2), b2.stride(0) if b2 is not None else 0,
           b2.shape[1] if b2 is not None else 0, len(segs), N.int_array([s[0] for s in segs]),
           N.int_array([s[1] for s in segs]), N.ptr(out), out.stride(0), N.ptr(res), res.stride(0) if res is not None else 0,
           N.ptr(gate), alpha, plan, N.ptr(ws), ws.numel() * 4 if ws is not None else 0, N.stream())


@pytest.mark.parametrize("M,Nn,Kd", [(1, 256, 64), (127, 256, 320), (129, 520, 256), (257, 1028, 448), (640, 512, 1024)])
@pytest.mark.parametrize("tile", [1, 2, 3])
@pytest.mark.parametrize("ranges", [1, 3])
def test_tiles_and_ranges(dev, M, Nn, Kd, tile, ranges):
    if ranges > Kd // 64:
        ranges = Kd // 64
    torch.manual_seed(M + Nn + Kd)
    a = torch.randn(M, Kd + 64, device=dev).bfloat16()[:, 64:]           # row stride > K
    b = torch.randn(Nn, Kd + 8, device=dev).bfloat16()[:, :Kd]
    gate = torch.rand(M, device=dev) > 0.3
    ref = (a.float() @ b.float().T) * gate.float()[:, None] * 0.5
    res = torch.randn(M, Nn + 4, device=dev)[:, :Nn]
    for dt, tol in ((torch.float32, 1e-5), (torch.bfloat16, 2.0 ** -8)):
        out = torch.full((M, Nn), float("nan"), device=dev, dtype=dt)
        _call(tile + 16 * ranges, a, b, None, None, [], out, None, gate, 0.5, ranges)
        assert _rel(out, ref) < tol, dt
        r = res.to(dt)
        out = torch.full((M, Nn), float("nan"), device=dev, dtype=dt)
        _call(tile + 16 * ranges, a, b, None, None, [], out, r, None, 1.0, ranges)
        assert _rel(out, a.float() @ b.float().T + r.float()) < tol, dt


@pytest.mark.parametrize("tile,ends", [(1, [256, 512, 768]), (2, [512, 768, 1024]), (3, [128, 384, 512])])
@pytest.mark.parametrize("K2", [32, 64, 96])
@pytest.mark.parametrize("ranges", [1, 2, 5])
def test_extension_segments(dev, tile, ends, K2, ranges):
    """The LoRA extension belongs to the last range; an extension of zeros changes no bit."""
    torch.manual_seed(K2 + ranges)
    M, Kd, Nn = 300, 320, ends[-1]
    a, b = torch.randn(M, Kd, device=dev).bfloat16(), torch.randn(Nn, Kd, device=dev).bfloat16()
    h, bl = torch.randn(M, 3 * K2, device=dev).bfloat16(), torch.randn(Nn, K2, device=dev).bfloat16()
    segs = [(e, j * K2) for j, e in enumerate(ends)]
    ref, lo = a.float() @ b.float().T, 0
    plain, zeros = torch.empty(M, Nn, device=dev), torch.empty(M, Nn, device=dev)
    for e, c in segs:
        ref[:, lo:e] += h[:, c:c + K2].float() @ bl[lo:e].float().T
        lo = e
    out = torch.empty(M, Nn, device=dev)
    _call(tile + 16 * ranges, a, b, h, bl, segs, out, None, None, 1.0, ranges)
    assert _rel(out, ref) < 1e-5
    _call(tile + 16 * ranges, a, b, None, None, [], plain, None, None, 1.0, ranges)
    _call(tile + 16 * ranges, a, b, torch.zeros_like(h), bl, segs, zeros, None, None, 1.0, ranges)
    assert torch.equal(plain, zeros)


@pytest.mark.parametrize("M,Nn", [(1, 4), (63, 64), (65, 100), (200, 192)])
@pytest.mark.parametrize("ranges", [1, 2, 7])
def test_skinny_ranges(dev, M, Nn, ranges):
    torch.manual_seed(M + Nn)
    a, b = torch.randn(M, 512, device=dev).bfloat16(), torch.randn(Nn, 512, device=dev).bfloat16()
    gate = torch.rand(M, device=dev) > 0.3
    out = torch.full((M, Nn), float("nan"), device=dev)
    _call(4 + 16 * ranges, a, b, None, None, [], out, None, gate, 0.75, ranges)
    assert _rel(out, 0.75 * (a.float() @ b.float().T) * gate.float()[:, None]) < 1e-5 or not gate.any()


@pytest.mark.parametrize("M,Nn,Kd", [(777, 4096, 4096), (64, 4096, 12288), (300, 64, 4096), (100, 1026, 2048),
                                     (130, 640, 200), (2100, 320, 8192)])
def test_chosen_plan_against_the_default_entry(dev, M, Nn, Kd):
    """gemm_nt's own choice (K ranges where they pay; the register-staged kernel for a K or N no tile
    takes) against fp32 and against the entry point without a workspace, which never splits K."""
    torch.manual_seed(M)
    a, b = torch.randn(M, Kd, device=dev).bfloat16(), torch.randn(Nn, Kd, device=dev).bfloat16()
    ref = a.float() @ b.float().T
    out = K.gemm_nt(a, b, out_dtype=torch.float32)
    one = torch.empty(M, Nn, device=dev)
    N.call("unok_gemm_nt", N.BF16, N.F32, M, Nn, Kd, N.ptr(a), Kd, N.ptr(b), Kd, None, 0, None, 0, 0, 0, None, None,
           N.ptr(one), Nn, None, 0, None, 1.0, N.stream())
    assert _rel(out, ref) < 1e-5 and _rel(one, ref) < 1e-5
    assert torch.equal(out, K.gemm_nt(a, b, out_dtype=torch.float32))


def test_plan_rejects_what_a_tile_does_not_take(dev):
    a, b = torch.randn(64, 200, device=dev).bfloat16(), torch.randn(256, 200, device=dev).bfloat16()
    out = torch.empty(64, 256, device=dev)
    with pytest.raises(ValueError, match="plan"):
        _call(1 + 16, a, b, None, None, [], out, None, None, 1.0, 1)       # K = 200 is no multiple of 64
    a, b = torch.randn(64, 256, device=dev).bfloat16(), torch.randn(256, 256, device=dev).bfloat16()
    with pytest.raises(ValueError, match="plan"):
        _call(4 + 16, a, b, None, None, [], out, None, None, 1.0, 1)       # 256 columns are not skinny
    with pytest.raises(ValueError, match="plan"):
        _call(1 + 16 * 2, a, b, None, None, [], out, None, None, 1.0, 1)   # ranges without a workspace
