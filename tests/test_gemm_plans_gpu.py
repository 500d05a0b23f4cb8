"""The tiles and K ranges unok_gemm_nt_ws chooses between (256x256, 192x256, 128x256, 128x128, 64 rows x all
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
@pytest.mark.parametrize("tile", [1, 2, 3, 6])
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


@pytest.mark.parametrize("tile,ends", [(1, [256, 512, 768]), (2, [512, 768, 1024]), (3, [128, 384, 512]),
                                       (6, [256, 512, 768])])
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


@pytest.mark.parametrize("M", [1, 100, 129, 300, 511, 2100])
@pytest.mark.parametrize("F,Kd,r", [(256, 128, 32), (1536, 512, 64)])
def test_fused_epilogues_on_any_row_count(dev, M, F, Kd, r):
    """The SwiGLU products on row counts between tiles (128-row tiles at these sizes): bit for bit the first
    M rows of the product over rows padded to a multiple of 256, and no row past M written."""
    assert {N.lib().unok_gemm_nt_fused_tile(m, n, Kd, 0) for m in (M, (M + 255) // 256 * 256) for n in (F, 2 * F)} == {2}
    torch.manual_seed(M + F)
    P = (M + 255) // 256 * 256
    bf = torch.bfloat16
    x, h = (torch.randn(P, Kd, device=dev) * 0.5).to(bf), (torch.randn(P, 2 * r, device=dev) * 0.5).to(bf)
    w, sb = (torch.randn(2 * F, Kd, device=dev) * 0.1).to(bf), (torch.randn(2 * F, 2 * r, device=dev) * 0.1).to(bf)
    gu_p = torch.empty(P, 2 * F, device=dev, dtype=bf)
    for kw, kw_p in (({}, {}), (dict(a2=h[:M], b2_interleaved=sb), dict(a2=h, b2_interleaved=sb))):
        gu = torch.full((P, 2 * F), 7.0, device=dev, dtype=bf)
        out = torch.full((P, F), 7.0, device=dev, dtype=bf)
        ref = K.gemm_nt_swiglu(x, w, gu=gu_p, **kw_p)
        K.gemm_nt_swiglu(x[:M], w, gu=gu[:M], out=out[:M], any_rows=True, **kw)
        assert torch.equal(out[:M], ref[:M]) and torch.equal(gu[:M], gu_p[:M])
        assert bool((out[M:] == 7).all()) and bool((gu[M:] == 7).all())
        out.fill_(7.0)
        K.gemm_nt_swiglu(x[:M], w, out=out[:M], any_rows=True, **kw)
        assert torch.equal(out[:M], ref[:M]) and bool((out[M:] == 7).all())
    dy, wt = x, (torch.randn(F, Kd, device=dev) * 0.1).to(bf)
    dgu = torch.full((P, 2 * F), 7.0, device=dev, dtype=bf)
    K.gemm_nt_swiglu_bwd(dy[:M], wt, h[:M, :r].contiguous(), sb[:F, :r].contiguous(), gu_p[:M], dgu=dgu[:M], any_rows=True)
    ref = K.gemm_nt_swiglu_bwd(dy, wt, h[:, :r].contiguous(), sb[:F, :r].contiguous(), gu_p)
    assert torch.equal(dgu[:M], ref[:M]) and bool((dgu[M:] == 7).all())
    if M % 256:
        with pytest.raises(ValueError, match="multiples of 256"):
            K.gemm_nt_swiglu(x[:M], w)


@pytest.mark.parametrize("M", [64, 200, 257, 777, 2100])     # the entry point takes M (nq + 2 nk) >= 512
@pytest.mark.parametrize("nq,nk,norm,lora", [(4, 2, True, True), (32, 8, True, False), (8, 8, False, True)])
def test_qkv_rope_on_any_row_count(dev, M, nq, nk, norm, lora):
    """The q|k|v projection with q/k norm + RoPE likewise: the first M rows of the padded product."""
    torch.manual_seed(M + nq)
    H, r, d, P = 512, 32, 128, (M + 255) // 256 * 256
    n = (nq + 2 * nk) * d
    x = (torch.randn(P, H, device=dev) * 0.5).bfloat16()
    w = (torch.randn(n, H, device=dev) * 0.05).bfloat16()
    h, b2 = (torch.randn(P, 3 * r, device=dev) * 0.3).bfloat16(), (torch.randn(n, r, device=dev) * 0.05).bfloat16()
    segs = [(nq * d, 0), ((nq + nk) * d, r), (n, 2 * r)]
    wq, wk = ((1 + 0.1 * torch.randn(d, device=dev)).bfloat16() if norm else None for _ in range(2))
    pos = torch.arange(P, device=dev) % 300
    inv = (1.0 / (1e6 ** (torch.arange(0, d, 2, dtype=torch.int64).float() / d))).to(dev)
    cos, sin = K.rope_table(300, inv)
    ref = K.gemm_nt_qkv_rope(x, w, nq, nk, wq, wk, pos, cos, sin, 1e-6, want_pre=True,
                             **(dict(a2=h, b2=b2, segments=segs) if lora else {}))
    got = K.gemm_nt_qkv_rope(x[:M], w, nq, nk, wq, wk, pos[:M], cos, sin, 1e-6, want_pre=True, any_rows=True,
                             **(dict(a2=h[:M], b2=b2, segments=segs) if lora else {}))
    for i, (a, b) in enumerate(zip(got, ref)):
        if i != 3 or norm:      # rstd is written with a norm only
            assert torch.equal(a, b[:M]), i


@pytest.mark.parametrize("M,Nn,Kd", [(1, 256, 64), (192, 256, 128), (193, 300, 192), (575, 516, 448)])
@pytest.mark.parametrize("ranges", [1, 2])
@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
def test_192_row_tiles(dev, M, Nn, Kd, ranges, out_dtype):
    """192x256 tiles (plan 6) at row and column remainders, with residual and row gate, bit for bit the
    256x256 tiles' result in one range (the same K order per output)."""
    if ranges > Kd // 64:
        pytest.skip("fewer K tiles than ranges")
    print(f"[192] {M}x{Nn}x{Kd} ranges {ranges} {out_dtype}", flush=True)
    torch.manual_seed(M + Nn)
    a, b = torch.randn(M, Kd, device=dev).bfloat16(), torch.randn(Nn, Kd, device=dev).bfloat16()
    res = torch.randn(M, Nn, device=dev).to(out_dtype)
    gate = torch.rand(M, device=dev) > 0.3
    outs = []
    for tile in (6, 1):
        out = torch.empty(M, Nn, device=dev, dtype=out_dtype)
        _call(tile + 16 * ranges, a, b, None, None, [(Nn, 0)], out, res, gate, 0.5, ranges)
        outs.append(out)
    ref = 0.5 * (a.float() @ b.float().T) * gate[:, None] + res.float()
    assert _rel(outs[0], ref) < (1e-5 if out_dtype == torch.float32 else 4e-3)
    assert torch.equal(*outs)


@pytest.mark.parametrize("M", [720, 777])
def test_192_row_tiles_fused_epilogues(dev, M):
    """The fused products at a row count for which 192-row tiles are the cheapest (the q|k|v product's are
    at others: test_fused_epilogues_by_tile), against the separate kernels: SwiGLU and its backward bit for
    bit, q|k|v with norm and RoPE to one bf16 rounding."""
    tile = N.lib().unok_gemm_nt_fused_tile
    assert tile(M, 24576, 1024, 0) == 6 and tile(M, 12288, 1024, 0) == 6 and tile(M, 6144, 1024, 0) == 2
    torch.manual_seed(M)
    H, F, nq, nk = 1024, 12288, 32, 8
    x = torch.randn(M, H, device=dev).bfloat16()
    w = (torch.randn(2 * F, H, device=dev) * 0.05).bfloat16()
    gu = torch.empty(M, 2 * F, device=dev, dtype=torch.bfloat16)
    s = K.gemm_nt_swiglu(x, K.interleave_gate_up(w, F), gu=gu, any_rows=True)
    assert torch.equal(gu, K.gemm_nt(x, w)) and torch.equal(s, K.swiglu_fwd(gu, F))
    assert torch.equal(s, K.gemm_nt_swiglu(x, K.interleave_gate_up(w, F), any_rows=True))
    wt = (torch.randn(F, H, device=dev) * 0.05).bfloat16()
    assert torch.equal(K.gemm_nt_swiglu_bwd(x, wt, None, None, gu, any_rows=True), K.swiglu_bwd(K.gemm_nt(x, wt), gu, F))
    wq, wk = (1 + 0.1 * torch.randn(2, 128, device=dev)).bfloat16()
    wqkv = (torch.randn(128 * (nq + 2 * nk), H, device=dev) * 0.05).bfloat16()
    inv = 1.0 / (1e6 ** (torch.arange(0, 128, 2, device=dev).float() / 128))
    pos = torch.randint(0, 500, (M,), device=dev)
    q, k, v, _, _ = K.gemm_nt_qkv_rope(x, wqkv, nq, nk, wq, wk, pos, *K.rope_table(500, inv), 1e-6, any_rows=True)
    q2, k2, v2, _ = K.qknorm_rope_fwd(K.gemm_nt(x, wqkv, out_dtype=torch.float32), nq, nk, 128, wq, wk, pos, inv, 1e-6,
                                      out_dtype=torch.bfloat16, with_v=True)
    for got, want in ((q, q2), (k, k2), (v, v2)):
        assert _rel(got, want) < 1e-3


@pytest.mark.parametrize("M,F,Kd,r", [(5, 256, 128, 0), (300, 1536, 512, 32), (777, 12288, 1024, 0), (2100, 5632, 320, 64)])
def test_swiglu_product_on_the_fused_projection_rows(dev, M, F, Kd, r):
    """The SwiGLU product reading [gate; up] weight rows as they are stored: bit for bit the one over
    interleaved rows, with and without an extension and the stored [gate | up]."""
    torch.manual_seed(M + F)
    bf = torch.bfloat16
    x, w = (torch.randn(M, Kd, device=dev) * 0.5).to(bf), (torch.randn(2 * F, Kd, device=dev) * 0.1).to(bf)
    kw = {}
    if r:
        kw = dict(a2=(torch.randn(M, 2 * r, device=dev) * 0.5).to(bf),
                  b2_interleaved=(torch.randn(2 * F, 2 * r, device=dev) * 0.1).to(bf))
    gus = [torch.empty(M, 2 * F, device=dev, dtype=bf) for _ in range(2)]
    wi = K.interleave_gate_up(w, F)
    ref = K.gemm_nt_swiglu(x, wi, gu=gus[0], any_rows=True, **kw)
    got = K.gemm_nt_swiglu(x, w, gu=gus[1], any_rows=True, plain_rows=True, **kw)
    assert torch.equal(got, ref) and torch.equal(*gus)
    assert torch.equal(K.gemm_nt_swiglu(x, w, any_rows=True, plain_rows=True, **kw), ref)


@pytest.mark.parametrize("M,Nn,Kd", [(300, 4096, 12288), (485, 4096, 12288), (777, 6144, 1024), (1196, 2048, 11008)])
@pytest.mark.parametrize("K2", [32, 128])
def test_zero_extension_changes_no_bit(dev, M, Nn, Kd, K2):
    """As above for the library's own choice: a product with an adapter of zeros is the plain product."""
    torch.manual_seed(M + K2)
    a, b = torch.randn(M, Kd, device=dev).bfloat16(), torch.randn(Nn, Kd, device=dev).bfloat16()
    h, bl = torch.randn(M, K2, device=dev).bfloat16(), torch.zeros(Nn, K2, device=dev).bfloat16()
    plain = K.gemm_nt(a, b, out_dtype=torch.float32)
    assert torch.equal(plain, K.gemm_nt(a, b, a2=h, b2=bl, out_dtype=torch.float32))


def _unsplit(a, b, a2=None, b2=None, segs=(), out_dtype=torch.bfloat16):
    """gemm_nt in one range of K (the entry point without a workspace)."""
    out = torch.empty(a.shape[0], b.shape[0], device=a.device, dtype=out_dtype)
    N.call("unok_gemm_nt", N.BF16, N.dtype_code(out_dtype), a.shape[0], b.shape[0], a.shape[1], N.ptr(a), a.stride(0),
           N.ptr(b), b.stride(0), N.ptr(a2), a2.stride(0) if a2 is not None else 0, N.ptr(b2),
           b2.stride(0) if b2 is not None else 0, b2.shape[1] if b2 is not None else 0, len(segs),
           N.int_array([s[0] for s in segs]), N.int_array([s[1] for s in segs]), N.ptr(out), out.stride(0), None, 0, None, 1.0,
           N.stream())
    return out


def _tile(M, n, Kd, K2):
    return N.lib().unok_gemm_nt_fused_tile(M, n, Kd, K2)


# tile chosen, rows (ragged and whole), hidden width, FFN width
@pytest.mark.parametrize("tile,M,H,F", [(1, 400, 1024, 12288), (1, 7655, 2048, 5632), (6, 300, 1024, 12288),
                                        (6, 384, 1024, 12288), (2, 150, 1024, 12288)])
@pytest.mark.parametrize("r", [0, 16, 32])
def test_swiglu_epilogue_by_tile(dev, tile, M, H, F, r):
    """SwiGLU in the epilogue of 256-, 192- and 128-row tiles with a last tile that is not full, with and
    without the LoRA extension (2 r columns) and the stored [gate | up]: bit for bit the plain product
    followed by the SwiGLU kernel, and no row past M written."""
    assert _tile(M, 2 * F, H, 2 * r) == tile
    torch.manual_seed(M + r)
    bf = torch.bfloat16
    x, w = (torch.randn(M, H, device=dev) * 0.5).to(bf), (torch.randn(2 * F, H, device=dev) * 0.05).to(bf)
    kw, ext = {}, ()
    if r:
        h, sb = (torch.randn(M, 2 * r, device=dev) * 0.5).to(bf), (torch.randn(2 * F, r, device=dev) * 0.1).to(bf)
        b2 = torch.zeros(F // 64, 2, 64, 2 * r, device=dev, dtype=bf)
        b2[:, 0, :, :r], b2[:, 1, :, r:] = sb[:F].view(-1, 64, r), sb[F:].view(-1, 64, r)
        kw = dict(a2=h, b2_interleaved=b2.view(2 * F, 2 * r))
        pad = torch.zeros(2 * F, 2 * r, device=dev, dtype=bf)      # the same extension over plain rows, same K order
        pad[:F, :r], pad[F:, r:] = sb[:F], sb[F:]
        ext = (h, pad, [(2 * F, 0)])
    want = _unsplit(x, w, *ext)
    s = K.swiglu_fwd(want, F)
    for store in (False, True):
        out, gu = torch.full((M + 300, F), 7.0, device=dev, dtype=bf), torch.full((M + 300, 2 * F), 7.0, device=dev, dtype=bf)
        K.gemm_nt_swiglu(x, w, out=out[:M], gu=gu[:M] if store else None, any_rows=True, plain_rows=True, **kw)
        assert torch.equal(out[:M], s) and bool((out[M:] == 7).all())
        if store:
            assert torch.equal(gu[:M], want) and bool((gu[M:] == 7).all())


@pytest.mark.parametrize("tile,M,H,F", [(1, 1000, 1024, 12288), (1, 7655, 2048, 5632), (6, 700, 1024, 12288),
                                        (6, 768, 1024, 12288), (2, 300, 1024, 12288)])
@pytest.mark.parametrize("r", [0, 32])
def test_swiglu_backward_epilogue_by_tile(dev, tile, M, H, F, r):
    """The SwiGLU backward likewise."""
    assert _tile(M, F, H, r) == tile
    torch.manual_seed(M + r)
    bf = torch.bfloat16
    dy, wt = (torch.randn(M, H, device=dev) * 0.5).to(bf), (torch.randn(F, H, device=dev) * 0.05).to(bf)
    gu = (torch.randn(M, 2 * F, device=dev) * 2).to(bf)
    a2, b2 = ((torch.randn(M, r, device=dev) * 0.5).to(bf), (torch.randn(F, r, device=dev) * 0.1).to(bf)) if r else (None, None)
    want = K.swiglu_bwd(_unsplit(dy, wt, a2, b2, [(F, 0)] if r else ()), gu, F)
    dgu = torch.full((M + 300, 2 * F), 7.0, device=dev, dtype=bf)
    K.gemm_nt_swiglu_bwd(dy, wt, a2, b2, gu, dgu=dgu[:M], any_rows=True)
    assert torch.equal(dgu[:M], want) and bool((dgu[M:] == 7).all())


@pytest.mark.parametrize("tile,M,H", [(1, 2000, 1024), (6, 1301, 1024), (6, 1344, 1024), (2, 700, 1024)])
@pytest.mark.parametrize("r", [0, 32, 64])
@pytest.mark.parametrize("pre_f32", [0, 1])
def test_qkv_rope_epilogue_by_tile(dev, tile, M, H, r, pre_f32):
    """q|k|v with norm and RoPE on 256-, 192- (in two 48-row passes) and 128-row tiles, with and without the
    LoRA extension: v and the kept pre-norm columns bit for bit the plain fp32 product's rounding, q and k
    within one bf16 rounding of the separate norm kernel, no row past M written."""
    nq, nk, d, bf = 32, 8, 128, torch.bfloat16
    n, e = d * (nq + 2 * nk), d * (nq + nk)
    assert _tile(M, n, H, r) == tile
    torch.manual_seed(M + r)
    x, w = torch.randn(M, H, device=dev).to(bf), (torch.randn(n, H, device=dev) * 0.05).to(bf)
    h, b2, segs = None, None, []
    if r:
        h, b2 = torch.randn(M, 3 * r, device=dev).to(bf), (torch.randn(n, r, device=dev) * 0.05).to(bf)
        segs = [(d * nq, 0), (e, r), (n, 2 * r)]
    wq, wk = (1 + 0.1 * torch.randn(2, d, device=dev)).to(bf)
    inv = 1.0 / (1e6 ** (torch.arange(0, d, 2, device=dev).float() / d))
    pos, (cos, sin) = torch.randint(0, 500, (M,), device=dev), K.rope_table(500, inv)
    P = M + 300
    full = lambda c, dt=bf: torch.full((P, c), 7.0, device=dev, dtype=dt)  # noqa: E731
    q, k, v, rstd = full(d * nq), full(d * nk), full(d * nk), full(nq + nk, torch.float32)
    pre = full(e, torch.float32 if pre_f32 else bf)
    N.call("unok_gemm_nt_qkv_rope_any", M, H, nq, nk, N.ptr(x), H, N.ptr(w), H, N.ptr(h), 3 * r, N.ptr(b2), r, r, len(segs),
           N.int_array([s[0] for s in segs]), N.int_array([s[1] for s in segs]), N.ptr(wq), N.ptr(wk), N.ptr(pos), N.ptr(cos),
           N.ptr(sin), 500, 1e-6, N.ptr(q), N.ptr(k), N.ptr(v), N.ptr(rstd), N.ptr(pre), pre_f32, N.stream())
    y = _unsplit(x, w, h, b2, segs, torch.float32)
    q2, k2, v2, rstd2 = K.qknorm_rope_fwd(y, nq, nk, d, wq, wk, pos, inv, 1e-6, out_dtype=bf, with_v=True)
    assert torch.equal(v[:M], v2) and torch.equal(pre[:M], y[:, :e].to(pre.dtype))
    assert _rel(q[:M], q2) < 1e-3 and _rel(k[:M], k2) < 1e-3 and _rel(rstd[:M], rstd2.view(M, -1)) < 1e-5
    for t in (q, k, v, rstd, pre):
        assert bool((t[M:] == 7).all())
