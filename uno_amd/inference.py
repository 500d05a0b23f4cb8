"""Draft forward of Uno's two-pass block decoding on the training step's kernels.

The inference side of the conditional LoRA (nano_vllm_uno/engine/two_pass_decoding.py:243-283,
draft_stage): each sequence feeds a block [seed, noise_1, ..., noise_(L-1)] through the decoder
over its KV cache; the LoRA update is gated per row -- off on the seed, on for the noise rows
(nano_vllm_uno/layers/linear.py:166-307, `lora_mask`) -- and attention is causal over the cache and
the block (nano_vllm_uno/layers/attention.py:628-668, BLOCK_DECODE: the block's K/V are stored into
the cache first, then flash attention with causal=True over the cached lengths). After the draft
the noise K/V are discarded: only the committed rows (the seed) advance the cache.

Kernels:
* the gated LoRA linears of a bf16 draft block are the few-row products (unok_gemm_nt_rows), which stream
  each weight once past the block's rows: the LoRA A rows are extra product columns, and the reduction
  forms h = m (.) (x A^T) and adds h (s B)^T (+ residual, or SwiGLU); a layer is one native call
  (unok_draft_layer). Other dtypes, and more than 512 rows, run the training step's GEMMs with the LoRA
  as their K-extension;
* the cache is head-major, [layers][B, Hkv, max_len, D] for K and V, so one (sequence, K/V head)
  pair's keys are contiguous rows; the block's queries of that pair (L rows x the q-heads sharing
  the K/V head, at most 128) are laid out as the 128 query rows of one attention workgroup over
  that key range, with per-row key intervals [start, start + cached + j + 1) -- the block-diffusion
  attention kernel then reads each cache row once per pair;
* a prefill (empty caches) is the clean stream's causal forward of the prompt (LoRA off, keys = the
  prompt itself).
"""
from __future__ import annotations

import ctypes

import torch

from . import _native as N
from . import kernels as K
from .adapter import MODULES
from .layers import Geometry, StreamContext, clean_layer


class BlockKVCache:
    """Per-layer K and V, head-major [B, Hkv, max_len, D], and the committed length per sequence."""

    def __init__(self, geo: Geometry, layers: int, batch: int, max_len: int, device, dtype):
        shape = (batch, geo.nk, max_len, geo.d)
        self.k = [torch.zeros(shape, device=device, dtype=dtype) for _ in range(layers)]
        self.v = [torch.zeros(shape, device=device, dtype=dtype) for _ in range(layers)]
        self.lengths = torch.zeros(batch, device=device, dtype=torch.int64)
        self.batch, self.max_len, self.geo = batch, max_len, geo


class BlockDecoder:
    """Runs prefill and draft blocks of a Uno model (UnoLoraModel or a base model with an
    adapter attached) on the HIP kernels."""

    def __init__(self, lm):
        base = lm.get_base_model() if hasattr(lm, "get_base_model") else lm
        self.base = base
        self.decoder = base.model
        self.lora = self.decoder._uno_lora
        if self.lora is None:
            raise RuntimeError("BlockDecoder needs a model with a LoRA adapter attached (create_lora_model).")
        self.geo = self.decoder.geo

    def new_cache(self, batch: int, max_len: int) -> BlockKVCache:
        return BlockKVCache(self.geo, len(self.decoder.layers), batch, max_len, self.base.device, self.base.dtype)

    # ---- public entry points ------------------------------------------------------------------
    @torch.no_grad()
    def prefill(self, cache: BlockKVCache, prompt_ids: torch.Tensor) -> torch.Tensor:
        """Causal forward of [B, P] prompt tokens into empty caches (LoRA off); returns logits
        [B, P, V] and commits all P rows."""
        if int(cache.lengths.max()) != 0:
            raise RuntimeError("prefill expects empty caches")
        return self._forward(cache, prompt_ids, None, commit=prompt_ids.shape[1], prefill=True)

    @torch.no_grad()
    def draft_block(self, cache: BlockKVCache, block_ids: torch.Tensor, lora_mask: torch.Tensor | None = None,
                    commit: int = 1) -> torch.Tensor:
        """One draft block [B, L] at positions cached + 0 .. L-1; returns logits [B, L, V]. The
        LoRA gate defaults to the draft layout (off on the seed row, on for the noise rows);
        ``commit`` rows (the seed) stay in the cache, the rest are discarded."""
        B, L = block_ids.shape
        if lora_mask is None:
            lora_mask = torch.ones((B, L), device=block_ids.device, dtype=torch.bool)
            lora_mask[:, 0] = False
        if tuple(lora_mask.shape) != (B, L):
            raise RuntimeError(f"LoRA row mask {tuple(lora_mask.shape)} does not match the block {(B, L)}")
        if not 0 <= commit <= L:
            raise ValueError(f"commit must lie in [0, {L}]")
        return self._forward(cache, block_ids, lora_mask.to(torch.bool), commit=commit, prefill=False)

    def capture_draft(self, cache: BlockKVCache, block_size: int, commit: int = 1) -> "DraftGraph":
        """A draft block of [cache.batch, block_size] rows over ``cache`` captured as one HIP graph
        (see DraftGraph)."""
        return DraftGraph(self, cache, block_size, commit)

    # ---- the decoder -----------------------------------------------------------------------------
    def _forward(self, cache: BlockKVCache, ids: torch.Tensor, gate: torch.Tensor | None, commit: int, prefill: bool,
                 check: bool = True):
        g, lora, dec = self.geo, self.lora, self.decoder
        B, L = ids.shape
        if B != cache.batch:
            raise RuntimeError(f"block batch {B} does not match the cache batch {cache.batch}")
        lengths = cache.lengths
        if check and int(lengths.max()) + L > cache.max_len:
            raise RuntimeError("the block does not fit in the KV cache")
        rep = g.nq // g.nk
        if not prefill and rep * L > 128:
            raise NotImplementedError(f"draft blocks hold at most 128 / {rep} rows per sequence (got {L})")
        dev = ids.device
        M = B * L
        h = K.embedding(ids.reshape(-1).contiguous().to(torch.int64), dec.embed_tokens.weight)
        if prefill:
            h = self._prefill_layers(h, cache, B, L)
        elif self._split_path(dev, cache) and self._rows_path(M, h.dtype, prefill):
            h = self._draft_layers(h, cache, gate.reshape(-1).contiguous(), B, L)
        else:
            gate_rows = gate.reshape(-1).contiguous()
            j = torch.arange(L, device=dev)
            pos = (lengths[:, None] + j[None, :]).reshape(-1).contiguous()            # [M] int64
            maps = self._maps(cache, lengths, B, L)
            for li, layer in enumerate(dec.layers):
                lw = layer.weights()
                h = self._layer(h, lw, li, pos, gate_rows, cache, maps, B, L)
        x, _ = K.rmsnorm_fwd(h, dec.norm.weight, g.eps)
        V = self.base.lm_head.weight.shape[0]
        head = K.gemm_nt_rows if self._rows_path(M, x.dtype, prefill) and V % 4 == 0 else K.gemm_nt
        logits = head(x, self.base.lm_head.weight)
        cache.lengths += commit
        return logits.view(B, L, -1)

    def _prefill_layers(self, h, cache, B: int, P: int):
        """All layers over B prompts of P tokens into empty caches: the clean stream's layer (no LoRA rows,
        so no adapter products), its K and V copied into the cache rows (b, head, t)."""
        g, dec, dev = self.geo, self.decoder, h.device
        t = torch.arange(P, device=dev)
        b = torch.arange(B, device=dev)
        iv = torch.zeros((B, P, 8), device=dev, dtype=torch.int32)
        iv[..., 0] = b[:, None] * P
        iv[..., 1] = b[:, None] * P + t + 1
        kv = torch.arange(g.nk, device=dev)
        store = ((b[:, None, None] * g.nk + kv) * cache.max_len + t[:, None]).reshape(-1).to(torch.int32)
        sc = StreamContext(t.repeat(B), dec.inv_freq, None, iv.view(B * P, 8), [], [])
        if h.dtype == torch.bfloat16 and g.d == 128:
            sc.rope_cos, sc.rope_sin = K.rope_table(P, dec.inv_freq)
        rows = B * P * g.nk
        for li, layer in enumerate(dec.layers):
            h, k, v = clean_layer(h, layer.weights(), g, sc)
            K.rows_copy(k.reshape(rows, g.d), cache.k[li].view(-1, g.d), rows, dmap=store)
            K.rows_copy(v.reshape(rows, g.d), cache.v[li].view(-1, g.d), rows, dmap=store)
        return h

    def _maps(self, cache, lengths, B, L):
        """Row maps of the cache store and of the decode query layout, and the key intervals."""
        g = self.geo
        dev = lengths.device
        i32 = dict(device=dev, dtype=torch.int32)
        rep = g.nq // g.nk
        out = {}
        if self._split_path(dev, cache):
            S = self._key_ranges(cache, B)
            out["ivs"], out["dst"] = K.decode_maps(lengths, B, L, g.nq, g.nk, cache.max_len, S)
            out["S"], out["QR"] = S, B * g.nk * 128
            return out
        slot = torch.arange(128, device=dev)
        pair = torch.arange(B * g.nk, device=dev)
        valid = slot < rep * L
        tt = slot % L
        start = pair[:, None] * cache.max_len                                           # [pairs, 1]
        lens = lengths[:, None].expand(B, g.nk).reshape(-1, 1)                          # [pairs, 1]
        seen = lens + tt[None, :] + 1                                                   # causal over cache + block
        b = torch.arange(B, device=dev)[:, None, None]
        t = torch.arange(L, device=dev)[None, :, None]
        kv = torch.arange(g.nk, device=dev)[None, None, :]
        # cache store: key row (b, t, head) of the block -> cache row (b, head, lengths_b + t)
        out["store"] = ((b * g.nk + kv) * cache.max_len + lengths[:, None, None] + t).reshape(-1).to(**i32)
        # decode layout: query (b, t, head h = kv * rep + r) -> row (b * nk + kv) * 128 + r * L + t
        r = torch.arange(rep, device=dev)
        qrow = ((b * g.nk + kv)[..., None] * 128 + r[None, None, None, :] * L + t[..., None])   # [B, L, nk, rep]
        out["qrow"] = qrow.reshape(-1).to(**i32)
        iv = torch.zeros((B * g.nk * 128, 8), **i32)
        # rows past rep * L are padding: they see the pair's first key and their output is dropped
        iv[:, 0] = start.expand(-1, 128).reshape(-1)
        iv[:, 1] = torch.where(valid[None, :], start + seen, start + 1).reshape(-1)
        out["iv"] = iv
        return out

    def _key_ranges(self, cache, B: int) -> int:
        """Key ranges per (sequence, K/V head) pair: as many as give one round of attention workgroups
        (one per pair and range, 256 CUs), at most eight."""
        return max(1, min(8, 256 // (B * self.geo.nk)))

    def _check_layer(self, lw, li: int, cache, B: int, dtype) -> None:
        """Shapes and dtypes of what unok_draft_layer reads by address in layer ``li``."""
        g = self.geo
        kv = (B, g.nk, cache.max_len, g.d)
        for what, t, shape in (("w_qkv", lw.w_qkv, (g.q + 2 * g.kv, g.H)), ("w_o", lw.w_o, (g.H, g.q)),
                               ("w_gu", lw.w_gu, (2 * g.F, g.H)), ("w_d", lw.w_d, (g.H, g.F)),
                               ("input norm", lw.ln_in, (g.H,)), ("post-attention norm", lw.ln_post, (g.H,)),
                               ("q norm", lw.q_norm, (g.d,)), ("k norm", lw.k_norm, (g.d,)),
                               ("cached keys", cache.k[li], kv), ("cached values", cache.v[li], kv)):
            if t is not None and (t.shape != shape or t.dtype != dtype or not t.is_contiguous()):
                raise RuntimeError(f"draft block: layer {li} {what} must be contiguous {dtype} {shape}, got {t.dtype} "
                                   f"{tuple(t.shape)}")
        s = self.lora.slots[li]
        dims = (g.H, g.q, g.H, g.kv, g.H, g.kv, g.q, g.H, g.H, g.F, g.H, g.F, g.F, g.H)
        if tuple(n for m in MODULES for n in (s[m].inp, s[m].out)) != dims:
            raise RuntimeError(f"draft block: the adapter's projections do not match layer {li}'s")

    def _draft_layers(self, h, cache, gate_rows, B: int, L: int):
        """All layers of a bf16 draft block, one native call each (see unok_draft_layer); the layers share
        one scratch buffer. Each layer's operands are checked as it is issued, behind the layers before it
        (all at once ahead of the first, the checks took 115 us of an 840 us block of eight layers)."""
        g, lora, dec = self.geo, self.lora, self.decoder
        lengths, inv_freq = cache.lengths, dec.inv_freq
        if h.shape[1] != g.H or not h.is_contiguous() or len(lora.slots) != len(dec.layers):
            raise RuntimeError("draft block: hidden size and layers must match the model's and the adapter's")
        if lora.copy.dtype != h.dtype or lora.copy.numel() != lora.numel or not lora.copy.is_contiguous():
            raise RuntimeError(f"draft block: the LoRA copy must be contiguous {h.dtype} [{lora.numel}]")
        if lengths.dtype != torch.int64 or lengths.shape != (B,) or inv_freq.dtype != torch.float32 or \
                inv_freq.numel() != g.d // 2:
            raise RuntimeError("draft block: int64 cache lengths [B] and fp32 inv_freq [D/2] required")
        if gate_rows.dtype not in (torch.bool, torch.uint8) or gate_rows.numel() != B * L:
            raise RuntimeError("draft block: bool gate [B, L] required")
        S = self._key_ranges(cache, B)
        ivs, dst = K.decode_maps(lengths, B, L, g.nq, g.nk, cache.max_len, S)
        a = N.DraftLayerArgs(B=B, L=L, nq=g.nq, nk=g.nk, D=g.d, H=g.H, F=g.F, r=lora.rank, S=S, max_len=cache.max_len,
                             eps=g.eps, scale=g.d ** -0.5, lengths=N.ptr(lengths), inv_freq=N.ptr(inv_freq),
                             gate=N.ptr(gate_rows), ivs=N.ptr(ivs), dst=N.ptr(dst))
        nbytes = N.lib().unok_draft_layer_scratch(ctypes.byref(a))
        if nbytes < 0:
            N.check(-1, "unok_draft_layer_scratch")
        scratch = torch.empty(nbytes + 256, device=h.device, dtype=torch.uint8)
        a.scratch, a.scratch_bytes = (N.ptr(scratch) + 255) // 256 * 256, nbytes
        other, stream = torch.empty_like(h), N.stream()
        for li, layer in enumerate(dec.layers):
            lw = layer.weights()
            parts = (("qkv", lw.w_qkv), ("o", lw.w_o), ("gu", lw.w_gu), ("d", lw.w_d))
            if not all(w.is_contiguous() for _, w in parts):
                # rows with a stride of their own: the products one by one, which take it
                maps = {"ivs": ivs, "dst": dst, "S": S, "QR": B * g.nk * 128}
                h, other = self._layer(h, lw, li, None, gate_rows, cache, maps, B, L), h
                continue
            self._check_layer(lw, li, cache, B, h.dtype)
            a.ln_in, a.ln_post, a.q_norm, a.k_norm = N.ptr(lw.ln_in), N.ptr(lw.ln_post), N.ptr(lw.q_norm), N.ptr(lw.k_norm)
            for part, w in parts:
                setattr(a, "w_" + part, N.ptr(w))
                la, lb = lora.group_ptrs(li, part)
                setattr(a, "a_" + part, la)
                setattr(a, "b_" + part, lb)
            a.kc, a.vc = N.ptr(cache.k[li]), N.ptr(cache.v[li])
            a.h, a.h_out = N.ptr(h), N.ptr(other)
            N.call("unok_draft_layer", ctypes.byref(a), stream)
            h, other = other, h
        return h

    def _split_path(self, dev, cache) -> bool:
        """bf16 draft blocks run the attention as prep + split-key attention + combine."""
        return cache.k[0].dtype == torch.bfloat16 and self.geo.d in (64, 128)

    def _rows_path(self, M: int, dtype, prefill: bool) -> bool:
        """Draft blocks in bf16 take the few-row products (K ranges over the whole chip) when every
        linear's shape fits them; prefills and fp32 models take gemm_nt."""
        g, r = self.geo, self.lora.rank
        return (not prefill and dtype == torch.bfloat16 and M <= 512 and r % 8 == 0 and 3 * r <= 512
                and all(k % 128 == 0 for k in (g.H, g.q, g.F)))

    def _layer(self, h0, lw, li, pos, gate_rows, cache, maps, B, L):
        g, lora = self.geo, self.lora
        r = lora.rank
        q_end, k_end = g.q, g.q + g.kv
        M = h0.shape[0]
        few = self._rows_path(M, h0.dtype, False)
        qkv_segments = [(q_end, 0), (k_end, r), (k_end + g.kv, 2 * r)]

        def linear(x, w, part, segments=None, residual=None, swiglu=False):
            """Gated LoRA linear: x w^T + (m (.) x A^T)[:, seg] (s B)^T (+ residual)."""
            if few:
                return K.gemm_nt_rows(x, w, lora_a=lora.a_c(li, part), lora_b=lora.sb_c(li, part),
                                      segments=segments, residual=residual, gate=gate_rows, swiglu=swiglu)
            h = K.gemm_nt(x, lora.a_c(li, part), gate=gate_rows)
            y = K.gemm_nt(x, w, a2=h, b2=lora.sb_c(li, part), segments=segments, residual=residual)
            return K.swiglu_fwd(y, y.shape[1] // 2) if swiglu else y

        x1, _ = K.rmsnorm_fwd(h0, lw.ln_in, g.eps)
        qkv = linear(x1, lw.w_qkv, "qkv", qkv_segments)
        ck = cache.k[li].view(-1, g.d)
        cv = cache.v[li].view(-1, g.d)
        if "ivs" in maps:
            # q/k norm + RoPE, cache store and query layout in one kernel; split-key attention; merge
            S, QR = maps["S"], maps["QR"]
            qd = torch.empty((QR, g.d), device=qkv.device, dtype=qkv.dtype)
            K.decode_prep(qkv, lw.q_norm, lw.k_norm, cache.lengths, self.decoder.inv_freq, g.eps, cache.k[li],
                          cache.v[li], qd, B, L, g.nq, g.nk, g.d)
            od, lse = K.attn_fwd_split(qd, ck, cv, maps["ivs"], QR, S, g.d)
            o = torch.empty((M, g.q), device=qkv.device, dtype=qkv.dtype)
            K.attn_split_combine(od, lse, maps["dst"], QR, S, g.d, o.view(M * g.nq, g.d))
            return self._mlp(o, h0, lw, li, linear)
        q, k, _ = K.qknorm_rope_fwd(qkv, g.nq, g.nk, g.d, lw.q_norm, lw.k_norm, pos, self.decoder.inv_freq, g.eps)
        v = qkv[:, k_end:]
        # the block's K/V into the cache rows (b, head, cached + t)
        K.rows_copy(k.reshape(M * g.nk, g.d), ck, M * g.nk, dmap=maps["store"])
        K.rows_copy(v.contiguous().view(M * g.nk, g.d), cv, M * g.nk, dmap=maps["store"])
        rows = maps["iv"].shape[0]
        qd = torch.zeros((rows, g.d), device=q.device, dtype=q.dtype)
        K.rows_copy(q.reshape(M * g.nq, g.d), qd, M * g.nq, dmap=maps["qrow"])
        od, _ = K.attn_fwd(qd, ck, cv, maps["iv"], 1, 1, g.d)
        o = torch.empty((M, g.q), device=q.device, dtype=q.dtype)
        K.rows_copy(od, o.view(M * g.nq, g.d), M * g.nq, smap=maps["qrow"])
        return self._mlp(o, h0, lw, li, linear)

    def _mlp(self, o, h0, lw, li, linear):
        """o projection (+ residual), post-attention norm and the SwiGLU MLP (+ residual)."""
        g, r = self.geo, self.lora.rank
        h1 = linear(o, lw.w_o, "o", residual=h0)
        x2, _ = K.rmsnorm_fwd(h1, lw.ln_post, g.eps)
        s = linear(x2, lw.w_gu, "gu", [(g.F, 0), (2 * g.F, r)], swiglu=True)
        return linear(s, lw.w_d, "d", residual=h1)


class DraftGraph:
    """A draft block of fixed shape [B, L] over one cache, captured as a single HIP graph.

    The decoder runs 13 kernels per layer; issued from Python, even as one call per layer, a block of few
    rows can cost more host time than device time. Replaying the captured graph is one host
    call per block. Everything that depends on the committed lengths (the positions, the cache
    store rows, the decode query layout and the key intervals) is computed on the device from
    ``cache.lengths`` inside the graph, so each replay drafts at the current lengths and then
    advances them by ``commit``, exactly as ``BlockDecoder.draft_block``.

    ``replay`` returns the graph's own logits buffer [B, L, V], overwritten by the next replay.
    The cache capacity is checked on the host against the longest committed length read at
    capture plus the commits since; after changing ``cache.lengths`` by other means, capture
    again."""

    def __init__(self, decoder: BlockDecoder, cache: BlockKVCache, block_size: int, commit: int = 1):
        B, L = cache.batch, block_size
        rep = decoder.geo.nq // decoder.geo.nk
        if rep * L > 128:
            raise NotImplementedError(f"draft blocks hold at most 128 / {rep} rows per sequence (got {L})")
        if not 0 <= commit <= L:
            raise ValueError(f"commit must lie in [0, {L}]")
        dev = cache.lengths.device
        self.cache, self.block_size, self.commit = cache, L, commit
        self.ids = torch.zeros((B, L), device=dev, dtype=torch.int64)
        self.gate = torch.ones((B, L), device=dev, dtype=torch.bool)
        self.gate[:, 0] = False
        self._len_max = int(cache.lengths.max())
        if self._len_max + L > cache.max_len:
            raise RuntimeError("the block does not fit in the KV cache")
        # One eager pass without commit before the capture: it sets each kernel's launch attributes
        # outside the graph. Its K/V rows lie past the committed lengths, where the first replay
        # writes them again.
        decoder._forward(cache, self.ids, self.gate, commit=0, prefill=False)
        torch.cuda.synchronize()
        self.graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(self.graph):
            self.logits = decoder._forward(cache, self.ids, self.gate, commit=commit, prefill=False, check=False)

    def replay(self, block_ids: torch.Tensor, lora_mask: torch.Tensor | None = None) -> torch.Tensor:
        """Draft one block [B, L] of token ids (device int64); ``lora_mask`` [B, L] replaces the
        default gate (off on the seed row, on for the noise rows) for this and later replays."""
        if tuple(block_ids.shape) != tuple(self.ids.shape):
            raise RuntimeError(f"block {tuple(block_ids.shape)} does not match the captured {tuple(self.ids.shape)}")
        if self._len_max + self.block_size > self.cache.max_len:
            raise RuntimeError("the block does not fit in the KV cache")
        self.ids.copy_(block_ids)
        if lora_mask is not None:
            if tuple(lora_mask.shape) != tuple(self.gate.shape):
                raise RuntimeError(f"LoRA row mask {tuple(lora_mask.shape)} does not match the block")
            self.gate.copy_(lora_mask)
        self.graph.replay()
        self._len_max += self.commit
        return self.logits
