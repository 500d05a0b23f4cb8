"""What a draft block checks before its layers are handed to the library by address (no GPU: the native
calls are replaced by a recorder)."""
import pytest
import torch

from uno_amd import _native as N
from uno_amd import kernels as K
from uno_amd.adapter import LoraState
from uno_amd.inference import BlockDecoder
from uno_amd.model import UnoQwen3Config, UnoQwen3ForCausalLM

BF = torch.bfloat16
B, L = 2, 4


def _decoder(rank=8, lora_dtype=BF, lora_cfg=None):
    cfg = UnoQwen3Config(vocab_size=64, hidden_size=128, intermediate_size=256, num_hidden_layers=2,
                         num_attention_heads=2, num_key_value_heads=1, head_dim=64, block_size=L)
    model = UnoQwen3ForCausalLM(cfg, device="cpu", dtype=BF)
    model.model._uno_lora = LoraState(lora_cfg or cfg, rank, 16.0, "cpu", lora_dtype)
    return BlockDecoder(model)


def _narrow(t):
    return t[..., : t.shape[-1] - 8]


FAULTS = {
    "w_qkv rows": lambda d, c: setattr(d.decoder.layers[1], "w_qkv", d.decoder.layers[1].w_qkv[:-8]),
    "w_o columns": lambda d, c: setattr(d.decoder.layers[0], "w_o", _narrow(d.decoder.layers[0].w_o).contiguous()),
    "w_gu dtype": lambda d, c: setattr(d.decoder.layers[1], "w_gu", d.decoder.layers[1].w_gu.float()),
    "w_d rows": lambda d, c: setattr(d.decoder.layers[1], "w_d", d.decoder.layers[1].w_d[:-1]),
    "LoRA dtype": lambda d, c: setattr(d.lora, "copy", d.lora.copy.float()),
    "LoRA length": lambda d, c: setattr(d.lora, "copy", d.lora.copy[:-16]),
    "LoRA widths": lambda d, c: setattr(d.lora.slots[1]["up_proj"], "out", 128),
    "LoRA layers": lambda d, c: d.lora.slots.pop(),
    "norm dtype": lambda d, c: setattr(d.decoder.layers[0].input_layernorm, "weight",
                                       torch.nn.Parameter(torch.ones(128), requires_grad=False)),
    "q norm length": lambda d, c: setattr(d.decoder.layers[0].self_attn.q_norm, "weight",
                                          torch.nn.Parameter(torch.ones(32, dtype=BF), requires_grad=False)),
    "cache rows": lambda d, c: c.k.__setitem__(1, c.k[1][:, :, :-1].contiguous()),
    "cache dtype": lambda d, c: c.v.__setitem__(0, c.v[0].float()),
    "cache layout": lambda d, c: c.v.__setitem__(0, c.v[0].repeat(1, 1, 1, 2)[..., :64]),
    "lengths dtype": lambda d, c: setattr(c, "lengths", c.lengths.int()),
}


def _run(monkeypatch, dec, cache):
    calls = []
    monkeypatch.setattr(N, "call", lambda name, *a: calls.append(name))
    monkeypatch.setattr(N, "stream", lambda: 0)
    monkeypatch.setattr(K, "decode_maps", lambda *a: (torch.zeros(8, dtype=torch.int32), torch.zeros(8, dtype=torch.int32)))
    h = torch.zeros(B * L, 128, dtype=BF)
    try:
        dec._draft_layers(h, cache, torch.ones(B * L, dtype=torch.bool), B, L)
    finally:
        assert set(calls) <= {"unok_draft_layer"}
    return len(calls)


def test_matching_operands_reach_every_layer(monkeypatch):
    if not N.LIB_PATH.exists():
        pytest.skip("libunok.so not built")
    dec = _decoder()
    assert _run(monkeypatch, dec, dec.new_cache(B, 32)) == 2


@pytest.mark.parametrize("fault", FAULTS)
def test_mismatched_operands_are_refused(monkeypatch, fault):
    if not N.LIB_PATH.exists():
        pytest.skip("libunok.so not built")
    dec = _decoder()
    cache = dec.new_cache(B, 32)
    FAULTS[fault](dec, cache)
    with pytest.raises(RuntimeError, match="draft block"):
        _run(monkeypatch, dec, cache)
