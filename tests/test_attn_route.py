"""Which attention a decoder's prompts take, on the CPU (the kernel's call replaced by a marker)."""
import pytest
import torch

from littlebit_amd.decode import DecoderConfig, LittleBitDecoder


@pytest.mark.parametrize("heads,kvh,hd,n,start,library", [
    (8, 2, 128, 65, 4031, False),   # 4,096 positions
    (8, 2, 128, 65, 4032, True),
    (8, 2, 128, 256, 4000, True),   # 64 blocks
    (8, 2, 128, 257, 4000, False),  # 66
    (4, 1, 64, 70, 6074, False),    # 6,144 positions
    (4, 1, 64, 70, 6075, True),
    (32, 8, 128, 65, 9000, False),  # 72 blocks
    (2, 2, 128, 64, 5000, None),    # a batch: neither
])
def test_prompt_attention_route(monkeypatch, heads, kvh, hd, n, start, library):
    d = LittleBitDecoder.__new__(LittleBitDecoder)
    d.config = DecoderConfig(hidden_size=heads * hd, intermediate_size=8, num_hidden_layers=1,
                             num_attention_heads=heads, num_key_value_heads=kvh, vocab_size=8, rms_norm_eps=1e-6)
    d._hip_attn, d.max_seq_len = True, start + n
    gen = torch.Generator().manual_seed(n)
    d.k_cache, d.v_cache = (torch.randn((1, kvh, start + n, hd), generator=gen) for _ in range(2))
    for name in ("_attention_prefill_hip", "_attention_batch_hip"):
        monkeypatch.setattr(LittleBitDecoder, name, lambda self, *a, name=name: name)
    q, k, v = (torch.randn((n, h * hd), generator=gen) for h in (heads, kvh, kvh))
    out = d._attention(0, q, k, v, start, start + n, None, None)
    if not library:
        assert out == ("_attention_prefill_hip" if library is False else "_attention_batch_hip")
        return
    # the library's products, causal
    j = heads // kvh - 1  # a head of the first group
    s = q.view(n, heads, hd)[:, j].double() @ d.k_cache[0, 0].double().t() * hd ** -0.5
    seen = torch.ones(n, start + n, dtype=torch.bool).tril(start)
    ref = torch.softmax(s.masked_fill(~seen, float("-inf")), -1) @ d.v_cache[0, 0].double()
    assert (out.view(n, heads, hd)[:, j] - ref).abs().max() <= 2e-5
