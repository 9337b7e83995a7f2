"""GPU: causal attention of more than 64 new tokens against float64, with
caches that hold NaN past the visible positions."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,start,heads,kvh,hd", [
    (1, 0, 2, 2, 64),        # one row, one position
    (65, 0, 4, 4, 64),       # a partial last tile, waves without a tile
    (65, 3, 6, 2, 128),      # rows of 3 heads straddle tiles; a partial cache tile
    (96, 31, 8, 8, 128),     # whole tiles after a cache one short of a tile
    (100, 32, 3, 1, 64),
    (129, 200, 24, 8, 64),
    (260, 0, 8, 2, 128),
])
def test_attention_prefill(gpu, N, start, heads, kvh, hd):
    import littlebit_amd._lib as L
    lib = L.load()
    gen = torch.Generator(device=gpu).manual_seed(N + start)
    r = lambda *s: torch.randn(s, generator=gen, device=gpu)  # noqa: E731
    max_seq = start + N + 7
    q, k, v = r(N, heads * hd), r(N, kvh * hd), r(N, kvh * hd)
    kc, vc = r(kvh, max_seq, hd), r(kvh, max_seq, hd)
    kc[:, start:], vc[:, start:] = float("nan"), float("nan")
    before = [c[:, :start].clone() for c in (kc, vc)]
    out = torch.full((N, heads * hd), float("nan"), device=gpu)
    stream = torch.cuda.current_stream(gpu).cuda_stream
    L.check(lib.lbk_attention_prefill(q.data_ptr(), k.data_ptr(), v.data_ptr(), kc.data_ptr(), vc.data_ptr(), N, heads,
                                      kvh, hd, max_seq, start, hd ** -0.5, out.data_ptr(), stream),
            "lbk_attention_prefill")
    torch.cuda.synchronize()
    for c, new, old in ((kc, k, before[0]), (vc, v, before[1])):
        assert torch.equal(c[:, :start], old)
        assert torch.equal(c[:, start:start + N], new.view(N, kvh, hd).transpose(0, 1))
        assert torch.isnan(c[:, start + N:]).all()
    i = torch.arange(N, device=gpu).view(N, 1)
    seen = torch.arange(start + N, device=gpu).view(1, -1) <= start + i
    for h in range(heads):
        j = h // (heads // kvh)
        s = q.view(N, heads, hd)[:, h].double() @ kc[j, :start + N].double().t().contiguous() * hd ** -0.5
        ref = torch.softmax(s.masked_fill(~seen, float("-inf")), -1) @ vc[j, :start + N].double()
        err = (out.view(N, heads, hd)[:, h] - ref).abs().max().item()
        # fp32 sums of hd and start + N terms of O(1): a few 2**-24 times their square roots
        assert err <= 2e-5, (h, err)


def test_attention_prefill_refuses(gpu):
    import littlebit_amd._lib as L
    lib = L.load()
    b = torch.zeros(1 << 16, device=gpu)
    call = lambda n, heads, kvh, hd, max_seq, start, off=0: lib.lbk_attention_prefill(  # noqa: E731
        b.data_ptr() + off, b.data_ptr(), b.data_ptr(), b.data_ptr(), b.data_ptr(), n, heads, kvh, hd, max_seq, start,
        1.0, b.data_ptr(), None)
    for args in [(0, 2, 2, 64, 10, 0), (4, 3, 2, 64, 10, 0), (4, 2, 2, 96, 10, 0), (4, 2, 2, 64, 10, 7),
                 (4, 2, 2, 64, 10, -1), (4, 2, 2, 64, 10, 0, 4)]:
        assert call(*args) == L.LBK_ERR_ARG, args


def test_decoder_prompt_matches_short_batches(gpu):
    """A prompt of 150 tokens in one call against the same tokens in batches
    of at most 64 (the batched attention), and again after a cached prefix."""
    from littlebit_amd.decode import DecoderConfig, LittleBitDecoder
    from littlebit_amd.synthetic import synthetic_runtime_state
    cfg = DecoderConfig(hidden_size=512, intermediate_size=1032, num_hidden_layers=2, num_attention_heads=8,
                        num_key_value_heads=4, vocab_size=128)
    st = synthetic_runtime_state(cfg, {"attn": 40, "mlp": 60}, seed=5, device=gpu, normalized=True)
    emb = st["model.embed_tokens.weight"]
    ids = [(7 * i + 3) % 128 for i in range(150)]
    one, many, two = (LittleBitDecoder(st, cfg, gpu, max_seq_len=160) for _ in range(3))
    with torch.no_grad():
        a = one.forward_batch(ids, emb)
        b = torch.cat([many.forward_batch(ids[i:i + 50], emb) for i in (0, 50, 100)])
        c = torch.cat([two.forward_batch(ids[:37], emb), two.forward_batch(ids[37:], emb)])
    for x in (b, c):
        err = ((a - x).norm() / a.norm()).item()
        assert err <= 1e-4, err
    assert ((one.k_cache - many.k_cache).norm() / one.k_cache.norm()).item() <= 1e-4
