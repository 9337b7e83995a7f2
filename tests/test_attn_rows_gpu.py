"""GPU: batched attention on both sides of the line between its two kernels,
against float64, with caches that hold NaN past the visible positions."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,start,heads,kvh,hd,tree,room", [
    (32, 40, 4, 4, 64, False, 0),       # the last count of the one kernel
    (33, 0, 4, 4, 64, False, 0),        # the first of the other: partial tiles, waves without a tile
    (35, 31, 6, 2, 128, True, 0),       # rows of 3 heads straddle tiles; a cache tile one short
    (64, 96, 8, 8, 64, True, 0),        # whole tiles
    (33, 1000, 32, 32, 128, True, 0),
    (64, 129, 3, 1, 64, False, 0),
    (64, 2000, 8, 2, 128, True, 0),     # several groups of tiles per chunk
    (17, 3133, 13, 13, 64, False, 0),   # heads * positions = 40,950: short of the many
    (17, 3134, 13, 13, 64, False, 0),   # 40,963
    (16, 3135, 13, 13, 64, False, 0),   # as many, one token fewer
    (2, 1279, 32, 8, 64, True, 0),      # groups: 40,992
    (2, 5119, 8, 8, 64, False, 0),      # as many, but no groups and few tokens
    (24, 5, 4, 2, 128, True, 3000),     # device start, few tokens
    (25, 5, 4, 2, 128, True, 3000),     # device start: a grid for 3,030 positions, most chunks empty
    (64, 700, 8, 8, 64, False, 1300),
    (40, 0, 2, 2, 64, True, 100),
    (3, 100, 32, 4, 64, False, 5017),   # device start: heads * positions = 163,840
    (3, 100, 32, 4, 64, False, 5018),   # 163,872
])
def test_attention_batch_routes(gpu, n, start, heads, kvh, hd, tree, room):
    import littlebit_amd._lib as L
    lib = L.load()
    gen = torch.Generator(device=gpu).manual_seed(n + start)
    r = lambda *s: torch.randn(s, generator=gen, device=gpu)  # noqa: E731
    max_seq = start + n + room
    q, k, v = r(n, heads * hd), r(n, kvh * hd), r(n, kvh * hd)
    kc, vc = r(kvh, max_seq, hd), r(kvh, max_seq, hd)
    kc[:, start:], vc[:, start:] = float("nan"), float("nan")
    before = [c[:, :start].clone() for c in (kc, vc)]
    mask = torch.ones(n, n, device=gpu).tril() > 0
    if tree:
        mask = (torch.rand(n, n, generator=gen, device=gpu) < 0.3) | torch.eye(n, dtype=torch.bool, device=gpu)
    bytes_ = mask.to(torch.uint8)
    out = torch.full((n, heads * hd), float("nan"), device=gpu)
    dev = torch.tensor([start], dtype=torch.int64, device=gpu) if room else None
    need = lib.lbk_attention_batch_partial_bytes(heads, n, max_seq - n if room else start, hd)
    part = torch.full((need // 4 + 64,), float("nan"), device=gpu)
    L.check(lib.lbk_attention_batch(q.data_ptr(), k.data_ptr(), v.data_ptr(), kc.data_ptr(), vc.data_ptr(), n, heads,
                                    kvh, hd, max_seq, dev.data_ptr() if room else None, 0 if room else start,
                                    bytes_.data_ptr() if tree else None, hd ** -0.5, part.data_ptr(), need,
                                    out.data_ptr(), torch.cuda.current_stream(gpu).cuda_stream), "lbk_attention_batch")
    torch.cuda.synchronize()
    assert torch.isnan(part[need // 4:]).all()
    for c, new, old in ((kc, k, before[0]), (vc, v, before[1])):
        assert torch.equal(c[:, :start], old)
        assert torch.equal(c[:, start:start + n], new.view(n, kvh, hd).transpose(0, 1))
        assert torch.isnan(c[:, start + n:]).all()
    seen = torch.cat([torch.ones(n, start, dtype=torch.bool, device=gpu), mask], dim=1)
    for h in range(heads):
        j = h // (heads // kvh)
        s = q.view(n, heads, hd)[:, h].double() @ kc[j, :start + n].double().t().contiguous() * hd ** -0.5
        ref = torch.softmax(s.masked_fill(~seen, float("-inf")), -1) @ vc[j, :start + n].double()
        err = (out.view(n, heads, hd)[:, h] - ref).abs().max().item()
        # fp32 sums of hd and start + n terms of O(1): a few 2**-24 times their square roots
        assert err <= 2e-5, (h, err)


def test_attention_batch_nothing_seen(gpu):
    """A token whose mask row is empty, with no cache, gives zeros."""
    import littlebit_amd._lib as L
    lib = L.load()
    n, heads, hd = 33, 2, 64
    q, k, v = (torch.randn(n, heads * hd, device=gpu) for _ in range(3))
    kc, vc = (torch.zeros(heads, n, hd, device=gpu) for _ in range(2))
    mask = torch.eye(n, dtype=torch.uint8, device=gpu)
    mask[7] = 0
    need = lib.lbk_attention_batch_partial_bytes(heads, n, 0, hd)
    part, out = torch.empty(need // 4, device=gpu), torch.empty(n, heads * hd, device=gpu)
    L.check(lib.lbk_attention_batch(q.data_ptr(), k.data_ptr(), v.data_ptr(), kc.data_ptr(), vc.data_ptr(), n, heads,
                                    heads, hd, n, None, 0, mask.data_ptr(), hd ** -0.5, part.data_ptr(), need,
                                    out.data_ptr(), torch.cuda.current_stream(gpu).cuda_stream), "lbk_attention_batch")
    torch.cuda.synchronize()
    assert not out[7].any()
    v[7] = 0
    assert torch.allclose(out, v, rtol=1e-6, atol=0)  # one position each: its own value


def test_attention_batch_of_very_many_heads(gpu):
    """Past 2**22 elements per token the calls of 33 to 64 tokens stay with
    the kernel that fewer tokens take (the other's offsets are 32-bit): its
    form of four query tiles, which no smaller shape reaches."""
    import littlebit_amd._lib as L
    lib = L.load()
    n, start, heads, hd = 40, 9, 65600, 64
    gen = torch.Generator(device=gpu).manual_seed(5)
    q, k, v = (torch.randn((n, heads * hd), generator=gen, device=gpu) for _ in range(3))
    kc, vc = (torch.randn((heads, start + n, hd), generator=gen, device=gpu) for _ in range(2))
    kc[:, start:], vc[:, start:] = float("nan"), float("nan")
    need = lib.lbk_attention_batch_partial_bytes(heads, n, start, hd)
    part, out = torch.empty(need // 4, device=gpu), torch.full((n, heads * hd), float("nan"), device=gpu)
    L.check(lib.lbk_attention_batch(q.data_ptr(), k.data_ptr(), v.data_ptr(), kc.data_ptr(), vc.data_ptr(), n, heads,
                                    heads, hd, start + n, None, start, None, hd ** -0.5, part.data_ptr(), need,
                                    out.data_ptr(), torch.cuda.current_stream(gpu).cuda_stream), "lbk_attention_batch")
    torch.cuda.synchronize()
    assert torch.equal(kc[:, start:], k.view(n, heads, hd).transpose(0, 1))
    assert torch.equal(vc[:, start:], v.view(n, heads, hd).transpose(0, 1))
    sample = torch.randint(0, heads, (64,), generator=gen, device=gpu).tolist() + [0, heads - 1]
    seen = torch.ones(n, start + n, dtype=torch.bool, device=gpu).tril(start)
    for h in sample:
        s = q.view(n, heads, hd)[:, h].double() @ kc[h].double().t().contiguous() * hd ** -0.5
        ref = torch.softmax(s.masked_fill(~seen, float("-inf")), -1) @ vc[h].double()
        err = (out.view(n, heads, hd)[:, h] - ref).abs().max().item()
        assert err <= 2e-5, (h, err)  # (as above)
    assert not torch.isnan(out).any()
