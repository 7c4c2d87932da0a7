"""Splits of more than 64 groups of 64 keys over pages: the places of the groups are fetched 64 at a time."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt,D,page", [("bf16", 64, 64), ("bf16", 128, 256), ("q8_0", 64, 192), ("q8_0", 128, 64)])
@pytest.mark.parametrize("L", [4095, 4096, 4097, 4161, 9000])
def test_long_splits_over_pages(fmt, D, page, L):
    import vesper_amd as va
    B, Hq, Hkv = 16, 32, 16   # 256 (row, kv head) pairs: one split each
    S = -(-L // page) * page
    g = torch.Generator(device="cuda").manual_seed(L)
    flat = va.KVCache(B, Hkv, S, D, fmt=fmt)
    paged = va.KVCache(B, Hkv, S, D, fmt=fmt, paging=(page, B * (S // page)))
    paged.page_table.copy_(torch.randperm(B * (S // page), generator=torch.Generator().manual_seed(L)).to(torch.int32).view(B, -1))
    for t in range(0, L, 3000):
        n = min(3000, L - t)
        k, v = (torch.randn((B, Hkv, n, D), device="cuda", generator=g).to(torch.bfloat16) for _ in range(2))
        for c in (flat, paged):
            c.update(k, v, t, return_views=False)
    q = torch.randn((B, Hq, 1, D), device="cuda", generator=g).to(torch.bfloat16)
    lens = torch.full((B,), L, dtype=torch.int32, device="cuda")
    want = va.decode_attention(q, flat)
    assert torch.equal(va.decode_attention(q, paged), want)
    assert torch.equal(va.decode_attention(q, paged, seq_lens=lens, max_len=L), va.decode_attention(q, flat, seq_lens=lens, max_len=L))
    k, v = (x.repeat_interleave(2, 1) for x in flat.read(0, L))
    s = torch.matmul(k, q.float().transpose(2, 3)).squeeze(-1) * D ** -0.5
    ref = torch.matmul(s.softmax(-1).unsqueeze(2), v)
    assert ((want.float() - ref).norm() / ref.norm()).item() < 1e-2
