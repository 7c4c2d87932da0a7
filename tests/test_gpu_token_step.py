"""One generated token per sequence: append and attention in one launch against the two calls it stands for."""
import numpy as np
import pytest
import torch

import _gpu as G

pytestmark = pytest.mark.gpu


def _case(fmt, B, Hq, Hkv, D, ctx, paged, seed):
    import vesper_amd as va
    g = torch.Generator(device="cuda").manual_seed(seed)
    dt = torch.float32 if fmt == "f32" else torch.bfloat16
    S = (ctx // 64 + 2) * 64
    caches = []
    for _ in range(2):
        if paged:
            c = va.KVCache(B, Hkv, S, D, fmt=fmt, paging=(64, B * (S // 64)))
            c.page_table.copy_(torch.arange(B * (S // 64), dtype=torch.int32).flip(0).view(B, -1))
        else:
            c = va.KVCache(B, Hkv, S, D, fmt=fmt)
        for i in range(4):  # what lies past the context is not a number in any format
            if c.raw_plane(i) is not None:
                c.raw_plane(i).fill_(0x7f if fmt == "q8_0" and i < 2 else 0xff)
        caches.append(c)
    fused = torch.randn((B, 1, Hq + 2 * Hkv, D), device="cuda", generator=g).to(dt)
    q, k, v = (fused[:, :, a:b].transpose(1, 2) for a, b in ((0, Hq), (Hq, Hq + Hkv), (Hq + Hkv, Hq + 2 * Hkv)))
    if ctx:
        kc, vc = (torch.randn((B, Hkv, ctx, D), device="cuda", generator=g).to(dt) for _ in range(2))
        for c in caches:
            c.update(kc, vc, 0, return_views=False)
    return caches, q, k, v


def _compare(fmt, caches, q, k, v, pos, rope):
    import vesper_amd as va
    one = va.attention_core(q, k, v, caches[0], pos, rope=rope)
    if rope is not None:
        qr = caches[1].rope_update(q, k, v, pos, rope)
    else:
        qr = q.contiguous()
        caches[1].update(k, v, pos, return_views=False)
    two = va.decode_attention(qr, caches[1])
    assert caches[0].current_seq_len() == caches[1].current_seq_len()
    for i in range(4):
        if caches[0].raw_plane(i) is not None:
            assert torch.equal(caches[0].raw_plane(i), caches[1].raw_plane(i)), i
    assert torch.isfinite(two).all()
    # P of the token is 1 exactly here and rounded there (bf16: 2^-9 of |v|; fp16 in a Q8_0 cache: 2^-12), every weight's normaliser
    # with it, and both outputs are rounded to bf16 (2^-9 each); fp32 differs by the order of its sums
    bound = (1e-5 if fmt == "f32" else 4 * 2.0 ** -9) * max(1.0, two.float().abs().max().item())
    assert (one.float() - two.float()).abs().max().item() <= bound


@pytest.mark.parametrize("fmt", ["f32", "bf16", "q8_0"])
@pytest.mark.parametrize("B,Hq,Hkv,D", [(1, 8, 2, 64), (2, 32, 8, 128), (1, 16, 16, 64), (40, 16, 16, 128)])
@pytest.mark.parametrize("ctx", [0, 1, 7, 63, 64, 255, 256, 257, 1000, 2304])
def test_one_launch_is_append_and_decode(fmt, B, Hq, Hkv, D, ctx):
    import vesper_amd as va
    caches, q, k, v = _case(fmt, B, Hq, Hkv, D, ctx, False, 11 * ctx + D)
    _compare(fmt, caches, q, k, v, ctx, va.RopeTable(ctx + 1, D) if ctx % 2 == 0 or ctx == 1 else None)


@pytest.mark.parametrize("fmt", ["bf16", "q8_0"])
@pytest.mark.parametrize("Hq,ctx", [(8, 0), (8, 64), (8, 700), (40, 127), (40, 3000)])
def test_paged_and_column_groups(fmt, Hq, ctx):
    import vesper_amd as va
    caches, q, k, v = _case(fmt, 2, Hq, 1 if Hq == 40 else 4, 128, ctx, True, ctx + Hq)
    _compare(fmt, caches, q, k, v, ctx, va.RopeTable(ctx + 1, 128))


@pytest.mark.parametrize("fmt", ["f32", "bf16", "q8_0"])
def test_positions_inside_and_behind_the_context(fmt):
    """A token that is not the last one is left to the two calls; one behind a gap attends to what the planes hold there."""
    import vesper_amd as va
    rope = va.RopeTable(512, 64)
    for pos in (100, 299, 305):
        caches, q, k, v = _case(fmt, 2, 8, 2, 64, 300, False, pos)
        for c in caches:
            for i in range(4):
                if c.raw_plane(i) is not None and pos > 300:
                    c.raw_plane(i).zero_()
        _compare(fmt, caches, q, k, v, pos, rope)


def test_rows_the_step_does_not_take():
    """Unaligned rows and fp32 rows over a bf16 cache go through the two calls, with the same result as before."""
    import vesper_amd as va
    caches, q, k, v = _case("bf16", 1, 8, 2, 64, 100, False, 5)
    big = torch.zeros((1, 2, 1, 68), device="cuda", dtype=torch.bfloat16)
    k2 = big[..., 1:65]
    k2.copy_(k)
    _compare("bf16", caches, q, k2, v, 100, va.RopeTable(128, 64))
    caches, q, k, v = _case("bf16", 1, 8, 2, 64, 100, False, 6)
    out = va.attention_core(q.float(), k.float(), v.float(), caches[0], 100, rope=va.RopeTable(128, 64), q_dtype=torch.bfloat16)
    qr = caches[1].rope_update(q.float(), k.float(), v.float(), 100, va.RopeTable(128, 64), out_dtype=torch.bfloat16)
    assert torch.equal(out, va.decode_attention(qr, caches[1]))


def test_graph_replays():
    """Captured after one eager step of the size; every replay equals the eager result."""
    import vesper_amd as va
    caches, q, k, v = _case("bf16", 1, 32, 8, 128, 2047, False, 9)
    rope = va.RopeTable(2048, 128)
    eager = va.attention_core(q, k, v, caches[0], 2047, rope=rope).clone()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        va.attention_core(q, k, v, caches[0], 2047, rope=rope)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s):
            out = va.attention_core(q, k, v, caches[0], 2047, rope=rope)
    for _ in range(4):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(G.bf16_bits(out), G.bf16_bits(eager))
        va.attention_core(q, k, v, caches[0], 2047, rope=rope)
