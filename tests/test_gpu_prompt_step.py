"""The first forward of a prompt with Q rotated inside the attention kernel, against rope_update + prefill."""
import pytest
import torch

import _gpu as G

pytestmark = pytest.mark.gpu


def _both(fmt, B, Hq, Hkv, D, T, paged=False, extra=64, seed=0):
    import vesper_amd as va
    g = torch.Generator(device="cuda").manual_seed(seed + T)
    S = -(-T // 64) * 64 + extra
    caches = []
    for _ in range(2):
        if paged:
            c = va.KVCache(B, Hkv, S, D, fmt=fmt, paging=(64, B * (S // 64)))
            c.page_table.copy_(torch.arange(B * (S // 64), dtype=torch.int32).flip(0).view(B, -1))
        else:
            c = va.KVCache(B, Hkv, S, D, fmt=fmt)
        caches.append(c)
    fused = torch.randn((B, T, Hq + 2 * Hkv, D), device="cuda", generator=g).to(torch.bfloat16)
    q, k, v = (fused[:, :, a:b].transpose(1, 2) for a, b in ((0, Hq), (Hq, Hq + Hkv), (Hq + Hkv, Hq + 2 * Hkv)))
    rope = va.RopeTable(S, D)
    one = va.attention_core(q, k, v, caches[0], 0, rope=rope)
    two = caches[1].prefill(caches[1].rope_update(q, k, v, 0, rope))
    assert caches[0].current_seq_len() == caches[1].current_seq_len() == T
    for i in range(4):
        if caches[0].raw_plane(i) is not None:
            assert torch.equal(caches[0].raw_plane(i), caches[1].raw_plane(i)), i
    return one, two


# a short prompt takes the key-group shape of the kernel here and another one there: P's sums are then taken in another order, so the
# outputs (of order one: averages of N(0, 1) rows) may differ by a bf16 step, 2^-8 of the value, plus what P's rounding (2^-9) adds
def _check(one, two, same_shape):
    assert torch.isfinite(two).all()
    if same_shape:
        assert torch.equal(one, two)
    else:
        assert ((one.float() - two.float()).abs() <= 2.0 ** -7 * two.float().abs().clamp_min(1.0)).all()


@pytest.mark.parametrize("D,Hq,Hkv", [(128, 32, 8), (64, 12, 12), (128, 4, 1)])
@pytest.mark.parametrize("T", [2, 7, 31, 32, 33, 64, 65, 96, 97, 128, 129, 300, 777])
def test_prompt_bf16(D, Hq, Hkv, T):
    _check(*_both("bf16", 2, Hq, Hkv, D, T), same_shape=T <= 32 or T > 128)


# with what some of them run: row groups, pipelined or not, shares of the context
@pytest.mark.parametrize("fmt,B,Hq,Hkv,D,T,paged,plan", [
    ("bf16", 1, 32, 8, 128, 900, False, (2, 0, 1)), ("bf16", 4, 32, 8, 128, 600, False, (4, 0, 1)),
    ("bf16", 1, 32, 8, 128, 1500, False, (4, 1, 1)), ("bf16", 1, 32, 8, 128, 2601, False, (4, 1, 1)),
    ("bf16", 1, 4, 2, 128, 4096, False, (1, 0, 1)), ("bf16", 1, 1, 1, 128, 4096, False, (1, 0, 4)),
    ("bf16", 3, 16, 16, 64, 1300, False, (2, 0, 1)), ("bf16", 3, 32, 8, 64, 5000, False, (4, 0, 1)),
    ("bf16", 2, 8, 2, 128, 500, True, (1, 0, 1)), ("bf16", 2, 32, 8, 128, 2700, True, (4, 1, 1)), ("bf16", 2, 8, 2, 64, 130, True, (1, 0, 1)),
    ("q8_0", 2, 8, 2, 64, 300, False, (1, 0, 1)), ("q8_0", 1, 32, 8, 128, 777, False, (2, 0, 1)), ("q8_0", 1, 32, 8, 128, 2601, False, (4, 1, 1)),
    ("q8_0", 2, 8, 2, 128, 31, True, (4, 0, 1)),
])
def test_prompt_shapes_and_formats(fmt, B, Hq, Hkv, D, T, paged, plan):
    import vesper_amd as va
    p = G.cached_plan(va.KVCache(B, Hkv, T, D, fmt=fmt), Hq, T, prompt=True)
    assert (p.row_groups, p.pipelined, p.shares) == plan
    _check(*_both(fmt, B, Hq, Hkv, D, T, paged), same_shape=True)


def test_prompts_the_step_does_not_take():
    """A cache that is longer than the prompt, or a prompt that does not start it, fails as it did, with the rows written."""
    import vesper_amd as va
    rope = va.RopeTable(256, 64)
    q, k, v = (torch.randn((1, h, 40, 64), device="cuda").to(torch.bfloat16) for h in (4, 2, 2))
    for start, have in ((0, 60), (5, 0)):
        c = va.KVCache(1, 2, 128, 64, fmt="bf16")
        if have:
            c.update(torch.randn((1, 2, have, 64), device="cuda"), torch.randn((1, 2, have, 64), device="cuda"), 0, return_views=False)
        with pytest.raises(va.VspError):
            va.attention_core(q, k, v, c, start, rope=rope)
        ref = va.KVCache(1, 2, 128, 64, fmt="bf16")
        ref.rope_update(q, k, v, start, rope)
        for plane_a, plane_b in zip(c.read(start, 40), ref.read(start, 40)):
            assert torch.equal(plane_a, plane_b)
    # rows that are not 16-byte aligned go through the two calls
    big = torch.zeros((1, 4, 40, 68), device="cuda", dtype=torch.bfloat16)
    q2 = big[..., 1:65]
    q2.copy_(q)
    a, b = (va.KVCache(1, 2, 64, 64, fmt="bf16") for _ in range(2))
    assert torch.equal(va.attention_core(q2, k, v, a, 0, rope=rope), b.prefill(b.rope_update(q, k, v, 0, rope)))


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("T", [2, 7, 8, 15, 16, 17, 47, 250])   # below 8 tokens the append is per element and the rows are read out
@pytest.mark.parametrize("paged", [False, True])
def test_prompt_q8_rows_left_for_the_attention(D, T, paged):
    # the append leaves the Q8_0 rows as a read gives them: the same outputs bit for bit, magnitudes that use all of the scales' range too
    import vesper_amd as va
    _check(*_both("q8_0", 2, 6, 2, D, T, paged, seed=5), same_shape=T <= 32 or T > 128)
    g = torch.Generator(device="cuda").manual_seed(T)
    rope = va.RopeTable(256, D)
    q, k, v = (torch.randn((1, h, T, D), device="cuda", generator=g) for h in (2, 1, 1))
    k, v = k * 1e-6, v * 10.0 ** torch.randint(-6, 5, (1, 1, T, 1), device="cuda", generator=g)
    q, k, v = (x.to(torch.bfloat16) for x in (q, k, v))
    a, b = (va.KVCache(1, 1, 256, D, fmt="q8_0") for _ in range(2))
    one, two = va.attention_core(q, k, v, a, 0, rope=rope), b.prefill(b.rope_update(q, k, v, 0, rope))
    if T <= 32 or T > 128:
        assert torch.equal(one, two)
    assert torch.isfinite(one).all()


# fp32: append with Q rotated and the attention over the planes in one host call, against the same two calls by themselves, bit for bit
@pytest.mark.parametrize("B,Hq,Hkv,D,T", [(1, 8, 2, 64, 2), (2, 4, 4, 128, 33), (1, 6, 2, 32, 70), (1, 4, 1, 80, 40), (2, 32, 8, 128, 300)])
def test_prompt_fp32(B, Hq, Hkv, D, T):
    import vesper_amd as va
    g = torch.Generator(device="cuda").manual_seed(T)
    fused = torch.randn((B, T, Hq + 2 * Hkv, D), device="cuda", generator=g)
    q, k, v = (fused[:, :, a:b].transpose(1, 2) for a, b in ((0, Hq), (Hq, Hq + Hkv), (Hq + Hkv, Hq + 2 * Hkv)))
    rope = va.RopeTable(T + 64, D)
    one, two = (va.KVCache(B, Hkv, T + 9, D, fmt="f32") for _ in range(2))
    got = va.attention_core(q, k, v, one, 0, rope=rope)
    rotated = two.rope_update(q, k, v, 0, rope)
    assert torch.equal(got, va.flash_attention(rotated, *two.views(), D ** -0.5, is_causal=True))
    assert one.current_seq_len() == T and all(torch.equal(one.raw_plane(i), two.raw_plane(i)) for i in range(2))
    one.set_len(T + 5)   # a cache that is further along: the scores would have more keys than the mask, refused as before
    with pytest.raises(va.VspError):
        va.attention_core(q, k, v, one, 0, rope=rope)
