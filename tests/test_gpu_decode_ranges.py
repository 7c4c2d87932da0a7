"""Ragged batches with their lengths on the device: the context cut into equal ranges over the whole batch, or into one round of splits.  Which of them a
shape takes is asserted against the library's plan (tests/test_abi_and_host.py holds the lists to every kernel instance, without a GPU)."""
import math

import pytest
import torch

import _gpu as G

pytestmark = pytest.mark.gpu


def _reference(c, q, lens, n_rep):
    """fp32 attention of the last T tokens of each row, row by row over what the cache holds."""
    T, D = q.shape[2], q.shape[3]
    kc, vc = c.read(0, max(lens))
    out = torch.zeros(q.shape, device=q.device)
    for b, L in enumerate(lens):
        if L == 0:
            continue
        for t in range(T):
            n = L - (T - 1 - t)
            if n <= 0:
                continue
            k, v = (x[b, :, :n].float().repeat_interleave(n_rep, 0) for x in (kc, vc))
            s = torch.matmul(k, q[b, :, t].float().unsqueeze(-1)).squeeze(-1) / math.sqrt(D)
            out[b, :, t] = torch.matmul(s.softmax(-1).unsqueeze(1), v).squeeze(1)
    return out


def _spread(n, hi, seed):
    g = torch.Generator().manual_seed(seed)
    return torch.randint(0, hi + 1, (n,), generator=g).tolist()


# Batches that are cut into equal ranges (RANGE kernels).
RANGES = [
    ("bf16", 64, 32, 128, 1, 0, [6400, 3, 0, 1, 70, 5], 6400),           # one long row holds nearly every range
    ("bf16", 32, 32, 128, 1, 0, [3, 0, 1, 65, 2, 0], 6400),              # fewer groups than workgroups
    ("bf16", 16, 16, 64, 1, 0, [0, 1, 64, 65, 4160, 4159, 4097] + _spread(8, 4160, 16), 4160),   # empty and tiny rows between long ones
    ("bf16", 16, 16, 64, 2, 64, _spread(15, 4160, 17), 4160),
    ("bf16", 8, 4, 64, 1, 64, _spread(64, 4160, 1), 4160),               # as many rows as lanes, paged
    ("bf16", 32, 8, 128, 1, 0, [0, 1] + _spread(28, 4160, 18), 4160),
    ("f32", 16, 16, 64, 2, 0, [0, 63] + _spread(13, 4160, 19), 4160),
    ("f32", 32, 8, 128, 1, 0, _spread(30, 4160, 20), 4160),
    # about one length: even parts (six of a row), whole rows
    ("bf16", 16, 8, 128, 1, 0, [4480, 4479, 4417, 4416] + [4300 + 7 * i for i in range(22)], 4480),
    ("bf16", 16, 8, 64, 2, 64, [4480] * 25 + [4033], 4480),
    ("f32", 16, 8, 128, 1, 0, [4480, 4479, 4417, 4416] + [4300 + 7 * i for i in range(22)], 4480),
    ("f32", 8, 4, 64, 1, 0, [8192 - i for i in range(64)], 8192),
    # bounds well above the rows: parts of one length where they are hardly longer than a range, else short ranges
    ("bf16", 32, 8, 128, 4, 0, [0, 3, 11980] + _spread(3, 12000, 6), 48000),
    ("bf16", 12, 12, 64, 1, 64, _spread(8, 3000, 7), 24000),
    ("f32", 32, 8, 128, 2, 0, _spread(27, 1600, 9), 8192),
    ("f32", 64, 8, 64, 1, 0, _spread(26, 3000, 10), 8192),
    ("f32", 8, 4, 64, 2, 0, [4000] + [0] * 62 + [1], 8192),
]
# Bounds of one to sixteen rounds of the plan's splits: a ragged batch's splits are as long as it takes to make one round, or two of many rows.
ROUND = [
    ("bf16", 32, 8, 128, 4, 256, [8000, 500, 4321, 64, 7999, 1, 6500, 3000], 8000),
    ("bf16", 32, 32, 128, 1, 0, [4500, 0, 2113], 4544),                        # 3/8 as many rows as splits
    ("bf16", 32, 32, 128, 4, 256, [4500, 0, 2113, 64, 2300, 4499], 4608),      # 3/4
    ("q8_0", 16, 16, 128, 1, 64, _spread(11, 6482, 13), 6528),
    ("q8_0", 64, 8, 128, 1, 0, [9681] + [1] * 22, 9728),                       # one long row
    ("bf16", 16, 16, 128, 1, 256, _spread(12, 4160, 14), 4160),                # as many rows as the rule takes
    ("f32", 10, 10, 128, 1, 0, _spread(17, 4160, 15), 4160),
    ("bf16", 16, 16, 64, 2, 64, [9000, 1, 0, 64, 65], 9024),                   # one long row holds the round, empty rows in it
    ("bf16", 64, 8, 128, 1, 0, [1] * 8 + [6451], 6464),
    ("bf16", 8, 1, 128, 1, 64, [60000, 3, 12801], 60032),                      # one kv head: over a hundred splits of a row
    ("f32", 8, 1, 64, 1, 0, [3, 12801, 60000], 60032),
    ("q8_0", 8, 1, 64, 1, 64, [300000, 40001, 0, 3, 300], 300032),             # two workgroups a CU
    ("f32", 8, 2, 128, 1, 0, [5, 29990, 100, 0, 64, 1], 60032),                # one long row makes all the splits
    ("bf16", 32, 8, 128, 2, 0, [9000, 5, 100, 0, 64, 1], 20480),
    ("q8_0", 16, 4, 128, 2, 0, [20000, 7001, 64, 15999, 0, 128], 20032),
    ("q8_0", 32, 8, 64, 1, 64, _spread(20, 6000, 11), 6016),
    ("q8_0", 32, 8, 64, 1, 0, _spread(20, 6000, 21), 6016),
    ("q8_0", 32, 8, 128, 1, 0, [300, 200, 100, 30], 30016),                    # far below the bound: no round yet
    ("q8_0", 32, 8, 128, 1, 0, [27000, 26999, 26900, 27003], 27072),           # about one length: equal parts
    ("f32", 16, 16, 64, 4, 0, [1490, 253, 700, 64, 63, 0], 1500),
    ("f32", 32, 8, 64, 4, 0, _spread(8, 2500, 22), 2500),                      # sixteen columns
    ("f32", 64, 8, 128, 1, 0, _spread(12, 2900, 12), 2944),
    # and what is not too large a batch for it, however long its rows
    ("bf16", 16, 16, 64, 1, 0, [0, 1, 64, 20000, 9999], 20032),
    ("bf16", 8, 2, 64, 1, 64, _spread(64, 8192, 1), 8192),
    ("q8_0", 8, 2, 128, 1, 0, _spread(64, 8192, 2), 8192),
    ("bf16", 16, 4, 64, 4, 256, [15000, 700, 3, 64, 30000, 8000, 1, 29999, 257, 12001], 30208),   # several tokens, longer than some rows
    ("f32", 8, 8, 64, 2, 0, [25000, 1, 12345, 63], 25024),
    ("f32", 16, 4, 128, 1, 0, _spread(20, 11000, 3), 11008),
    ("bf16", 32, 8, 128, 1, 0, [20480, 20479, 20417, 20416, 20000, 20480, 20300, 19999], 20480),
    ("q8_0", 32, 8, 128, 1, 0, [16384] * 16, 16384),
    ("bf16", 32, 8, 128, 1, 0, _spread(8, 6525, 5), 26112),
    ("bf16", 16, 4, 128, 1, 0, _spread(24, 5000, 8), 20032),
    ("bf16", 8, 2, 64, 2, 0, [4000] + [0] * 62 + [1], 8192),
    ("f32", 16, 4, 128, 2, 0, _spread(7, 6525, 9), 52224),
    ("f32", 8, 2, 64, 1, 0, _spread(32, 3000, 10), 12032),
    ("f32", 8, 8, 64, 1, 0, [13000, 12999, 12990, 13000, 12801, 12930, 12800], 13056),
]
# Neither.
SPLITS = [
    ("q8_0", 16, 4, 64, 4, 64, _spread(12, 20000, 4), 20032),
    ("q8_0", 16, 16, 128, 1, 0, _spread(13, 4160, 15), 4160),                  # one row more than the rule for rounds takes
    ("f32", 16, 16, 128, 2, 0, _spread(12, 2449, 14), 2496),                   # whole rows
    ("bf16", 8, 1, 128, 1, 64, [40000, 3, 12801], 40000),                      # less than a round
    ("q8_0", 8, 1, 64, 1, 0, [100000, 40001], 100032),
]


def _cache(fmt, B, Hkv, D, page, S):
    import vesper_amd as va
    if not page:
        return va.KVCache(B, Hkv, S, D, fmt=fmt)
    S = -(-S // page) * page
    c = va.KVCache(B, Hkv, S, D, fmt=fmt, paging=(page, B * (S // page)))
    c.page_table.copy_(torch.randperm(B * (S // page), generator=torch.Generator().manual_seed(7)).to(torch.int32).view(B, -1))
    return c


def _check(kind, fmt, Hq, Hkv, D, T, page, lens, bound):
    import vesper_amd as va
    from vesper_amd import _ffi
    B = len(lens)
    c = _cache(fmt, B, Hkv, D, page, max(bound, max(lens)))
    p = G.decode_plan(c, Hq, T, bound)
    assert kind == ("ranges" if p.ranges else "round" if p.round else "splits")
    g = torch.Generator(device="cuda").manual_seed(B * D + T)
    dt = torch.float32 if fmt == "f32" else torch.bfloat16
    for t in range(0, c._c.S_max, 4096):
        n = min(4096, c._c.S_max - t)
        c.update(*(torch.randn((B, Hkv, n, D), device="cuda", generator=g).to(dt) for _ in range(2)), t, return_views=False)
    q = torch.randn((B, Hq, T, D), device="cuda", generator=g).to(dt)
    sl = torch.tensor(lens, dtype=torch.int32, device="cuda")
    ws = torch.empty(_ffi.lib.vsp_attn_decode_workspace_bytes(B * T, Hq, D, bound), dtype=torch.uint8, device="cuda")
    step = va.decode_attention if T == 1 else va.decode_attention_multi
    two = step(q, c, seq_lens=sl, max_len=bound, workspace=ws)
    for _ in range(3):  # the counters are back at zero after each call
        assert torch.equal(step(q, c, seq_lens=sl, max_len=bound), two)
    outs = [two]
    if T == 1:
        out = torch.empty_like(q)
        assert torch.equal(va.decode_attention_noalloc(q, c, out, seq_lens=sl, max_len=bound), two)
        odd = torch.zeros(B, Hq, 1, D + 1, dtype=dt, device="cuda")  # output rows that are not aligned: splits, merged a lane an element
        va.decode_attention(q, c, seq_lens=sl, max_len=bound, out=odd[..., :D])
        assert not odd[..., D].any()
        outs.append(odd[..., :D])
    want = _reference(c, q, lens, Hq // Hkv)
    for out in outs:
        err = (out.float() - want).norm(dim=-1) / want.norm(dim=-1).clamp_min(1e-3)
        # bf16: P and the output are rounded (2^-9 each); a row's error is at most a few of those relative to its norm
        assert err.max().item() < (2e-5 if fmt == "f32" else 2e-2)


@pytest.mark.parametrize("fmt,Hq,Hkv,D,T,page,lens,bound", RANGES)
def test_ranges(fmt, Hq, Hkv, D, T, page, lens, bound):
    _check("ranges", fmt, Hq, Hkv, D, T, page, lens, bound)


@pytest.mark.parametrize("fmt,Hq,Hkv,D,T,page,lens,bound", ROUND)
def test_one_round(fmt, Hq, Hkv, D, T, page, lens, bound):
    _check("round", fmt, Hq, Hkv, D, T, page, lens, bound)


@pytest.mark.parametrize("fmt,Hq,Hkv,D,T,page,lens,bound", SPLITS)
def test_neither(fmt, Hq, Hkv, D, T, page, lens, bound):
    _check("splits", fmt, Hq, Hkv, D, T, page, lens, bound)


def _splits_made(fmt, Hq, Hkv, D, T, page, lens, bound):
    """Splits of each row (of one kv head) that a call in two launches leaves partials of, and its plan."""
    import vesper_amd as va
    from vesper_amd import _ffi
    B = len(lens)
    c = _cache(fmt, B, Hkv, D, page, bound)
    plan = G.decode_plan(c, Hq, T, bound)
    assert plan.round, "not cut into a round"
    q = torch.zeros((B, Hq, T, D), device="cuda", dtype=torch.float32 if fmt == "f32" else torch.bfloat16)
    need = B * Hq * T * plan.max_splits * (D + 2)
    assert 4 * need <= _ffi.lib.vsp_attn_decode_workspace_bytes(B * T, Hq, D, bound)
    ws = torch.full((_ffi.lib.vsp_attn_decode_workspace_bytes(B * T, Hq, D, bound) // 4,), 1e30, device="cuda")
    (va.decode_attention if T == 1 else va.decode_attention_multi)(
        q, c, seq_lens=torch.tensor(lens, dtype=torch.int32, device="cuda"), max_len=bound, workspace=ws.view(torch.uint8))
    ml = ws[B * Hq * T * plan.max_splits * D:need].view(B, Hq, T, plan.max_splits, 2)
    made = (ml[:, 0, 0, :, 1] != 1e30).sum(-1).tolist()
    assert all(n <= plan.max_splits for n in made) and sum(made) * Hkv <= plan.workgroups
    return made, plan


# The host's bound says how long a row may be, not how long the rows are: they make about a workgroup per CU whatever it is.
@pytest.mark.parametrize("bound", [12000, 24000])
@pytest.mark.parametrize("fmt,Hkv,D,T,page,lens", [
    ("bf16", 8, 64, 2, 256, [3000, 1415, 2900, 2000, 2222, 1500, 2700]),
    ("q8_0", 4, 128, 1, 64, [2999, 689, 3000, 1, 2000, 64, 1500, 2500, 1900, 2048]),
    ("bf16", 8, 128, 1, 256, [1000, 3000, 2000, 1500, 100, 2500]),
])
def test_a_round_follows_the_lengths_not_their_bound(fmt, Hkv, D, T, page, lens, bound):
    made, plan = _splits_made(fmt, 4 * Hkv, Hkv, D, T, page, lens, bound)
    shortest = sum(-(-n // 256) for n in lens)  # in the shortest splits there are
    assert sum(made) * 10 >= min(plan.round, shortest) * 7, made
    _check("round", fmt, 4 * Hkv, Hkv, D, T, page, lens, bound)


# Keys of 64 bytes make rounds of two workgroups a CU; splits shorter than the plan's make one.
@pytest.mark.parametrize("Hkv,T,page,lens,bound", [
    (12, 1, 0, [658, 2111, 1900, 1500, 2000, 1203, 1777, 900, 2048], 4224),
    (16, 1, 64, [18054, 1, 300, 9000, 12000, 64, 7000, 15000, 0, 50, 3000, 11000, 500], 72192),
    (2, 4, 0, [44808, 18, 30000, 100, 41000, 300, 38000, 25000], 179200),
])
def test_shorter_splits_of_narrow_keys_make_a_workgroup_per_cu(Hkv, T, page, lens, bound):
    made, plan = _splits_made("q8_0", Hkv, Hkv, 64, T, page, lens, bound)
    short = sum(n * 24 <= max(lens) for n in lens)  # more than those that are not counted (is_short)
    whole = sum(-(-n // plan.chunk) for n in lens)
    assert sum(made) <= max(256 // Hkv + short, whole), made
    _check("round", "q8_0", Hkv, Hkv, 64, T, page, lens, bound)


# Short rows come last and are not counted as splits of the round: a long row is cut as it would be without them, wherever it stands.
@pytest.mark.parametrize("where", [0, 7, 15])
@pytest.mark.parametrize("fmt,D,page,hi", [("q8_0", 128, 0, 24000), ("bf16", 128, 256, 12000), ("f32", 128, 0, 16000)])
def test_short_rows_of_a_round(fmt, D, page, hi, where):
    lens = [100, 0, 1, 64, 65, 128, 127, 2, 90, 0, 101, 63, 99, 126, 110]
    lens.insert(where, hi)
    made, plan = _splits_made(fmt, 32, 8, D, 1, page, lens, hi)
    assert made[where] * 10 >= min(plan.round, plan.max_splits) * 8 and all(n == (L > 0) for L, n in zip(lens, made) if L < hi), made
    _check("round", fmt, 32, 8, D, 1, page, lens, hi)


@pytest.mark.parametrize("kind,B,S,most", [("ranges", 28, 4160, 4160), ("ranges", 64, 4160, 900), ("round", 8, 16384, 16384), ("round", 8, 16384, 2000)])
def test_under_a_graph(kind, B, S, most):
    import vesper_amd as va
    Hkv, D = 8, 64
    g = torch.Generator(device="cuda").manual_seed(3)
    c = va.KVCache(B, Hkv, S, D, fmt="bf16")
    p = G.decode_plan(c, 16, 1, S)
    assert kind == ("ranges" if p.ranges else "round" if p.round else "splits")
    c.update(*(torch.randn((B, Hkv, S, D), device="cuda", generator=g).to(torch.bfloat16) for _ in range(2)), 0, return_views=False)
    q = torch.randn((B, 16, 1, D), device="cuda", generator=g).to(torch.bfloat16)
    lens = torch.tensor(_spread(B, most, 9), dtype=torch.int32, device="cuda")
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        va.decode_attention(q, c, seq_lens=lens, max_len=S)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s):
            out = va.decode_attention(q, c, seq_lens=lens, max_len=S)
    for i in range(4):  # the lengths are read by each replay
        lens.copy_(torch.tensor(_spread(B, most // (1 + i % 2), 20 + i), dtype=torch.int32))
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, va.decode_attention(q, c, seq_lens=lens, max_len=S))
