"""The native host side of the Python view (vesper_amd/csrc/py_host.cpp): what its per-stream state means to captured
graphs, and what its calls mean to the program's other Python threads."""
import ctypes as C
import threading
import time

import pytest
import torch

import _gpu as G
import _inputs as I

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def va():
    import vesper_amd
    return vesper_amd


def test_other_python_threads_run_while_a_launch_waits_for_room_in_the_queue(va):
    lens = torch.zeros(4, dtype=torch.int32, device=G.dev())
    start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    for _ in range(2):  # the second one is timed: the first pays for loading
        start.record()
        torch.cuda._sleep(1_000_000)
        end.record()
        torch.cuda.synchronize()
    cycles = int(1_000_000 * 1000.0 / start.elapsed_time(end))  # one kernel of about a second
    va._host.advance(lens, None, 0, 4, 8)
    torch.cuda.synchronize()

    def launches():  # more than a hardware queue holds: the last of them wait for the long kernel
        for _ in range(24000):
            va._host.advance(lens, None, 0, 4, 8)

    torch.cuda._sleep(cycles)
    t = threading.Thread(target=launches)
    t0 = last = time.perf_counter()
    gap = 0.0
    t.start()
    while t.is_alive():
        time.sleep(0.001)
        now = time.perf_counter()
        gap, last = max(gap, now - last), now
    took = last - t0
    t.join()
    torch.cuda.synchronize()
    if took < 0.5:
        pytest.skip(f"the launches never waited ({took:.3f} s for all of them)")
    assert gap < 0.3, f"no other thread ran for {gap:.2f} of {took:.2f} s"


def _token_step(va, seed, B, L):
    """A decode step of few splits (one launch, partials merged through the counters), its queries and their eager results."""
    Hq, Hkv, D = 32, 8, 128
    c = va.KVCache(B, Hkv, L, D, fmt="bf16")
    k, v = (G.to_bf16_dev(I.normal(seed + i, (B, Hkv, L, D))) for i in (1, 2))
    c.update(k, v, 0, return_views=False)
    qs = [G.to_bf16_dev(I.normal(seed + 3 + i, (B, Hq, 1, D))) for i in range(4)]
    ws = torch.empty(va._ffi.lib.vsp_attn_decode_workspace_bytes(B, Hq, D, L), dtype=torch.uint8, device=G.dev())
    return c, qs, [va.decode_attention(q, c, workspace=ws).clone() for q in qs]  # through the launch of its own


# several splits merged by the last workgroup; one split, straight to the output
@pytest.mark.parametrize("L", [2000, 200])
def test_a_captured_step_in_the_default_workspace_outlives_its_growth(va, L):
    c, qs, want = _token_step(va, 9100, 1, L)
    big, big_qs, big_want = _token_step(va, 9200, 4, 3000)
    side = torch.cuda.Stream()
    sq, out = torch.empty_like(qs[0]), torch.empty_like(qs[0])
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(side):
        va.decode_attention(qs[0], c)  # sizes the stream's workspace
        torch.cuda.synchronize()
        with torch.cuda.graph(graph, stream=side):
            va.decode_attention(sq, c, out=out)
        size = va.api._WS[("cuda", 0, side.cuda_stream)][0].numel()
        for i, q in enumerate(qs):
            sq.copy_(q)
            out.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, want[i]), f"replay {i}"
            # the program's own work between replays: a step on the same stream, from the second replay on a larger one
            assert torch.equal(va.decode_attention(qs[i - 1], c), want[i - 1])
            if i:
                assert torch.equal(va.decode_attention(big_qs[i], big), big_want[i])
                assert va.api._WS[("cuda", 0, side.cuda_stream)][0].numel() > size
                # whatever the stream's allocations get now is not what the graph writes to
                junk = [torch.full((size,), 0xFF, dtype=torch.uint8, device=G.dev()) for _ in range(4)]
                graph.replay()
                torch.cuda.synchronize()
                assert torch.equal(out, want[i]) and all(bool((j == 0xFF).all()) for j in junk)
                del junk


def test_growth_during_capture_is_refused_and_leaves_the_stream_usable(va):
    c, qs, want = _token_step(va, 9300, 1, 2000)
    side = torch.cuda.Stream()
    out = torch.empty_like(qs[0])
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        refused = None
        with torch.cuda.graph(torch.cuda.CUDAGraph(), stream=side):
            try:
                va.decode_attention(qs[0], c, out=out)
            except RuntimeError as e:
                refused = str(e)
        assert refused and "grow during stream capture" in refused
        assert torch.equal(va.decode_attention(qs[1], c), want[1])
    torch.cuda.synchronize()


@pytest.mark.parametrize("Hq,Hkv,D,T,L", [(16, 4, 128, 39, 848), (8, 2, 64, 124, 3503)])
def test_a_capture_without_room_for_partials_records_the_chunk_unsplit(va, Hq, Hkv, D, T, L):
    """A stream that has no workspace yet: the chunk's attention is recorded as it is without shares of the context, and the stream
    takes the eager call with shares afterwards."""
    c = va.KVCache(1, Hkv, L, D, fmt="bf16")
    c.update(*(G.to_bf16_dev(I.normal(9400 + i, (1, Hkv, L, D))) for i in (1, 2)), 0, return_views=False)
    q = G.to_bf16_dev(I.normal(9403, (1, Hq, T, D)))
    assert va._ffi.lib.vsp_attn_prefill_cached_best_workspace_bytes(C.byref(c._c), 0, 0, Hq, T) > 0  # eager, it is cut into shares
    whole, sq = c.prefill(q, split=False), torch.empty_like(q)
    side, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    va.api._WS.pop(("cuda", 0, side.cuda_stream), None)  # torch hands out its streams in turn
    with torch.cuda.stream(side):
        with torch.cuda.graph(graph, stream=side):
            out = c.prefill(sq)
        for i in range(3):
            sq.copy_(q)
            out.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, whole), f"replay {i}"
            shares = c.prefill(q)  # the program's own work between replays
            G.assert_bf16_close(G.bf16_to_np(shares), G.bf16_to_np(whole), "in shares")
            sq.zero_()
    torch.cuda.synchronize()


def _step(T, Hkv=2, D=64, B=1, fmt="bf16"):
    """A cache, one step's q, k, v (T tokens) and a table long enough for it."""
    import vesper_amd
    g = torch.Generator().manual_seed(T)
    cache = vesper_amd.KVCache(B, Hkv, 64, D, fmt=fmt)
    dt = torch.float32 if fmt == "f32" else torch.bfloat16
    q, k, v = (torch.randn((B, h, T, D), generator=g).to(dt).to(G.dev()) for h in (4 * Hkv, Hkv, Hkv))
    return cache, q, k, v, vesper_amd.RopeTable(64, D)


@pytest.mark.parametrize("T", [1, 5])
@pytest.mark.parametrize("fmt", ["f32", "bf16", "q8_0"])
@pytest.mark.parametrize("which", ["k", "v", "table", "k without a rope", "v without a rope"])
def test_operands_in_host_memory_are_refused_before_anything_is_launched(va, T, fmt, which):
    cache, q, k, v, rope = _step(T, fmt=fmt)
    before = [p.clone() for p in map(cache.raw_plane, range(4)) if p is not None]
    if which[0] == "k":
        k = k.cpu()
    elif which[0] == "v":
        v = v.cpu()
    else:
        rope = va.RopeTable(64, 64, device="cpu")
    with pytest.raises(RuntimeError, match="expected a tensor on the GPU"):
        va.attention_core(q, k, v, cache, 0, rope=None if "without" in which else rope)
    assert cache.current_seq_len() == 0
    torch.cuda.synchronize()
    for p, was in zip((p for p in map(cache.raw_plane, range(4)) if p is not None), before):
        assert torch.equal(p, was)


def test_host_tensors_are_refused_by_every_operator(va):
    cache, q, k, v, rope = _step(3)
    va.attention_core(q, k, v, cache, 0, rope=rope)
    one, lens, host = q[:, :, :1].contiguous(), torch.tensor([3], dtype=torch.int32), lambda t: t.cpu()
    out, lse = va.flash_attention(q, k, v, 0.125, True, return_lse=True)
    f = q.float(), k.float(), v.float()
    fo, fl = va.flash_attention_split(*f, 0.125, True, return_lse=True)
    ws = torch.empty(1 << 20, dtype=torch.uint8)
    calls = [
        lambda: va.flash_attention_split(f[0], host(f[1]), f[2], 0.125),
        lambda: va.flash_attention_split(*f, 0.125, workspace=ws),
        lambda: va.flash_attention_backward(host(out), q, k, v, out, lse, 0.125),
        lambda: va.flash_attention_backward(out, q, k, v, out, host(lse), 0.125),
        lambda: va.flash_attention_backward(out, q, k, v, out, lse, 0.125, workspace=ws),
        lambda: va.flash_attention_backward_split(fo, *f, fo, host(fl), 0.125),
        lambda: cache.update(k, host(v), 0),
        lambda: cache.update(k, v, 0, start_pos_dev=lens),
        lambda: cache.rope_update(q, k, v, 0, rope, out=torch.empty(q.shape, dtype=q.dtype)),
        lambda: cache.prefill(q, seq_lens=lens),
        lambda: cache.prefill(q, chunk_lens=lens),
        lambda: va.decode_attention(one, cache, seq_lens=lens),
        lambda: va.decode_attention(one, cache, out=host(one)),
        lambda: va.decode_attention(one, cache, workspace=ws),
        lambda: va.decode_attention_proj(one, cache, torch.zeros((8, 512), dtype=q.dtype)),
    ]
    for i, call in enumerate(calls):
        with pytest.raises(RuntimeError, match="expected a tensor on the GPU"):
            call()
            print("accepted:", i)
    torch.cuda.synchronize()


@pytest.mark.parametrize("T", [1, 5])
def test_pinned_operands_take_the_two_calls(va, T):
    cache, q, k, v, rope = _step(T)
    two, _, _, _, _ = _step(T)
    want_q = two.rope_update(q, k, v, 0, rope)
    want = va.decode_attention(want_q, two) if T == 1 else two.prefill(want_q)
    pinned = [torch.empty(t.shape, dtype=t.dtype, pin_memory=True).copy_(t) for t in (k, v)]
    assert torch.equal(va.attention_core(q, *pinned, cache, 0, rope=rope), want)
    assert torch.equal(cache.raw_plane(0), two.raw_plane(0)) and torch.equal(cache.raw_plane(1), two.raw_plane(1))
