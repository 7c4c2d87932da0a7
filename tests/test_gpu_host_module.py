"""The native host side of the Python view (vesper_amd/csrc/py_host.cpp): what its per-stream state means to captured
graphs, and what its calls mean to the program's other Python threads."""
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
