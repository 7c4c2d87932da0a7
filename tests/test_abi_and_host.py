"""CPU-side checks of the product: the C-ABI library loads and exports every symbol include/vsp_attn.h
declares, the host-side format helpers are bit-exact against the oracle, and argument validation that needs
no GPU behaves like the reference.  No compute kernel is launched here."""
import ctypes as C
import os
import re
import subprocess

import numpy as np
import pytest

import _oracle as O

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def ffi():
    from vesper_amd import _ffi
    return _ffi


def test_library_exports_every_declared_symbol(ffi):
    header = open(os.path.join(ROOT, "include", "vsp_attn.h")).read()
    declared = set(re.findall(r"\b(vsp_[a-z0-9_]+)\s*\(", header))
    declared -= {"vsp_tensor", "vsp_kv_cache"}
    assert declared == set(ffi.SYMBOLS), declared ^ set(ffi.SYMBOLS)
    for name in declared:
        assert hasattr(ffi.lib, name), name
    assert ffi.lib.vsp_attn_abi_version() == 2


def test_status_strings_are_the_reference_messages(ffi):
    assert ffi.lib.vsp_status_str(0) == b"ok"
    for code in (1, 2, 3, 4, 5):  # same numbering and text as the oracle's restatement of the reference throws
        assert ffi.lib.vsp_status_str(code) == O.orc.orc_strerror(code)
    assert ffi.lib.vsp_status_str(7) == O.orc.orc_strerror(7)


def test_host_bf16_f16_bit_exact(ffi):
    rng = np.random.default_rng(0)
    bits = rng.integers(0, 2**32, size=30000, dtype=np.uint64).astype(np.uint32)
    f = bits.view(np.float32)
    f = f[~np.isnan(f)]
    assert all(ffi.lib.vsp_f32_to_bf16(float(x)) == O.orc.orc_f32_to_bf16(float(x)) for x in f[:5000])
    with np.errstate(over="ignore"):
        want = f.astype(np.float16).view(np.uint16)
    got = np.array([ffi.lib.vsp_f32_to_f16(float(x)) for x in f[:20000]], np.uint16)
    assert np.array_equal(got, want[:20000])
    small = (rng.standard_normal(5000) * 1e-5).astype(np.float32)
    assert all(ffi.lib.vsp_f32_to_f16(float(x)) == int(np.float16(x).view(np.uint16)) for x in small)
    for h in list(range(0, 65536, 7)) + [0x0001, 0x03FF, 0x0400, 0x7BFF, 0x7C00, 0xFC00, 0x8001]:
        w = np.uint16(h).view(np.float16).astype(np.float32)
        if not np.isnan(w):
            assert np.float32(ffi.lib.vsp_f16_to_f32(h)).view(np.uint32) == w.view(np.uint32), hex(h)


def test_host_q8_0_matches_oracle(ffi):
    rng = np.random.default_rng(1)
    x = np.concatenate([rng.standard_normal((40, 128)).astype(np.float32), np.zeros((2, 128), np.float32),
                        (rng.standard_normal((8, 128)) * 1e-6).astype(np.float32)])
    want_d, want_q = O.q8_0_quantize(x)
    d = np.empty_like(want_d)
    q = np.empty_like(want_q)
    ffi.lib.vsp_q8_0_quantize_row(x.ctypes.data, x.size, d.ctypes.data, q.ctypes.data)
    assert np.array_equal(d, want_d) and np.array_equal(q, want_q)
    back = np.empty_like(x)
    ffi.lib.vsp_q8_0_dequantize_row(d.ctypes.data, q.ctypes.data, x.size, back.ctypes.data)
    assert np.array_equal(back, O.q8_0_dequantize(want_d, want_q))


def test_slice_and_gqa_config_match_oracle(ffi):
    for dim in (0, 1, 16):
        for start in range(-20, 21):
            for T in (0, 1, 5):
                s, n = C.c_int64(), C.c_int64()
                ffi.lib.vsp_slice_bounds(dim, start, start + T, C.byref(s), C.byref(n))
                ws, wn = O.slice_bounds(dim, start, start + T, 1)
                assert (n.value, s.value if n.value else 0) == (wn, ws if wn else 0), (dim, start, T)
    hd, nr = C.c_int64(), C.c_int64()
    assert ffi.lib.vsp_gqa_config(64, 8, 2, C.byref(hd), C.byref(nr)) == 0 and (hd.value, nr.value) == (8, 4)
    assert ffi.lib.vsp_gqa_config(64, 8, 3, None, None) == ffi.ERR_GQA_HEADS
    assert ffi.lib.vsp_gqa_config(60, 8, 2, None, None) == ffi.ERR_GQA_EMBED


def test_plane_sizes_follow_the_documented_layouts(ffi):
    pb = ffi.lib.vsp_kv_plane_bytes
    assert pb(ffi.KV_F32, 2, 3, 100, 64, 0) == 2 * 3 * 100 * 64 * 4 and pb(ffi.KV_F32, 2, 3, 100, 64, 2) == 0
    assert pb(ffi.KV_BF16, 2, 3, 100, 64, 1) == 2 * 3 * 128 * 64 * 2  # S_pad = 128
    assert pb(ffi.KV_Q8_0, 1, 8, 65536, 128, 0) == 8 * 65536 * 128 and pb(ffi.KV_Q8_0, 1, 8, 65536, 128, 3) == 8 * 65536 * 4 * 2


def test_validation_that_needs_no_gpu(ffi):
    t = ffi.VspTensor()
    t.ndim, t.dtype = 3, ffi.BF16
    assert ffi.lib.vsp_attn_prefill(C.byref(t), C.byref(t), C.byref(t), C.byref(t), None, 1.0, 1, 0.0, 0, None) == ffi.ERR_NDIM
    assert ffi.lib.vsp_attn_prefill(None, None, None, None, None, 1.0, 1, 0.0, 0, None) == ffi.ERR_NULL
    q, k = ffi.VspTensor(), ffi.VspTensor()
    for d, shape in ((q, (1, 4, 8, 64)), (k, (1, 2, 9, 64))):
        d.ndim, d.dtype = 4, ffi.BF16
        for i, s in enumerate(shape):
            d.shape[i] = s
    assert ffi.lib.vsp_attn_prefill(C.byref(q), C.byref(k), C.byref(q), C.byref(q), None, 1.0, 1, 0.0, 0, None) == ffi.ERR_SHAPE
    assert ffi.lib.vsp_attn_prefill(C.byref(q), C.byref(k), C.byref(k), C.byref(q), None, 1.0, 1, 1.5, 0, None) == ffi.ERR_DROPOUT
    c = ffi.VspKVCache()
    c.format, c.B, c.Hkv, c.S_max, c.D = 7, 1, 1, 8, 64
    assert ffi.lib.vsp_kv_cache_reset(C.byref(c), None) == ffi.ERR_UNSUPPORTED
    c.format = ffi.KV_BF16
    assert ffi.lib.vsp_kv_cache_reset(C.byref(c), None) == ffi.ERR_NULL  # planes missing


def test_backward_validation_that_needs_no_gpu(ffi):
    # every rejection below is decided on the host before anything is launched (the pointers are never followed)
    def tens(shape, dtype, ptr=0x10000, strides=None):
        t = ffi.VspTensor()
        t.ndim, t.dtype, t.data = len(shape), dtype, ptr
        st = strides or [int(np.prod(shape[i + 1:])) for i in range(len(shape))]
        for i, (n, m) in enumerate(zip(shape, st)):
            t.shape[i], t.stride[i] = n, m
        return t

    def call(dout, q, k, v, out, lse, dq, dk, dv, ws=0x20000, ws_bytes=1 << 30):
        a = [C.byref(x) if x is not None else None for x in (dout, q, k, v, out, lse, dq, dk, dv)]
        return ffi.lib.vsp_attn_prefill_backward(*a, 0.125, 1, ws, ws_bytes, None)

    B, Hq, Hkv, N, D = 1, 4, 2, 8, 64
    q, k, lse = tens((B, Hq, N, D), ffi.BF16), tens((B, Hkv, N, D), ffi.BF16), tens((B, Hq, N), ffi.F32)
    assert ffi.lib.vsp_attn_backward_workspace_bytes(B, Hq, N) == 2 * B * Hq * N * 4
    assert ffi.lib.vsp_attn_backward_workspace_bytes(0, Hq, N) == 0
    assert call(q, None, k, k, q, lse, q, k, k) == ffi.ERR_NULL
    assert call(q, tens((B, Hq, N), ffi.BF16), k, k, q, lse, q, k, k) == ffi.ERR_NDIM
    k3 = tens((B, 3, N, D), ffi.BF16)
    assert call(q, q, k3, k3, q, lse, q, k3, k3) == ffi.ERR_SHAPE                       # 4 query heads over 3 kv heads
    assert call(q, q, k, tens((B, Hkv, N + 1, D), ffi.BF16), q, lse, q, k, k) == ffi.ERR_SHAPE
    assert call(q, q, k, tens((B, Hkv, N, D), ffi.F32), q, lse, q, k, k) == ffi.ERR_DTYPE  # one dtype for all
    assert call(q, q, k, k, q, tens((B, Hq, N), ffi.BF16), q, k, k) == ffi.ERR_DTYPE       # lse is fp32
    q32, k32 = tens((B, Hq, N, 32), ffi.BF16), tens((B, Hkv, N, 32), ffi.BF16)
    assert call(q32, q32, k32, k32, q32, lse, q32, k32, k32) == ffi.ERR_UNSUPPORTED        # head dim 32
    assert call(q, q, k, k, q, lse, q, k, k, ws=None) == ffi.ERR_WORKSPACE
    assert call(q, q, k, k, q, lse, q, k, k, ws_bytes=16) == ffi.ERR_WORKSPACE
    off = tens((B, Hq, N, D), ffi.BF16, ptr=0x10008)                                       # rows not 16-byte aligned
    assert call(q, off, k, k, q, lse, q, k, k) == ffi.ERR_ALIGN
    narrow = tens((B, Hq, N, D), ffi.BF16, strides=[Hq * N * 32, N * 32, 32, 1])           # rows overlap: stride < D
    assert call(q, narrow, k, k, q, lse, q, k, k) == ffi.ERR_STRIDE
    inner = tens((B, Hq, N, D), ffi.BF16, strides=[Hq * N * D * 2, N * D * 2, D * 2, 2])   # innermost stride != 1
    assert call(q, inner, k, k, q, lse, q, k, k) == ffi.ERR_STRIDE
    empty = tens((B, Hq, 0, D), ffi.BF16)
    ek, el = tens((B, Hkv, 0, D), ffi.BF16), tens((B, Hq, 0), ffi.F32)
    assert call(empty, empty, ek, ek, empty, el, empty, ek, ek) == 0                       # nothing to do


def test_cache_descriptor_validation_that_needs_no_gpu(ffi):
    # check_cache (behind every cache entry point) through vsp_kv_cache_reset, plus the argument checks of
    # vsp_kv_read and vsp_seq_lens_advance that come before any launch
    def cache(fmt=None, **kw):
        c = ffi.VspKVCache()
        c.format, c.B, c.Hkv, c.S_max, c.D = ffi.KV_BF16 if fmt is None else fmt, 2, 2, 256, 128
        c.k = c.v = c.k_scale = c.v_scale = 0x10000
        for key, val in kw.items():
            setattr(c, key, val)
        return c

    reset = lambda c: ffi.lib.vsp_kv_cache_reset(C.byref(c), None)
    assert reset(cache(len=257)) == ffi.ERR_ARG                      # length beyond the capacity
    assert reset(cache(D=96)) == ffi.ERR_UNSUPPORTED                 # bf16 / q8_0 planes exist for D 64 and 128
    assert reset(cache(fmt=ffi.KV_F32, D=6)) == ffi.ERR_UNSUPPORTED
    assert reset(cache(k=0x10008)) == ffi.ERR_ALIGN
    assert reset(cache(fmt=ffi.KV_Q8_0, k_scale=None)) == ffi.ERR_NULL
    paged = dict(page_table=0x30000, page_tokens=64, pages_per_seq=4, n_pages=10)
    assert reset(cache(fmt=ffi.KV_F32, **paged)) == ffi.ERR_UNSUPPORTED          # paging is for the compact formats
    assert reset(cache(**dict(paged, page_tokens=48))) == ffi.ERR_ARG            # pages are multiples of 64 tokens
    assert reset(cache(**dict(paged, pages_per_seq=3))) == ffi.ERR_ARG           # pages_per_seq * page_tokens == S_max
    assert reset(cache(page_tokens=64)) == ffi.ERR_ARG                           # paging fields without a table
    c = cache()
    assert ffi.lib.vsp_kv_read(C.byref(c), 200, 100, None, None, None) == ffi.ERR_ARG    # past the capacity
    assert ffi.lib.vsp_kv_read(C.byref(c), 0, 10, None, None, None) == ffi.ERR_NULL      # neither output given
    t = ffi.VspTensor()
    t.ndim, t.dtype = 4, ffi.BF16
    for i, n in enumerate((2, 2, 11, 128)):
        t.shape[i] = n
    assert ffi.lib.vsp_kv_read(C.byref(c), 0, 10, C.byref(t), None, None) == ffi.ERR_NUMEL
    assert ffi.lib.vsp_seq_lens_advance(None, None, 1, -1, 8, None) == ffi.ERR_ARG
    assert ffi.lib.vsp_seq_lens_advance(None, None, 1, 0, 8, None) == 0
    assert ffi.lib.vsp_seq_lens_advance(None, None, 1, 4, 8, None) == ffi.ERR_NULL


def _decode_splits(ffi, fmt, B, Hq, Hkv, D, T, max_len, device_lens, paged=False):
    """Splits per row of the plan of vsp_attn_decode_multi: the smallest workspace that is not refused holds that many partials.
    A workspace that is large enough goes on to a pointer check that fails, so nothing is ever launched."""
    c = ffi.VspKVCache()
    c.format, c.B, c.Hkv, c.S_max, c.D, c.len = fmt, B, Hkv, max_len, D, max_len
    c.k = c.v = c.k_scale = c.v_scale = 0x10000
    if paged:
        c.S_max = -(-max_len // 64) * 64
        c.page_table, c.page_tokens, c.pages_per_seq, c.n_pages = 0x50000, 64, c.S_max // 64, B * c.S_max // 64
    q = ffi.VspTensor()
    q.ndim, q.dtype, q.data = 4, ffi.F32 if fmt == ffi.KV_F32 else ffi.BF16, 0x20000
    for i, (n, m) in enumerate(zip((B, Hq, T, D), (Hq * T * D, T * D, D, 1))):
        q.shape[i], q.stride[i] = n, m
    for n in range(1, max_len // 256 + 3):
        rc = ffi.lib.vsp_attn_decode_multi(C.byref(q), C.byref(c), 0x30000 if device_lens else None, max_len, C.byref(q), 0.1, 0x40008,
                                           B * Hq * T * n * (D + 2) * 4, None)
        if rc == ffi.ERR_ALIGN:  # the workspace's address, looked at after its size
            return n
        assert rc == ffi.ERR_WORKSPACE, rc


def _decode_route(ffi, fmt, B, Hq, Hkv, D, T, max_len, device_lens=True, page=0):
    """vsp_attn_decode_plan of a cache that holds the bound and no more."""
    c, p = ffi.VspKVCache(), ffi.VspDecodePlan()
    c.format, c.B, c.Hkv, c.S_max, c.D, c.len = fmt, B, Hkv, -(-max_len // (page or 1)) * (page or 1), D, 0 if device_lens else max_len
    if page:
        c.page_table, c.page_tokens, c.pages_per_seq, c.n_pages = 0x50000, page, c.S_max // page, B * c.S_max // page
    ffi.check(ffi.lib.vsp_attn_decode_plan(C.byref(c), int(device_lens), max_len, Hq, T, C.byref(p)))
    return p


def test_decode_routes(ffi):
    bf16, f32, q8 = ffi.KV_BF16, ffi.KV_F32, ffi.KV_Q8_0
    route = lambda *a, **k: _decode_route(ffi, *a, **k)
    kind = lambda p: "ranges" if p.ranges else "round" if p.round else "splits"
    p = route(bf16, 32, 32, 8, 128, 1, 32768)
    assert kind(p) == "ranges" and p.workgroups == p.ranges == 512 and not p.one_launch
    p = route(bf16, 8, 32, 8, 128, 4, 8000, page=256)
    assert kind(p) == "round" and p.round == 32 and not p.or_two and p.one_launch
    p = route(q8, 16, 64, 8, 128, 1, 65536)
    assert kind(p) == "round" and p.or_two
    p = route(f32, 1, 32, 8, 128, 1, 2048, device_lens=False)
    assert kind(p) == "splits" and p.one_launch and p.workgroups == 8 * p.max_splits
    assert kind(route(bf16, 32, 32, 8, 128, 1, 100)) == "splits"
    rng = np.random.default_rng(3)
    for _ in range(2000):  # the splits are those that the workspace is asked for
        B, Hkv, n_rep, L = (int(np.exp(rng.uniform(0, np.log(top)))) for top in (64, 32, 8, 60000))
        fmt, D, T, dev = int(rng.choice([bf16, f32, q8])), int(rng.choice([64, 128])), int(rng.choice([1, 2])), bool(rng.integers(2))
        p = route(fmt, B, Hkv * n_rep, Hkv, D, T, L, device_lens=dev)
        if B * Hkv * L < 200000:  # a round may have more where the workspace has room for them
            least = _decode_splits(ffi, fmt, B, Hkv * n_rep, Hkv, D, T, L, dev)
            assert least <= p.max_splits <= -(-L // 256) if p.round else p.max_splits == least
        assert not (p.ranges and p.round) and (dev or kind(p) == "splits") and p.workgroups <= B * Hkv * max(p.max_splits, -(-L // 256))
    # one long row among short ones makes all of a round's splits: merged by one workgroup only up to so many of so many columns
    assert kind(route(bf16, 14, 32, 8, 64, 2, 8964)) == "ranges" and kind(route(bf16, 21, 32, 8, 64, 4, 8739)) == "ranges"  # two rounds with a merge of their own
    p = route(f32, 8, 8, 4, 128, 4, 24000)  # and is cut into all of them
    assert kind(p) == "round" and not p.one_launch and p.max_splits >= p.round == 64
    for L, one in ((50000, False), (24000, False), (16000, True)):
        p = route(q8, 16, 16, 4, 128, 4, L)
        assert kind(p) == "round" and p.one_launch == one and (p.max_splits <= 16) == one
    p = route(f32, 11, 8, 2, 128, 1, 74964)
    assert kind(p) == "round" and p.one_launch and p.max_splits >= p.round == 128
    # a small batch of many rows keeps the plan's splits: the search for two lengths costs what it saves
    assert kind(route(f32, 19, 32, 8, 128, 1, 621)) == "splits" and kind(route(q8, 14, 32, 8, 128, 1, 4378)) == "round"
    counted = 0
    for _ in range(4000):
        B, Hkv, n_rep, L = (int(np.exp(rng.uniform(0, np.log(top)))) for top in (64, 33, 9, 100000))
        fmt, D, T, page = int(rng.choice([bf16, f32, q8])), int(rng.choice([64, 128])), int(rng.choice([1, 2])), int(rng.choice([0, 64]))
        p = route(fmt, B, Hkv * n_rep, Hkv, D, T, L, page=0 if fmt == f32 else page)
        if p.round and p.one_launch and p.max_splits > 16:
            counted += 1
            assert min(p.max_splits, max(p.uniform_splits, p.round << p.or_two)) * n_rep * T <= (512 if n_rep * T <= 4 else 256)
    assert counted > 40
    c = ffi.VspKVCache()
    c.format, c.B, c.Hkv, c.S_max, c.D, c.len = bf16, 2, 2, 256, 128, 0
    plan = lambda c, *a: ffi.lib.vsp_attn_decode_plan(C.byref(c), *a, C.byref(p))
    assert ffi.lib.vsp_attn_decode_plan(C.byref(c), 1, 0, 4, 1, None) == ffi.ERR_NULL
    assert plan(c, 1, 257, 4, 1) == ffi.ERR_ARG and plan(c, 1, 0, 3, 1) == ffi.ERR_SHAPE and plan(c, 1, 0, 4, 9) == ffi.ERR_UNSUPPORTED
    assert plan(c, 1, 0, 4, 1) == ffi.OK and plan(c, 0, 0, 4, 1) == ffi.OK


def test_ragged_decode_cases_take_the_kernels_they_are_about(ffi):
    # the GPU tests' lists, by the library's plan: every row on its path, and a row for every instance of the kernels
    import test_gpu_decode_ranges as R
    fmts = {"bf16": ffi.KV_BF16, "f32": ffi.KV_F32, "q8_0": ffi.KV_Q8_0}
    seen, odd, even = set(), set(), set()
    for want, rows in (("ranges", R.RANGES), ("round", R.ROUND), ("splits", R.SPLITS)):
        for fmt, Hq, Hkv, D, T, page, lens, bound in rows:
            p = _decode_route(ffi, fmts[fmt], len(lens), Hq, Hkv, D, T, bound, page=page)
            assert want == ("ranges" if p.ranges else "round" if p.round else "splits"), (fmt, Hq, Hkv, D, T, page, len(lens), bound)
            seen.add((want, fmt, D, Hq // Hkv * T <= 4 if fmt == "f32" else page > 0))
            if want == "round" and T == 1 and p.max_splits > 1:
                odd.add(("f32" if fmt == "f32" else "bf16", 8 if p.max_splits <= 8 else 16 if p.max_splits <= 16 else 32))
            if want == "ranges" and p.uniform_splits and sum(lens) * 10 >= max(lens) * len(lens) * 9.1:
                even.add((fmt, p.uniform_splits > 1))
    assert {x for x in seen if x[0] == "round"} == {("round", f, D, b) for f in fmts for D in (64, 128) for b in (False, True)}
    assert {x for x in seen if x[0] == "ranges"} == {("ranges", f, D, b) for f in ("bf16", "f32") for D in (64, 128) for b in (False, True)} - {("ranges", "bf16", 128, True)}
    assert odd == {(t, n) for t in ("f32", "bf16") for n in (8, 16, 32)}
    assert even >= {("bf16", True), ("f32", True)}
    # up to eleven splits of up to eight columns, more than half a workgroup per CU: one launch; twelve, or nine columns: two
    for fmt in fmts.values():
        counted = lambda L, Hq=16: _decode_route(ffi, fmt, 7, Hq, 2, 128, 1, L)
        assert [(counted(L).max_splits, counted(L).one_launch) for L in (2560, 2816, 2817)] == [(10, 1), (11, 1), (12, 0)]
        assert 128 < counted(2560).workgroups and not counted(2816, 18).one_launch and not counted(2816).round


def test_decode_plan_of_several_tokens_per_sequence(ffi):
    # 256 CUs (the value without a GPU).  The bound on the partials belongs to vsp_attn_decode_noalloc, which takes one token:
    # four tokens get the 2048-key splits that measured fastest over long ragged batches and over batches that make one round of them
    bf16, f32, q8 = ffi.KV_BF16, ffi.KV_F32, ffi.KV_Q8_0
    splits = lambda fmt, B, Hq, Hkv, T, L, paged=False: _decode_splits(ffi, fmt, B, Hq, Hkv, 128, T, L, True, paged)
    assert splits(bf16, 32, 32, 8, 4, 32768) == 16 and splits(bf16, 32, 32, 8, 2, 32768) == 16
    assert splits(bf16, 10, 32, 8, 4, 6525) == 4 and splits(f32, 10, 32, 8, 4, 6525) == 4 and splits(bf16, 10, 32, 8, 4, 6525, True) == 4
    assert splits(bf16, 8, 32, 8, 4, 6525) == 13 and splits(bf16, 8, 32, 8, 4, 6525, True) == 13
    assert splits(bf16, 3, 32, 8, 4, 19674) == 10 and splits(bf16, 3, 32, 8, 4, 19674, True) == 20
    assert splits(bf16, 8, 32, 8, 4, 19674) == 10 and splits(f32, 24, 32, 8, 4, 30000) == 15
    assert splits(bf16, 14, 32, 8, 4, 7621) == 15 and splits(bf16, 6, 32, 8, 4, 6525) == 7
    assert splits(f32, 32, 32, 8, 4, 16384) == 32
    # one token: as before
    assert splits(bf16, 32, 32, 8, 1, 32768) == 32 and splits(bf16, 8, 32, 8, 1, 6525) == 7
    assert splits(q8, 32, 32, 8, 4, 32768) == 8


def test_decode_plan_of_a_small_ragged_batch(ffi):
    # splits are halved for want of items only where the halves still make about one round (two thirds of the bound's items, 256 CUs):
    # 1024 keys here, where 512 would make a round and a few items more
    splits = lambda fmt, B, Hq, Hkv, L, paged=False: _decode_splits(ffi, fmt, B, Hq, Hkv, 128, 1, L, True, paged)
    for fmt in (ffi.KV_BF16, ffi.KV_Q8_0):
        assert splits(fmt, 4, 32, 8, 6525) == 8 and splits(fmt, 6, 16, 4, 9739) == 10
    assert splits(ffi.KV_Q8_0, 4, 32, 8, 6525, True) == 13  # Q8_0 pages: shorter items
    assert splits(ffi.KV_BF16, 5, 16, 4, 9680) == 19 and splits(ffi.KV_BF16, 8, 32, 8, 2509) == 5  # still halved
    assert splits(ffi.KV_BF16, 1, 32, 8, 7543) == 30


def test_every_planned_shape_has_a_kernel(ffi):
    # 128-row workgroups, 64-row ones with two key groups, and in the forward 32-row ones with four (split operands: at head_dim 64); the pipelined kernel at
    # head_dim 128 with 128 rows.  Anything else is an error at the launch, and here
    rng = np.random.default_rng(2)
    p, c, lib = ffi.VspAttnPlan(), ffi.VspKVCache(), ffi.lib
    seen = set()
    for _ in range(4000):
        B, Hkv, n_rep, T, past = (int(np.exp(rng.uniform(0, np.log(top)))) for top in (16, 32, 16, 16384, 65536))
        D, flag, Hq = int(rng.choice([64, 128])), int(rng.integers(2)), Hkv * n_rep
        c.format, c.B, c.Hkv, c.S_max, c.len, c.D = int(rng.choice([ffi.KV_BF16, ffi.KV_Q8_0])), B, Hkv, T + past, T + past, D
        for what, call in (("forward", lambda: lib.vsp_attn_prefill_plan(B, Hq, Hkv, T, T + flag * past, D, flag, 0, C.byref(p))),
                           ("cached", lambda: lib.vsp_attn_prefill_cached_plan(C.byref(c), flag, 0, Hq, T, 0, C.byref(p))),
                           ("prompt", lambda: lib.vsp_attn_prefill_cached_plan(C.byref(c), 0, 0, Hq, T, 1, C.byref(p))),
                           ("split", lambda: lib.vsp_attn_prefill_plan(B, Hq, Hkv, T, T, D, flag, 1, C.byref(p))),
                           ("backward", lambda: lib.vsp_attn_backward_plan(B, Hq, Hkv, T, D, flag, 0, C.byref(p))),
                           ("split backward", lambda: lib.vsp_attn_backward_plan(B, Hq, Hkv, T, D, flag, 1, C.byref(p)))):
            assert call() == ffi.OK and p.row_groups * p.key_groups == 4 and p.shares >= 1, what
            seen.add((what, D, p.row_groups, p.pipelined))
    both = lambda what, rows, pipe=0: {(what, D, r, pipe) for D in (64, 128) for r in rows}
    assert seen == (both("forward", (1, 2, 4)) | both("cached", (1, 2, 4)) | both("prompt", (1, 2, 4)) | both("split", (2, 4)) | {("split", 64, 1, 0)} |
                    both("backward", (2, 4)) | both("split backward", (2, 4)) | {(what, 128, 4, 1) for what in ("forward", "cached", "prompt")})


def test_more_rows_than_a_workgroup_numbers(ffi):
    # 2^30 rows of all heads of a kv head and more: rows of one head each, as many as there may be (refused once); the backward's rows as they are
    p = ffi.VspAttnPlan()
    plan = lambda T, n_rep, D=64: ffi.lib.vsp_attn_prefill_plan(1, n_rep, 1, T, 200, D, 0, 0, C.byref(p)) or p.packed
    for D in (64, 128):
        assert plan(1 << 25, 31, D) == 1 and plan(1 << 25, 33, D) == 0 and plan(1 << 26, 64, D) == 0 and plan((1 << 30) - 1, 2, D) == 0
    assert ffi.lib.vsp_attn_prefill_plan(1, 1, 1, 1 << 30, 200, 64, 0, 0, C.byref(p)) == ffi.ERR_ARG
    back = lambda B, Hq, Hkv, N: ffi.lib.vsp_attn_backward_plan(B, Hq, Hkv, N, 64, 1, 0, C.byref(p))
    assert back(1, 64, 1, 1 << 24) == ffi.OK and back(1, 64, 1, (1 << 25) - 2) == ffi.OK and back(63, 32, 32, 1 << 20) == ffi.OK
    assert back(1, 64, 1, 1 << 25) == ffi.ERR_ARG and back(64, 32, 32, 1 << 20) == ffi.ERR_ARG


def test_room_for_shares_of_512_keys(ffi):
    # the size that the C++ adapter passes: room for the plan's shares wherever these hold 512 keys (8 x 64 / 8 heads, 16 tokens of 32768, was given none: it
    # was taken for 512 workgroups, one a head, and is 64 with rows of all heads of a kv head), and never less than it was
    rng, p, more = np.random.default_rng(2), ffi.VspAttnPlan(), 0
    for B, Hkv, n_rep, T, L in [(8, 8, 8, 16, 32768)] + [tuple(int(np.exp(rng.uniform(np.log(lo), np.log(hi)))) for lo, hi in ((1, 16), (1, 16), (1, 16), (2, 1024), (1024, 65536)))
                                                        for _ in range(3000)]:
        c = ffi.VspKVCache()
        c.format, c.B, c.Hkv, c.S_max, c.D, c.len = ffi.KV_BF16, B, Hkv, max(T, L), 128, max(T, L)
        share, tiles, heads = B * Hkv * n_rep * T * 130 * 4, -(-c.len // 32), B * Hkv * n_rep * -(-T // 128)
        n = ffi.lib.vsp_attn_prefill_cached_split_workspace_bytes(C.byref(c), 0, 0, Hkv * n_rep, T) // share
        ffi.check(ffi.lib.vsp_attn_prefill_cached_plan(C.byref(c), 0, 0, Hkv * n_rep, T, 0, C.byref(p)))
        assert (n if n > 1 else 1) >= (p.shares if p.shares <= tiles // 16 else 1), (B, Hkv, n_rep, T, L)
        was = min(-(-512 // heads), tiles // 16, 64) if heads <= 256 else 1
        was = -(-tiles // -(-tiles // was)) if was > 1 else 0
        assert n >= was, (B, Hkv, n_rep, T, L)
        more += n > was
    assert more > 100


def test_partials_of_a_context_in_shares_are_bounded(ffi):
    # the Python view keeps their block for the stream: no shape may ask for gigabytes
    rng = np.random.default_rng(1)
    most = 0
    for _ in range(20000):
        B, Hkv, n_rep, T, past = (int(np.exp(rng.uniform(0, np.log(top)))) for top in (64, 64, 64, 16384, 1000000))
        c = ffi.VspKVCache()
        c.format, c.B, c.Hkv, c.S_max, c.D = ffi.KV_BF16, B, Hkv, T + past, int(rng.choice([64, 128]))
        c.len = c.S_max
        most = max(most, ffi.lib.vsp_attn_prefill_cached_best_workspace_bytes(C.byref(c), 0, 0, Hkv * n_rep, T))
    assert 50e6 < most <= 140e6 + 256


def test_adapter_host_side_checks():
    exe = os.path.join(ROOT, "tests", "cpp", "adapter_test")
    if not os.path.exists(exe):
        pytest.skip("tests/cpp/adapter_test not built (python -c 'import __graft_entry__ as g; g.build()')")
    r = subprocess.run([exe, "--cpu-only"], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr


def test_decode_plan_of_long_even_rows(ffi):
    # one round of a workgroup per CU (16 x 8 rows in halves) up to 24576 keys a part of narrow keys, whole rounds of two beyond
    splits = lambda L, fmt=ffi.KV_Q8_0: _decode_splits(ffi, fmt, 16, 64, 8, 128, 1, L, False)
    assert [splits(L) for L in (8192, 36000, 49152, 49153, 65536)] == [2, 2, 2, 4, 4]
    assert splits(65536, ffi.KV_BF16) == 2


def test_whole_numbers_are_taken_as_int_takes_them():
    import torch
    from vesper_amd import _host
    q = torch.zeros(1, 1, 1, 64)  # on the CPU: refused, but only after the arguments have been read
    decode = lambda max_len: _host.decode(0, q, None, max_len, 1.0, None, None, 0)
    for bad, error in ((float("nan"), ValueError), (float("inf"), OverflowError), (None, TypeError), (1 << 70, OverflowError)):
        with pytest.raises(error):
            decode(bad)
    for good in (7, 7.9, np.int32(7), torch.tensor(7)):
        with pytest.raises(RuntimeError, match="expected a tensor on the GPU"):
            decode(good)


def test_build_takes_python_and_torch_from_the_interpreter_that_runs_it(monkeypatch):
    import __graft_entry__ as entry
    calls = []
    monkeypatch.setattr(entry.subprocess, "check_call", lambda cmd, **kw: calls.append(cmd))
    monkeypatch.setattr(entry.sys, "executable", "/some/python")
    entry.build()
    made = [c for c in calls if c[0] == "make" and "all" in c]
    assert made and all("PYTHON=/some/python" in c for c in made)


def test_product_never_touches_the_oracle():
    # the shipped package must not import, load or link anything under oracle/
    for dirpath, _, files in os.walk(os.path.join(ROOT, "vesper_amd")):
        if "build" in dirpath:
            continue
        for f in files:
            if f.endswith((".py", ".hip", ".cpp", ".hpp", ".h")) or f == "Makefile":
                src = open(os.path.join(dirpath, f), errors="ignore").read()
                assert "oracle" not in src.lower(), os.path.join(dirpath, f)
