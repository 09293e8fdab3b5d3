"""Attention on the matrix cores (attention_mfma.hip; all of it from 16 query
rows, the scores below)
against the C restatement of the reference's attendRow, bit for bit: query
heads per kv head that do and do not divide the row tiles, both sum tiles
(4 and 16 rows a wave), ragged last tiles, sequences that start inside a value
block, rows that see no key, a row clipped to max_keys, and infinities and NaN
in every cache entry that no row of the call may use. The addresses are
checked on the CPU over adversarial ranges in test_attention_bounds.py."""
import numpy as np
import pytest


def _call(gpu, q, kc, vc, kend, kstart, maxk, shift=0):
    """shift: floats from a 16-byte boundary to q."""
    import hiprt as rt

    T, H, D = q.shape
    Hkv, C, _ = kc.shape
    bufs = [rt.DeviceBuffer.from_array(np.ascontiguousarray(a))
            for a in (np.concatenate([np.zeros(shift, np.float32), q.ravel()]), kc, gpu.pack_vcache(vc), kend,
                      kstart if kstart is not None else kend)]
    out = rt.DeviceBuffer.from_array(np.full(q.shape, 7, np.float32))
    wsb = gpu.attention_workspace_bytes(T, H, maxk)
    ws, s = rt.DeviceBuffer(wsb), rt.Stream()
    gpu.attention_dev(bufs[0].ptr + 4 * shift, bufs[1].ptr, bufs[2].ptr, bufs[3].ptr, bufs[4].ptr if kstart is not None else None,
                      T, H, Hkv, D, C, maxk, kc.dtype == np.float16, out.ptr, ws.ptr, wsb, s.handle)
    s.sync()
    return out.download(np.float32).reshape(q.shape)


@pytest.mark.gpu
@pytest.mark.parametrize("f16", [False, True], ids=["f32cache", "f16cache"])
@pytest.mark.parametrize("T,H,Hkv,D,slots,C", [(16, 4, 4, 64, 1, 40), (17, 6, 2, 128, 1, 130), (33, 8, 1, 64, 1, 300),
                                               (40, 12, 4, 128, 3, 77), (257, 32, 8, 128, 1, 261),
                                               (65, 64, 64, 64, 2, 129), (300, 10, 10, 128, 5, 90),
                                               (23, 14, 2, 64, 2, 1030), (257, 32, 8, 64, 1, 300),
                                               (16, 4, 4, 64, 1, 270), (17, 6, 2, 128, 1, 300),
                                               (300, 32, 8, 128, 7, 61), (300, 32, 8, 64, 150, 13),
                                               (21, 6, 3, 192, 2, 90), (40, 4, 1, 256, 3, 77)])
def test_rows_and_tiles(gpu, oracle, f16, T, H, Hkv, D, slots, C):
    rng = np.random.default_rng(T * 10 + H + C)
    L = slots * C
    kc = rng.standard_normal((Hkv, L, D)).astype(np.float16 if f16 else np.float32)
    vc = rng.standard_normal((Hkv, L, D)).astype(kc.dtype)
    q = rng.standard_normal((T, H, D)).astype(np.float32)
    slot = np.arange(T) % slots if T < 100 else np.arange(T) * slots // T
    start = (slot * C).astype(np.int64)
    pos = (C - T + np.arange(T)) if slots == 1 and C > T else rng.integers(0, C - 1, T)
    pos[0], pos[T // 2] = 0, C - 2 if C - 2 >= 0 else 0
    end = start + pos
    used = np.zeros(L, bool)
    for t in range(T):
        used[start[t]:end[t] + 1] = True
    kc[:, ~used], vc[:, ~used] = np.nan, np.inf
    empty = T // 3
    want = oracle.attention(q, kc, vc, end, start, threads=8)
    gend = end.copy()
    gend[empty] = start[empty] - 1  # sees no key: zeros
    want[empty] = 0
    if slots == 1:
        got = _call(gpu, q, kc, vc, gend, None, C)
    else:
        got = _call(gpu, q, kc, vc, gend, start, C)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), np.argwhere(got != want)[:5]


@pytest.mark.gpu
@pytest.mark.parametrize("f16", [False, True], ids=["f32cache", "f16cache"])
@pytest.mark.parametrize("T,H,Hkv,D,C", [(4, 16, 8, 64, 520), (3, 24, 8, 128, 705), (9, 10, 2, 64, 961),
                                         (8, 64, 8, 128, 321), (2, 14, 2, 128, 4100), (1, 32, 8, 64, 2049)])
def test_decode_scores(gpu, oracle, f16, T, H, Hkv, D, C):
    """Decode batches, a sequence a row: 2 to 8 query heads a kv head, every
    count of keys mod 4, the last tile of one key and full."""
    rng = np.random.default_rng(T * 10 + H + C)
    kc = rng.standard_normal((Hkv, T * C, D)).astype(np.float16 if f16 else np.float32)
    vc = rng.standard_normal((Hkv, T * C, D)).astype(kc.dtype)
    q = rng.standard_normal((T, H, D)).astype(np.float32)
    start = (np.arange(T) * C).astype(np.int64)
    end = start + C - 1 - np.array([t if t < 6 else 64 * t for t in range(T)])
    for t in range(T):
        kc[:, end[t] + 1:(t + 1) * C], vc[:, end[t] + 1:(t + 1) * C] = np.nan, np.inf
    got = _call(gpu, q, kc, vc, end, start, C)
    want = oracle.attention(q, kc, vc, end, start, threads=8)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), np.argwhere(got != want)[:5]


@pytest.mark.gpu
@pytest.mark.parametrize("f16", [False, True], ids=["f32cache", "f16cache"])
@pytest.mark.parametrize("T,H,Hkv,D,C", [(3, 16, 8, 64, 705), (5, 8, 4, 128, 1290), (2, 32, 8, 128, 1023), (9, 64, 32, 128, 257),
                                         (15, 4, 2, 64, 519)])
def test_decode_scores_pairs(gpu, oracle, f16, T, H, Hkv, D, C):
    """Two query heads a kv head, and four at D = 128: the vector kernel and
    the matrix cores on either side of the line by cache type."""
    test_decode_scores(gpu, oracle, f16, T, H, Hkv, D, C)


@pytest.mark.gpu
@pytest.mark.parametrize("f16", [False, True], ids=["f32cache", "f16cache"])
@pytest.mark.parametrize("T,H,Hkv,D,slots,L", [(16, 4, 4, 64, 16, 261), (33, 6, 2, 128, 40, 83), (64, 8, 8, 128, 64, 29),
                                               (40, 8, 2, 64, 40, 300), (50, 4, 2, 128, 25, 131), (90, 3, 3, 64, 23, 71),
                                               (19, 1, 1, 128, 5, 700), (140, 2, 2, 128, 140, 7)])
def test_few_rows_a_sequence(gpu, oracle, f16, T, H, Hkv, D, slots, L):
    """Up to four (query, head) rows a sequence on average: 1 to 4 query heads a
    kv head, sequences that start inside value blocks, several queries of one
    sequence, waves of 32 keys that several sequences share, rows without a key."""
    rng = np.random.default_rng(T + D)
    kc = rng.standard_normal((Hkv, slots * L, D)).astype(np.float16 if f16 else np.float32)
    vc = rng.standard_normal((Hkv, slots * L, D)).astype(kc.dtype)
    q = rng.standard_normal((T, H, D)).astype(np.float32)
    start = (np.arange(T) * slots // T * L).astype(np.int64)
    end = start + rng.integers(0, L - 1, T)  # every sequence's last entry unused
    end[0], end[T - 1] = start[0], start[T - 1] + L - 2
    used = np.zeros(slots * L, bool)
    for t in range(T):
        used[start[t]:end[t] + 1] = True
    kc[:, ~used], vc[:, ~used] = np.nan, np.inf
    want = oracle.attention(q, kc, vc, end, start, threads=8)
    end[T // 3] = start[T // 3] - 1
    want[T // 3] = 0
    got = _call(gpu, q, kc, vc, end, start, L)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), np.argwhere(got != want)[:5]


@pytest.mark.gpu
@pytest.mark.parametrize("T,slots,L,D", [(40, 40, 64, 128), (9 * 4, 36, 50, 64)])
def test_prompt_among_many_sequences(gpu, oracle, T, slots, L, D):
    """One sequence's rows in a cache of as many sequences as there are rows:
    waves of both kinds (few and many rows) in one call."""
    H, Hkv = 16, 16
    rng = np.random.default_rng(T)
    kc, vc = (rng.standard_normal((Hkv, slots * L, D)).astype(np.float16) for _ in range(2))
    q = rng.standard_normal((T, H, D)).astype(np.float32)
    start = np.full(T, 3 * L, np.int64)
    start[::9] = 5 * L + 1
    end = start + np.minimum(np.arange(T), L - 2)
    got = _call(gpu, q, kc, vc, end, start, L)
    want = oracle.attention(q, kc, vc, end, start, threads=8)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), np.argwhere(got != want)[:5]


@pytest.mark.gpu
@pytest.mark.parametrize("T,D,f16", [(20, 128, True), (17, 64, False)])
def test_unaligned_q(gpu, oracle, T, D, f16):
    """q four bytes past a 16-byte boundary: the vector kernels, same bits."""
    H, Hkv, C = 8, 4, 150
    rng = np.random.default_rng(T)
    kc, vc = (rng.standard_normal((Hkv, C, D)).astype(np.float16 if f16 else np.float32) for _ in range(2))
    q = rng.standard_normal((T, H, D)).astype(np.float32)
    end = (np.arange(T) * 5 + 3).astype(np.int64)
    got = _call(gpu, q, kc, vc, end, None, C, shift=1)
    want = oracle.attention(q, kc, vc, end, None, threads=8)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), np.argwhere(got != want)[:5]


@pytest.mark.gpu
@pytest.mark.parametrize("T,maxk", [(20, 50), (300, 257)])
def test_max_keys_and_nonfinite(gpu, oracle, T, maxk):
    """Rows past max_keys see their first max_keys keys; a NaN key gives NaN
    rows, an infinite value infinite (or NaN) dims, as the reference's."""
    H, Hkv, D, C = 32, 8, 128, 400
    rng = np.random.default_rng(T)
    kc, vc = (rng.standard_normal((Hkv, C, D)).astype(np.float16) for _ in range(2))
    kc[1, 30, 5], vc[2, 7, 9], vc[3, 8, 11] = np.nan, np.inf, np.nan
    q = rng.standard_normal((T, H, D)).astype(np.float32)
    end = (np.arange(T) + 10).astype(np.int64)
    got = _call(gpu, q, kc, vc, end, None, maxk)
    want = oracle.attention(q, kc, vc, np.minimum(end, maxk - 1), None, threads=8)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    fin = ~np.isnan(want)
    assert np.array_equal(got[fin].view(np.uint32), want[fin].view(np.uint32))


@pytest.mark.gpu
@pytest.mark.parametrize("T,H,Hkv,D", [(40, 16, 4, 64), (257, 32, 8, 128)], ids=["4x4x1", "16x16x1"])
@pytest.mark.parametrize("exponents", [(0, 2), (0, 255)], ids=["subnormal", "all"])
def test_value_classes(gpu, oracle, T, H, Hkv, D, exponents):
    """The weighted sum's chains on both instructions: values of every finite
    class (products of a weight in [0, 1] and sums that are subnormal, that
    overflow), bit for bit the fmas of the oracle; NaN where it has one."""
    C = T
    rng = np.random.default_rng(T + exponents[1])
    kc = rng.standard_normal((Hkv, C, D)).astype(np.float32)
    bits = rng.integers(0, 1 << 23, kc.shape, dtype=np.uint32) | rng.integers(*exponents, kc.shape, dtype=np.uint32) << 23
    vc = (bits | rng.integers(0, 2, kc.shape, dtype=np.uint32) << 31).view(np.float32)
    q = (3 * rng.standard_normal((T, H, D))).astype(np.float32)
    end = np.arange(T, dtype=np.int64)
    got = _call(gpu, q, kc, vc, end, None, C)
    want = oracle.attention(q, kc, vc, end, None, threads=8)
    if exponents[1] == 2:  # values below 2^-125, averaged with random signs: 76 and 88 % of the outputs are subnormal
        assert np.count_nonzero((np.abs(want) < np.finfo(np.float32).tiny) & (want != 0)) > want.size // 2
    same = (got.view(np.uint32) == want.view(np.uint32)) | (np.isnan(got) & np.isnan(want))
    assert same.all(), f"{(~same).sum()} of {same.size} differ, first at {np.argwhere(~same)[0]}"


@pytest.mark.gpu
@pytest.mark.parametrize("f16", [False, True], ids=["f32cache", "f16cache"])
@pytest.mark.parametrize("T,H,Hkv,D,slots,C", [(16, 1, 1, 64, 1, 16), (64, 2, 1, 128, 1, 64), (128, 4, 2, 64, 1, 64),
                                               (256, 1, 1, 64, 1, 256), (128, 1, 1, 128, 1, 255), (129, 2, 2, 64, 1, 256),
                                               (128, 2, 2, 128, 1, 65), (32, 4, 4, 128, 8, 31), (257, 1, 1, 128, 3, 90)])
def test_small_grids(gpu, oracle, f16, T, H, Hkv, D, slots, C):
    """16 queries and more in one launch (att_decode_kernel): on the line of 512
    workgroups at 256 keys and of 1024 at 64, and past each."""
    rng = np.random.default_rng(T + H + C)
    L = slots * C
    kc = rng.standard_normal((Hkv, L, D)).astype(np.float16 if f16 else np.float32)
    vc = rng.standard_normal((Hkv, L, D)).astype(kc.dtype)
    q = rng.standard_normal((T, H, D)).astype(np.float32)
    start = (np.arange(T) % slots * C).astype(np.int64)
    end = start + np.minimum(np.arange(T), C - 2)
    for s in range(slots):
        kc[:, s * C + C - 1], vc[:, s * C + C - 1] = np.nan, np.inf  # seen by no query
    end[T // 2] = start[T // 2] - 1
    want = oracle.attention(q, kc, vc, np.maximum(end, start), start, threads=8)
    want[T // 2] = 0
    got = _call(gpu, q, kc, vc, end, start if slots > 1 else None, C)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), np.argwhere(got != want)[:5]
