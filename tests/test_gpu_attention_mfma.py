"""Attention on the matrix cores (attention_mfma.hip; all of it from 16 query
rows, the scores below)
against the C restatement of the reference's attendRow, bit for bit: query
heads per kv head that do and do not divide the row tiles, both sum tiles
(4 and 16 rows a wave), ragged last tiles, sequences that start inside a value
block, rows that see no key, a row clipped to max_keys, and infinities and NaN
in every cache entry that no row of the call may use. The addresses are
checked on the CPU over adversarial ranges."""
import numpy as np
import pytest


def _call(gpu, q, kc, vc, kend, kstart, maxk):
    import hiprt as rt

    T, H, D = q.shape
    Hkv, C, _ = kc.shape
    bufs = [rt.DeviceBuffer.from_array(np.ascontiguousarray(a))
            for a in (q, kc, gpu.pack_vcache(vc), kend, kstart if kstart is not None else kend)]
    out = rt.DeviceBuffer.from_array(np.full(q.shape, 7, np.float32))
    wsb = gpu.attention_workspace_bytes(T, H, maxk)
    ws, s = rt.DeviceBuffer(wsb), rt.Stream()
    gpu.attention_dev(bufs[0].ptr, bufs[1].ptr, bufs[2].ptr, bufs[3].ptr, bufs[4].ptr if kstart is not None else None,
                      T, H, Hkv, D, C, maxk, kc.dtype == np.float16, out.ptr, ws.ptr, wsb, s.handle)
    s.sync()
    return out.download(np.float32).reshape(q.shape)


@pytest.mark.gpu
@pytest.mark.parametrize("f16", [False, True], ids=["f32cache", "f16cache"])
@pytest.mark.parametrize("T,H,Hkv,D,slots,C", [(16, 4, 4, 64, 1, 40), (17, 6, 2, 128, 1, 130), (33, 8, 1, 64, 1, 300),
                                               (40, 12, 4, 128, 3, 77), (257, 32, 8, 128, 1, 261),
                                               (65, 64, 64, 64, 2, 129), (300, 10, 10, 128, 5, 90),
                                               (23, 14, 2, 64, 2, 1030)])
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


def _ranges(T, C, maxk, slots, rng):
    start = rng.integers(0, slots, T) * (C // slots)
    end = start + rng.integers(-1, max(C // slots, 1), T)
    for t, (e, s) in enumerate([(-5, -1), (C + 9, C + 3), (C - 1, C - 1), (C * 2, -7), (maxk + 50, 0)]):
        end[t], start[t] = e, s
    k0 = np.clip(start, 0, C - 1)
    return k0, np.clip(np.minimum(np.minimum(end + 1 - k0, C - k0), maxk), 0, None)


@pytest.mark.parametrize("D,f16", [(64, True), (64, False), (128, True), (128, False)])
@pytest.mark.parametrize("T,H,Hkv,C,maxk,slots", [(16, 4, 4, 7, 8192, 1), (37, 6, 2, 301, 100, 3), (65, 8, 1, 8200, 8192, 2),
                                                  (257, 8, 8, 130, 130, 4)])
def test_addresses_in_bounds(D, f16, T, H, Hkv, C, maxk, slots):
    G, rows = H // Hkv, T * (H // Hkv)
    k0, n = _ranges(T, C, maxk, slots, np.random.default_rng(T + C))
    head = lambda hk, rho: min(rho, rows - 1) // G * H + hk * G + min(rho, rows - 1) % G
    vblocks = (C + 7) // 8
    for hk in {0, Hkv - 1}:
        # scores_kernel: 32 rows, tiles of 128 keys, keys clamped to the cache
        for rho0 in range(0, rows, 32):
            ts = [r // G for r in range(rho0, min(rho0 + 32, rows)) if n[r // G] > 0]
            if ts:
                kfin = max(k0[t] + n[t] for t in ts)
                assert min(kfin - 1 + 127, C - 1) < C and min(k0[t] for t in ts) >= 0
                assert all(n[t] <= maxk and t * H + hk * G + G - 1 < T * H for t in ts)
        # wsum_kernel: R rows, one first key at a time
        wide = (rows + 31) // 32 * Hkv >= 256
        R, KC = (32, 64) if wide else (8, D)
        for rho0 in range(0, rows, R):
            tile = [(k0[r // G], n[r // G]) for r in range(rho0, min(rho0 + R, rows))]
            assert all(0 <= head(hk, rho0 + i) < T * H for i in range(R))  # a row past the last: the last one's
            for first in {k for k, c in tile if c > 0}:
                nall = max(c for k, c in tile if k == first)
                off, nblk = first % 8, (first % 8 + nall + 7) // 8
                assert first // 8 + nblk - 1 < vblocks  # value blocks, clamped to the last
                assert nall - 1 < maxk                  # scores, clamped to the row's last
                assert (off + nall + KC - 1) // KC * KC >= off + nall
