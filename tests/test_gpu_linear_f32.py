"""dequant_matmul.v1 in the reference's float order (linear_f32.hip) against
the C restatement, bit for bit: the GEMV up to 8 rows and the matrix-core
tiles above, at ragged rows and weight rows around their tiles (8 weight rows;
32 x 32 and 32 x 64), one and several stages of K, Q8_0 rows that end inside a
stage, non-finite activations and scales, and the value classes of a chain."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

Q8_0, Q4_K, Q6_K = 64, 66, 67


def check(gpu, oracle, dt, n, k, rows, seed, bias=False, edit=None):
    import hiprt

    wb = oracle.synthetic_weight(dt, n, k, seed=seed)
    x = oracle.synthetic_acts(rows, k, seed=seed + 1)
    if edit:
        edit(wb, x)
    b = oracle.synthetic_acts(1, n, seed=seed + 2)[0] if bias else None
    W = gpu.Weight(wb, dt, n, k)
    # x one float past a 16-byte boundary: the entry point asks no alignment
    xd, yd, s = hiprt.DeviceBuffer((rows * k + 1) * 4), hiprt.DeviceBuffer(rows * n * 4), hiprt.Stream()
    xd.upload(np.concatenate([np.zeros(1, np.float32), x.ravel()]))
    bd = hiprt.DeviceBuffer.from_array(b) if bias else None
    gpu.linear_f32_dev(W, xd.ptr + 4, rows, bd.ptr if bias else None, yd.ptr, s.handle)
    s.sync()
    got = yd.download(np.float32).reshape(rows, n)
    W.release()
    want = oracle.linear_f32(x, wb, dt, n, k, bias=b, threads=8)
    same = (got.view(np.uint32) == want.view(np.uint32)) | (np.isnan(got) & np.isnan(want))
    assert same.all(), f"{(~same).sum()} of {same.size} differ, first at {np.argwhere(~same)[0]}"


@pytest.mark.parametrize("dt,k", [(Q4_K, 256), (Q4_K, 2304), (Q6_K, 512), (Q6_K, 1280), (Q8_0, 32), (Q8_0, 288),
                                  (Q8_0, 1120), (Q8_0, 1024)])
@pytest.mark.parametrize("rows,n", [(1, 9), (2, 8), (5, 70), (8, 31), (9, 33), (32, 64), (33, 1), (64, 97), (131, 40)])
def test_rows_and_tiles(gpu, oracle, dt, k, rows, n):
    check(gpu, oracle, dt, n, k, rows, seed=rows + n, bias=rows % 2 == 1)


# Q8_0 above 8 rows: chunks of the GEMV up to 768 workgroups of eight rows, a
# last chunk of one to eight rows, and the tiles just past them
@pytest.mark.parametrize("k", [32, 288, 1120, 1024])
@pytest.mark.parametrize("rows,n", [(9, 3072), (9, 3080), (17, 2050), (33, 1297), (64, 768), (64, 801), (131, 401),
                                    (10, 1100), (200, 33)])
def test_q8_0_chunks_and_tiles(gpu, oracle, k, rows, n):
    check(gpu, oracle, Q8_0, n, k, rows, seed=rows + n, bias=rows % 2 == 1)


# up to 8 rows in chunks of one, two and four and in one pass
@pytest.mark.parametrize("dt,k", [(Q4_K, 512), (Q6_K, 256), (Q8_0, 96)])
@pytest.mark.parametrize("rows,n", [(2, 1024), (2, 1025), (4, 512), (4, 1030), (6, 600), (8, 250), (8, 300), (8, 1024), (8, 2056),
                                    (7, 290), (7, 300), (8, 4100)])
def test_gemv_chunks(gpu, oracle, dt, k, rows, n):
    check(gpu, oracle, dt, n, k, rows, seed=rows + n, bias=rows % 4 == 0)


@pytest.mark.parametrize("dt", [Q4_K, Q6_K, Q8_0])
@pytest.mark.parametrize("rows", [3, 40])
def test_non_finite(gpu, oracle, dt, rows):
    def edit(wb, x):
        x[0, 5], x[1, 7], x[2, 3] = np.inf, np.nan, -np.inf
        w = wb.reshape(40, -1)
        at = {Q4_K: 0, Q6_K: 208, Q8_0: 0}[dt]
        w[4, at:at + 2] = np.frombuffer(np.float16(np.inf).tobytes(), np.uint8)
        w[9, at:at + 2] = np.frombuffer(np.float16(np.nan).tobytes(), np.uint8)

    check(gpu, oracle, dt, 40, 768, rows, seed=3, edit=edit)


@pytest.mark.parametrize("dt", [Q4_K, Q6_K, Q8_0])
@pytest.mark.parametrize("rows", [3, 40])
def test_subnormal(gpu, oracle, dt, rows):
    """Rows whose products, sums and outputs are all subnormal: subnormal
    activations, and small normal ones."""
    n, k = 40, 768
    wb = oracle.synthetic_weight(dt, n, k, seed=5)
    x = oracle.synthetic_acts(rows, k, seed=6) * np.float32(1e-39)
    x[1::2] *= np.float32(0.01)
    W = gpu.Weight(wb, dt, n, k)
    got = gpu.dequant_matmul(W, x)
    W.release()
    want = oracle.linear_f32(x, wb, dt, n, k, threads=8)
    assert np.all(np.abs(want) < np.finfo(np.float32).tiny) and np.count_nonzero(want) > want.size // 2
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))


def _bits(rng, exponents, shape):
    """Floats of random sign and mantissa, biased exponents from a range."""
    e = rng.integers(*exponents, shape, dtype=np.uint32)
    return (rng.integers(0, 1 << 23, shape, dtype=np.uint32) | e << 23 | rng.integers(0, 2, shape, dtype=np.uint32) << 31).view(np.float32)


@pytest.mark.parametrize("exponents", [(0, 255), (0, 30), (90, 160), (225, 255)], ids=["all", "tiny", "middle", "huge"])
def test_matrix_core_chain_is_fma(gpu, oracle, exponents):
    """A chain on v_mfma_f32_32x32x1 against the same chain on the vector
    unit's fmaf: for Q8_0 weights the rows of one call of 40 (matrix cores)
    have the steps of calls of at most 8 (fmaf). Every value class of the
    activations, f16 scales of every finite class; a row with one NaN keeps
    its sign and payload (several NaNs: which one survives is the adds')."""
    n, k, rows = 1300, 1056, 40
    rng = np.random.default_rng(exponents[0] * 1000 + exponents[1])
    wb = rng.integers(0, 256, (n, k // 32, 34), dtype=np.uint8)
    d = rng.integers(0, 0x7C00, (n, k // 32), dtype=np.uint16) | rng.integers(0, 2, (n, k // 32), dtype=np.uint16) << 15
    wb[:, :, :2] = d.astype("<u2").view(np.uint8).reshape(n, k // 32, 2)
    x = _bits(rng, exponents, (rows, k))
    x[3, 7], x[4, 100] = np.inf, -np.inf
    nans = {5: (1000, 0x7FC12345), 6: (31, 0xFFC00001), 7: (0, 0x7FABCDEF), 39: (1055, 0x7FFFFFFF)}
    for m, (c, u) in nans.items():
        x[m] = _bits(rng, (90, 130), k)  # no other NaN arises in the row
        x.view(np.uint32)[m, c] = u
    W = gpu.Weight(wb.reshape(-1), Q8_0, n, k)
    got = gpu.dequant_matmul(W, x)
    want = np.concatenate([gpu.dequant_matmul(W, np.ascontiguousarray(x[m:m + 8])) for m in range(0, rows, 8)])
    W.release()
    ok = np.isnan(got) & np.isnan(want)
    ok[list(nans)] = False
    same = (got.view(np.uint32) == want.view(np.uint32)) | ok
    assert same.all(), f"{(~same).sum()} of {same.size} differ, first at {np.argwhere(~same)[0]}"
    assert np.isnan(got[list(nans)]).all()
    ref = oracle.linear_f32(x, wb.reshape(-1), Q8_0, n, k, threads=8)
    same = (got.view(np.uint32) == ref.view(np.uint32)) | (np.isnan(got) & np.isnan(ref))
    assert same.all(), f"{(~same).sum()} of {same.size} differ from the oracle"
