"""dequant_matmul.v1 in the reference's float order (linear_f32.hip) against
the C restatement, bit for bit: the GEMV up to 8 rows and the matrix-core
tiles above, at ragged rows and weight rows around their tiles (8 weight rows;
32 x 32 and 32 x 64), one and several stages of K, Q8_0 rows that end inside a
stage, and non-finite activations and scales."""
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


@pytest.mark.parametrize("dt", [Q4_K, Q6_K, Q8_0])
@pytest.mark.parametrize("rows", [3, 40])
def test_non_finite(gpu, oracle, dt, rows):
    def edit(wb, x):
        x[0, 5], x[1, 7], x[2, 3] = np.inf, np.nan, -np.inf
        x[2, 100:140] = 1e-42  # subnormal products
        w = wb.reshape(40, -1)
        at = {Q4_K: 0, Q6_K: 208, Q8_0: 0}[dt]
        w[4, at:at + 2] = np.frombuffer(np.float16(np.inf).tobytes(), np.uint8)
        w[9, at:at + 2] = np.frombuffer(np.float16(np.nan).tobytes(), np.uint8)

    check(gpu, oracle, dt, 40, 768, rows, seed=3, edit=edit)
