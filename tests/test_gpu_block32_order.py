"""Products with activation blocks of 32 for many rows in the reference's
lane order (gemm_b32_ref.hip) against the C restatement, bit for bit: ragged
row and weight-row counts around the tiles (16, 32 and 64 rows; 16 weight rows
a wave), odd block counts, bias, and refused rows."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

Q8_0, Q4_K, Q6_K = 64, 66, 67


def check(gpu, oracle, dt, n, k, rows, seed, bias=False, edit=None):
    wb = oracle.synthetic_weight(dt, n, k, seed=seed)
    x = oracle.synthetic_acts(rows, k, seed=seed + 1)
    if edit:
        edit(wb, x)
    b = oracle.synthetic_acts(1, n, seed=seed + 2)[0] if bias else None
    W = gpu.Weight(wb, dt, n, k)
    got = gpu.dequant_matmul_a8(W, x, bias=b, block=32)
    W.release()
    want = oracle.linear_a8(x, wb, dt, n, k, bias=b, block=32, threads=8)
    same = (got.view(np.uint32) == want.view(np.uint32)) | (np.isnan(got) & np.isnan(want))
    assert same.all(), f"{(~same).sum()} of {same.size} differ, first at {np.argwhere(~same)[0]}"


@pytest.mark.parametrize("dt,k", [(Q8_0, 32), (Q8_0, 96), (Q8_0, 1056), (Q8_0, 4096)])
@pytest.mark.parametrize("rows,n", [(9, 65), (16, 15), (17, 130), (33, 64), (40, 300)])
def test_rows_and_tiles(gpu, oracle, dt, k, rows, n):
    check(gpu, oracle, dt, n, k, rows, seed=rows + n, bias=rows % 2 == 1)


# grids of at least 256 workgroups with 16, 32 and 64 activation rows a tile
@pytest.mark.parametrize("rows,n", [(16, 16384), (150, 3300), (261, 3300)])
def test_wide_grids(gpu, oracle, rows, n):
    check(gpu, oracle, Q8_0, n, 352, rows, seed=rows, bias=True)


@pytest.mark.parametrize("rows,n", [(20, 80), (150, 3300)])
def test_refusals(gpu, oracle, rows, n):
    def edit(wb, x):
        x[3, 7], x[5, 100], x[9] = np.nan, 2.0**61, 0.0
        w = wb.reshape(n, -1)
        w[4, 0:2] = np.frombuffer(np.float16(np.inf).tobytes(), np.uint8)
        w[70, 34:36] = np.frombuffer(np.float16(np.nan).tobytes(), np.uint8)

    check(gpu, oracle, Q8_0, n, 288, rows, seed=7, bias=True, edit=edit)


@pytest.mark.parametrize("dt,k", [(Q8_0, 32), (Q8_0, 1056), (Q8_0, 2080), (Q4_K, 256), (Q4_K, 2304), (Q6_K, 512),
                                  (Q6_K, 1280)])
@pytest.mark.parametrize("rows,n", [(1, 9), (2, 64), (3, 7), (4, 33), (5, 16), (6, 1), (7, 41), (8, 24)])
def test_gemv(gpu, oracle, dt, k, rows, n):
    """gemv_b32.hip: rows of one and several stages of 1024, ending inside one."""
    check(gpu, oracle, dt, n, k, rows, seed=rows + n, bias=rows % 2 == 0)


@pytest.mark.parametrize("dt", [Q8_0, Q4_K, Q6_K])
@pytest.mark.parametrize("rows", [1, 7])
def test_gemv_refusals(gpu, oracle, dt, rows):
    def edit(wb, x):
        x[rows - 1, 7] = np.inf
        w = wb.reshape(21, -1)
        at = {Q4_K: 2, Q6_K: 208, Q8_0: 34}[dt]
        w[4, at:at + 2] = np.frombuffer(np.float16(np.inf).tobytes(), np.uint8)

    check(gpu, oracle, dt, 21, 1280, rows, seed=11, bias=True, edit=edit)


# gemv_b32.hip's direct form: a group of eight lanes a weight row; on its line
# and a row below it, rows that end inside a workgroup of 32
@pytest.mark.parametrize("dt,n,k", [(Q4_K, 12000, 1024), (Q4_K, 11999, 1024), (Q4_K, 8193, 1536), (Q4_K, 5001, 256),
                                    (Q6_K, 12001, 256), (Q6_K, 32769, 512), (Q8_0, 22001, 2048), (Q8_0, 20505, 96),
                                    (Q8_0, 6143, 512), (Q8_0, 8200, 32)])
@pytest.mark.parametrize("rows", [1, 2, 3, 4, 5, 6, 7, 8])
def test_gemv_direct(gpu, oracle, dt, n, k, rows):
    check(gpu, oracle, dt, n, k, rows, seed=rows + n, bias=rows % 2 == 0)


@pytest.mark.parametrize("dt,n,k,rows", [(Q8_0, 8200, 1056, 7), (Q4_K, 12001, 1280, 3), (Q6_K, 12010, 256, 8)])
def test_direct_refusals(gpu, oracle, dt, n, k, rows):
    def edit(wb, x):
        x[rows - 1, 7] = np.inf
        w = wb.reshape(n, -1)
        at = {Q4_K: 2, Q6_K: 208, Q8_0: 0}[dt]
        w[[4, n - 1], at:at + 2] = np.frombuffer(np.float16(np.inf).tobytes(), np.uint8)

    check(gpu, oracle, dt, n, k, rows, seed=11, bias=True, edit=edit)
