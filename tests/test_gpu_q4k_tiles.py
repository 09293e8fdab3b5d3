"""Q4_K prefill tiles (gemm_q4k.hip): 128 weight rows by 32 activation rows
from 96 workgroups of those (129 at a short K and wide grids), by 64 above 256; bit for bit the
oracle, at the edges of both tiles, on both sides of the rules, with bias and
refusals (reference amx_test.go:41-141)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

Q4_K = 66


def check(gpu, oracle, rows, n, k, edit=None, bias=False):
    wb = oracle.synthetic_weight(Q4_K, n, k, seed=rows + n)
    x = oracle.synthetic_acts(rows, k, seed=rows + 1)
    if edit:
        edit(wb, x)
    b = oracle.synthetic_acts(1, n, seed=rows + 2)[0] if bias else None
    W = gpu.Weight(wb, Q4_K, n, k)
    got = gpu.dequant_matmul_a8(W, x, bias=b, block=256)
    W.release()
    want = oracle.linear_a8(x, wb, Q4_K, n, k, bias=b, block=256, threads=8)
    same = (got.view(np.uint32) == want.view(np.uint32)) | (np.isnan(got) & np.isnan(want))
    assert same.all(), f"{(~same).sum()} of {same.size} differ, first at {np.argwhere(~same)[0]}"


# 95 and 96 tiles of 32 rows at a longer K and, with few tiles of the other
# kernel, at a short one, 128 and 130 at a short one, 256 and 272 tiles of 64 rows,
# a lone last row of a tile in each direction, one block and several
@pytest.mark.parametrize("rows,n,k", [(31, 12160, 1280), (31, 12161, 1280), (97, 3073, 1536), (64, 6144, 512),
                                      (64, 6145, 256), (33, 8192, 512), (33, 8193, 512), (33, 12289, 256), (97, 6145, 768),
                                      (192, 4096, 1024), (1024, 2048, 256), (1025, 2048, 512), (65, 16513, 256),
                                      (2047, 1025, 1024)])
def test_tiles_and_rules(gpu, oracle, rows, n, k):
    check(gpu, oracle, rows, n, k, bias=rows % 2 == 1)


@pytest.mark.parametrize("rows,n", [(250, 3100), (300, 7000)])
def test_refusals(gpu, oracle, rows, n):
    def edit(wb, x):
        blocks = wb.reshape(n, 2, 144)
        blocks[5, 0, 2:4] = (0x00, 0x7C)          # dmin = inf
        blocks[n - 1, 1, 0:2] = (0x01, 0x7E)      # d = NaN
        x[7, 3] = np.nan
        x[rows - 1, 100] = np.float32(1e30)

    check(gpu, oracle, rows, n, 512, edit=edit, bias=True)


@pytest.mark.parametrize("rows,n", [(250, 3100), (300, 7000)])
def test_subnormal_scale_products(gpu, oracle, rows, n):
    """Scale products d * dx and dmin * dx that are subnormal, zero or among
    the smallest normal numbers: the outer product on the matrix cores rounds
    them as the multiplication does."""
    def edit(wb, x):
        rng = np.random.default_rng(n)
        blocks = wb.reshape(n, 2, 144)
        d = rng.integers(0, 0x0800, (n, 2, 2), dtype=np.uint16)  # f16 up to 2^-13, subnormal ones among them
        blocks[:, :, :4] = d.astype("<u2").view(np.uint8).reshape(n, 2, 4)
        x *= (10.0 ** rng.uniform(-38, -28, (rows, 1))).astype(np.float32)

    check(gpu, oracle, rows, n, 512, edit=edit)
