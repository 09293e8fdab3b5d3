"""One-row K-quant GEMV (gemv_kquant.hip): 2 to 32 weight rows a workgroup
by the pairs that fill a pass, ragged last tiles, several matrices, bias and
refused rows, and the gate/up launch with 16 rows; bit for bit the oracle and
the separate launches."""
import numpy as np
import pytest

from test_gpu_parity import _dev_linear

pytestmark = pytest.mark.gpu

Q4_K, Q6_K = 66, 67


def same(got, want):
    eq = (got.view(np.uint32) == want.view(np.uint32)) | (np.isnan(got) & np.isnan(want))
    assert eq.all(), f"{(~eq).sum()} of {eq.size} differ, first at {np.argwhere(~eq)[0]}"


# rows a workgroup: 16 (K = 1024, 2048), 32 (one pass; three passes), 4, 8 and
# 2, each at a ragged row count; the last two keep the smaller tile
@pytest.mark.parametrize("dt", [Q4_K, Q6_K])
@pytest.mark.parametrize("n,k", [(16385, 1024), (16400, 2048), (32801, 768), (49153, 2560), (2051, 8192), (4099, 4096),
                                 (1030, 8192), (16383, 1024), (40001, 2816)])
def test_rows_per_workgroup(gpu, oracle, dt, n, k):
    wb = oracle.synthetic_weight(dt, n, k, seed=n + k)
    blocks = wb.reshape(n, k // 256, -1)
    blocks[n - 1, -1, (0 if dt == Q4_K else 208):][:2] = (0x00, 0x7C)  # the last row refused
    x = oracle.synthetic_acts(1, k, seed=k)
    W = gpu.Weight(wb, dt, n, k)
    got = _dev_linear(gpu, [W], x, prequant=True)[0]
    W.release()
    same(got, oracle.linear_a8(x, wb, dt, n, k, block=256, threads=16))


def test_two_matrices(gpu, oracle):
    """Two matrices in one launch with 16 rows a workgroup, tiles of each its own."""
    k, ns = 2048, (9000, 8001)
    wbs = [oracle.synthetic_weight(Q6_K, n, k, seed=n) for n in ns]
    x = oracle.synthetic_acts(1, k, seed=3)
    W = [gpu.Weight(wb, Q6_K, n, k) for wb, n in zip(wbs, ns)]
    got = _dev_linear(gpu, W, x, prequant=True)
    for w, wb, n, g in zip(W, wbs, ns, got):
        w.release()
        same(g, oracle.linear_a8(x, wb, Q6_K, n, k, block=256, threads=16))


@pytest.mark.parametrize("n,k,bad", [(4096, 2048, None), (4104, 1024, "weight"), (8192, 512, "act"), (4100, 2048, None),
                                     (4088, 2048, "weight")])
def test_gate_up(gpu, oracle, n, k, bad):
    import hiprt as rt

    x = oracle.synthetic_acts(1, k, seed=k)
    wbs = [oracle.synthetic_weight(Q4_K, n, k, seed=n + i) for i in range(2)]
    if bad == "weight":
        wbs[0].reshape(n, k // 256, 144)[n - 1, 0, :2] = (0x00, 0x7C)
        wbs[1].reshape(n, k // 256, 144)[13, 1, 2:4] = (0x01, 0x7E)
    if bad == "act":
        x[0, 7] = np.float32(3e18)
    W = [gpu.Weight(wb, Q4_K, n, k) for wb in wbs]
    bias = [oracle.synthetic_acts(1, n, seed=i)[0] for i in range(2)]
    s, dx, wsb = rt.Stream(), rt.DeviceBuffer.from_array(x), gpu.a8_workspace_bytes(1, k)
    dbs = [rt.DeviceBuffer.from_array(b) for b in bias]
    ws, out, g, u, want = rt.DeviceBuffer(wsb), *(rt.DeviceBuffer(n * 4) for _ in range(4))
    gpu.quantize_act_dev(dx.ptr, 1, k, 256, ws.ptr, wsb, s.handle)
    gpu.matmul_a8_quantized_swiglu_dev(W, dx.ptr, 1, [b.ptr for b in dbs], 256, out.ptr, 16, ws.ptr, wsb, s.handle)
    gpu.matmul_a8_quantized_group_dev(W, dx.ptr, 1, [b.ptr for b in dbs], 256, [g.ptr, u.ptr], ws.ptr, wsb, s.handle)
    gpu.swiglu_dev(g.ptr, u.ptr, want.ptr, n, 16, s.handle)
    s.sync()
    same(out.download(np.float32), want.download(np.float32))
    for w, wb, b, y in zip(W, wbs, bias, (g, u)):
        same(y.download(np.float32)[None], oracle.linear_a8(x, wb, Q4_K, n, k, bias=b, block=256, threads=16))
        w.release()
