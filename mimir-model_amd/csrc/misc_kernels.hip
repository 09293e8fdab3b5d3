// Smaller kernels of the path: the per-row refusal scan of a weight, block
// decode (mim.Dequantize) and a streaming read.
#include "f32path.hpp"
#include "mimg_device.hpp"
#include "mimg_kernels.hpp"

namespace mimg {

// wref[j] = 1 if a block scale of row j is not finite: the 8-bit kernels
// refuse such rows (reference RowDot.DotQ8, internal/kernels/q8.go:125-130;
// dotQ8KRef checks d and dmin of Q4_K, d of Q6_K and Q8_0).
__global__ void weight_refusals_kernel(uint32_t dt, const uint8_t* __restrict__ w, int64_t n,
                                       int64_t nblk, int64_t bbytes, uint8_t* __restrict__ wref) {
    int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n) return;
    const uint8_t* row = w + j * nblk * bbytes;
    uint8_t bad = 0;
    for (int64_t b = 0; b < nblk; b++) {
        const uint8_t* blk = row + b * bbytes;
        if (dt == DT_Q4_K) bad |= (uint8_t)(!f16_finite(load_u16(blk)) || !f16_finite(load_u16(blk + 2)));
        else if (dt == DT_Q6_K) bad |= (uint8_t)!f16_finite(load_u16(blk + 208));
        else bad |= (uint8_t)!f16_finite(load_u16(blk));
    }
    wref[j] = bad;
}

hipError_t launch_weight_refusals(uint32_t dt, const uint8_t* w, int64_t n, int64_t k, uint8_t* wref,
                                  hipStream_t stream) {
    if (n <= 0) return hipSuccess;
    int64_t be = dt == DT_Q8_0 ? 32 : 256;
    int64_t bb = dt == DT_Q4_K ? Q4K_BYTES : dt == DT_Q6_K ? Q6K_BYTES : Q80_BYTES;
    hipLaunchKernelGGL(weight_refusals_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream,
                       dt, w, n, k / be, bb, wref);
    return hipGetLastError();
}

// Block decode, bit-exact with mim.Dequantize (reference quant.go:197-344).
template <uint32_t DT>
__global__ void dequantize_kernel(const uint8_t* __restrict__ src, int64_t n, float* __restrict__ dst) {
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n;
         e += (int64_t)gridDim.x * blockDim.x)
        dst[e] = decode_weight<DT>(src, e);
}

hipError_t launch_dequantize(uint32_t dt, const uint8_t* src, int64_t n, float* dst, hipStream_t stream) {
    if (n <= 0) return hipSuccess;
    int64_t blocks = (n + 255) / 256;
    dim3 grid((unsigned)(blocks < 65536 ? blocks : 65536)), blk(256);
    switch (dt) {
    case DT_Q4_K: hipLaunchKernelGGL(dequantize_kernel<DT_Q4_K>, grid, blk, 0, stream, src, n, dst); break;
    case DT_Q6_K: hipLaunchKernelGGL(dequantize_kernel<DT_Q6_K>, grid, blk, 0, stream, src, n, dst); break;
    case DT_Q8_0: hipLaunchKernelGGL(dequantize_kernel<DT_Q8_0>, grid, blk, 0, stream, src, n, dst); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// Streaming read of up to three byte ranges, the measuring stick of the
// HBM-bound kernels: workgroup w reads PER*4 KB of one range with 16-byte
// nontemporal loads, all of a thread's loads issued before any is used, and
// folds them with XOR. A store that depends on every loaded value (taken
// only for one bit pattern that random weights never produce) keeps the
// loads, so the kernel writes nothing in practice.
template <int PER>
__global__ __launch_bounds__(256) void stream_read_kernel(ReadRanges r, uint32_t* __restrict__ sink) {
    int64_t wg = blockIdx.x;
    int i = 0;
    while (i + 1 < r.count && wg >= r.wgs[i]) wg -= r.wgs[i++];
    constexpr int64_t CHUNK = (int64_t)PER * 256 * 16;
    const int64_t off = wg * CHUNK;
    const int64_t n16 = (r.len[i] - off < CHUNK ? r.len[i] - off : CHUNK) / 16;
    const u32x4* p = (const u32x4*)(r.src[i] + off);
    u32x4 v[PER];
#pragma unroll
    for (int k = 0; k < PER; k++) {
        const int64_t idx = threadIdx.x + 256 * k;
        v[k] = idx < n16 ? __builtin_nontemporal_load(p + idx) : u32x4{0, 0, 0, 0};
    }
    uint32_t x = 0;
#pragma unroll
    for (int k = 0; k < PER; k++) x ^= v[k].x ^ v[k].y ^ v[k].z ^ v[k].w;
    if (x == 0x9E3779B9u) sink[blockIdx.x & 1023] = x;
}

hipError_t launch_stream_read(const ReadRanges& r0, int per, uint32_t* sink, hipStream_t s) {
    ReadRanges r = r0;
    const int64_t chunk = (int64_t)per * 256 * 16;
    int64_t total = 0;
    for (int i = 0; i < r.count; i++) total += (r.wgs[i] = (r.len[i] + chunk - 1) / chunk);
    if (total <= 0 || total > 0x7fffffff) return hipErrorInvalidValue;
    const dim3 grid((unsigned)total);
    switch (per) {
    case 2: hipLaunchKernelGGL(stream_read_kernel<2>, grid, dim3(256), 0, s, r, sink); break;
    case 4: hipLaunchKernelGGL(stream_read_kernel<4>, grid, dim3(256), 0, s, r, sink); break;
    case 8: hipLaunchKernelGGL(stream_read_kernel<8>, grid, dim3(256), 0, s, r, sink); break;
    case 16: hipLaunchKernelGGL(stream_read_kernel<16>, grid, dim3(256), 0, s, r, sink); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace mimg
