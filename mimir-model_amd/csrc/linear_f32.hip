// dequant_matmul.v1 (reference linearF32/linearCols, interp/fast.go:161-183)
// in the reference's float order, bit for bit f32dot_g8 (f32path.hpp): per
// output 32 fused multiply-add chains (Y_r of SIMD lane l, r = 0..3,
// l = 0..7), each over K/32 weights in order, and the reference's HSUM of
// the 32 sums. Which weight belongs to which chain depends on the row count:
//   more than 8 rows: weight 32 s + 8 r + l is step s of chain (l, r);
//   up to 8 rows (the fused kernels, kernels.go:83-100), per block of 256
//     Q4_K  weight 64 c + 32 b + 8 st + l: chain (l, 2 (st & 1) + b), step 2 c + st / 2
//     Q6_K  weight 128 h + 32 p + 8 st + l: chain (l, p), step 4 h + st
//     Q8_0  as above
// A chain's steps must run one after another, each with its own rounding, so
// the work is K/32 steps deep and 32 * rows * N chains wide.
#include "f32path.hpp"
#include "mimg_device.hpp"
#include "mimg_kernels.hpp"

namespace mimg {
namespace lf32 {
typedef float v32f __attribute__((ext_vector_type(32)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4a4 __attribute__((ext_vector_type(4), aligned(4)));  // x may start at any float

// ---- more than 8 activation rows: the matrix cores -------------------------
//
// v_mfma_f32_32x32x1_2b_f32 is 2048 fused multiply-adds acc += a * b, one per
// (activation row, weight row, block), each rounded once: with its two blocks
// on two chains it is one step of both for a 32 x 32 tile (its results equal
// fmaf bit for bit, subnormals, infinities and NaN payloads included). Wave r
// of a 32 x 32 tile holds the eight chains of Y_r (128 accumulators a
// thread); a workgroup has WM such tiles side by side on one set of decoded
// weights. K runs in stages of 128, double-buffered in LDS in K order, a
// row's 16-byte chunk c at c ^ (row % 32): the operands of four MFMAs are one
// float4 of each row, and 16 rows of a read fall in 16 different chunks of
// banks. The activations are copied there directly (global_load_lds); each
// thread decodes 16 / WM weights of the next stage between the MFMAs of this
// one, from raw bytes loaded a stage earlier. Of the two waves on a SIMD one
// decodes before its MFMAs and the other after them (waves w and w ^ 4, or
// w and w ^ 1, share a SIMD), so that the matrix core and the vector unit of
// the SIMD work at the same time.
// Bound: the fp32 matrix rate (141 TFLOP/s for this instruction on MI355X);
// the decode, the copies and the sums at the end keep it at half of that.
// Measured on MI355X against a group of eight lanes per output, each weight
// decoded for each activation row: Q6_K 2048 x 8192 at 181 rows 3622 ->
// 107 us (57 TFLOP/s), Q4_K 8192 x 2048 at 512 rows 7577 -> 235 us (73),
// Q8_0 4096 x 4096 at 64 rows 394 -> 35 us, Q4_K 960 x 768 at 129 rows
// 76 -> 11 us. Without the decode between the MFMAs (both waves decoding
// first) 115 and 257 us; with the activations staged through registers
// 115 and 237 us.
constexpr int BN = 32, KS = 128;

// 8 weights of unit v (elements 8 v..8 v + 7 of the stage) as loaded.
struct VRaw {
    u32x4 h;           // Q4_K: the block's header; Q6_K: dwords 0..2 of the ql window, scale byte
    uint32_t a[4];     // Q4_K: 8 quant bytes; Q6_K: dwords of the qh window, d; Q8_0: dwords of the quants, d
};

template <uint32_t DT>
__device__ __forceinline__ VRaw vload(const uint8_t* row, int s, int v, int64_t K) {
    VRaw r = {};
    const int j = v >> 2, st = v & 3;
    if constexpr (DT == DT_Q4_K) {
        const uint8_t* blk = row + (int64_t)s * Q4K_BYTES;
        r.h = *(const u32x4*)blk;
        const uint2 q = *(const uint2*)(blk + 16 + 32 * (j >> 1) + 8 * st);
        r.a[0] = q.x, r.a[1] = q.y;
    } else if constexpr (DT == DT_Q6_K) {
        const uint8_t* blk = row + (int64_t)s * Q6K_BYTES;
        const int h = j >> 2, p = j & 3;
        const uint32_t* ql = (const uint32_t*)__builtin_align_down(blk + 64 * h + 32 * (p & 1) + 8 * st, 4);
        const uint32_t* qh = (const uint32_t*)__builtin_align_down(blk + 128 + 32 * h + 8 * st, 4);
        r.h.x = ql[0], r.h.y = ql[1], r.h.z = ql[2];
        r.h.w = blk[192 + 8 * h + 2 * p + (st >> 1)];
        r.a[0] = qh[0], r.a[1] = qh[1], r.a[2] = qh[2];
        r.a[3] = load_u16(blk + 208) | ((uint32_t)((uintptr_t)blk & 3) << 16);
    } else {
        const uint8_t* blk = row + min((int64_t)(8 * s + j), K / 32 - 1) * Q80_BYTES;
        const uint32_t* q = (const uint32_t*)__builtin_align_down(blk + 2 + 8 * st, 4);
        r.a[0] = q[0], r.a[1] = q[1], r.a[2] = q[2];
        r.a[3] = load_u16(blk) | ((uint32_t)((uintptr_t)(blk + 2) & 3) << 16);
    }
    return r;
}

template <uint32_t DT>
__device__ __forceinline__ void vdecode(const VRaw& r, int v, float (&out)[8]) {
    const int j = v >> 2;
    if constexpr (DT == DT_Q4_K) {
        const float d = f16_to_f32(r.h.x & 0xFFFFu), dmin = f16_to_f32(r.h.x >> 16);
        const Q4KScales s = q4k_scales(r.h.y, r.h.z, r.h.w);
        const float ds = d * (float)byte_of(s.sc, j), ms = dmin * (float)byte_of(s.m, j);
        const int sh = (j & 1) * 4;
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const uint32_t q = (r.a[k] >> sh) & 0x0F0F0F0Fu;
#pragma unroll
            for (int i = 0; i < 4; i++) out[4 * k + i] = ds * (float)((q >> (8 * i)) & 0xFFu) - ms;
        }
    } else if constexpr (DT == DT_Q6_K) {
        const uint32_t sh = r.a[3] >> 16, p = (uint32_t)j & 3;
        const uint32_t ql[2] = {__builtin_amdgcn_alignbyte(r.h.y, r.h.x, sh), __builtin_amdgcn_alignbyte(r.h.z, r.h.y, sh)};
        const uint32_t qh[2] = {__builtin_amdgcn_alignbyte(r.a[1], r.a[0], sh), __builtin_amdgcn_alignbyte(r.a[2], r.a[1], sh)};
        const float s = f16_to_f32(r.a[3] & 0xFFFFu) * (float)(int8_t)r.h.w;
        const uint32_t lsh = (p >> 1) * 4, hsh = 2 * p;
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const uint32_t q = ((ql[k] >> lsh) & 0x0F0F0F0Fu) | (((qh[k] >> hsh) & 0x03030303u) << 4);
#pragma unroll
            for (int i = 0; i < 4; i++) out[4 * k + i] = s * (float)((int)((q >> (8 * i)) & 0xFFu) - 32);
        }
    } else {
        const uint32_t sh = r.a[3] >> 16;
        const uint32_t q[2] = {__builtin_amdgcn_alignbyte(r.a[1], r.a[0], sh), __builtin_amdgcn_alignbyte(r.a[2], r.a[1], sh)};
        const float d = f16_to_f32(r.a[3] & 0xFFFFu);
#pragma unroll
        for (int i = 0; i < 8; i++) out[i] = d * (float)(int8_t)(q[i >> 2] >> (8 * (i & 3)));
    }
}

template <int WM>
struct Tile {
    static constexpr int T = 256 * WM, BM = 32 * WM;
    static constexpr int BUF = (BN + BM) * KS;  // floats: weights, then activations
};

// KT: K is a multiple of it (KS, or 32 for a Q8_0 row that ends inside a
// stage). XA: the activation rows are 16-byte aligned.
template <uint32_t DT, int WM, int KT, bool XA>
__global__ __launch_bounds__(256 * WM, 2) void gemm_kernel(const uint8_t* __restrict__ W, int64_t rb, int64_t N,
                                                           int64_t K, const float* __restrict__ x, int M,
                                                           const float* __restrict__ bias, float* __restrict__ y,
                                                           int64_t tiles_n) {
    using L = Tile<WM>;
    constexpr int BM = L::BM, T = L::T;
    __shared__ __align__(16) float smem[2 * L::BUF];
    const int t = threadIdx.x, l = t & 63, wave = t >> 6;
    const int cw = wave & 3, wm = wave >> 2;
    const bool leader = ((wave ^ (wave >> 2)) & 1) == 0;
    // Consecutive workgroups of an XCD take the weight tiles of one
    // activation tile, whose rows (BM * K floats) then stay in its L2.
    const int64_t nwg = gridDim.x;
    int64_t wg = blockIdx.x;
    if (nwg % 8 == 0) wg = (wg % 8) * (nwg / 8) + wg / 8;
    const int64_t n0 = wg % tiles_n * BN;
    const int m0 = (int)(wg / tiles_n) * BM;

    const int nst = (int)((K + KS - 1) / KS);
    // decoded by this thread: units of 8 weights UW t.. of a stage's 32 x 16
    constexpr int UW = 2 / WM;
    const int wr = t * UW >> 4, u = t * UW & 15;
    const uint8_t* wrow = W + min(n0 + wr, N - 1) * rb;
    auto load_w = [&](int s, VRaw (&raw)[UW]) {
#pragma unroll
        for (int i = 0; i < UW; i++) raw[i] = vload<DT>(wrow, s >> 1, 16 * (s & 1) + u + i, K);
    };
    auto store_w = [&](int s, const VRaw (&raw)[UW]) {
        float* lw = smem + (s & 1) * L::BUF + wr * KS;
#pragma unroll
        for (int i = 0; i < UW; i++) {
            float v[8];
            vdecode<DT>(raw[i], 16 * (s & 1) + u + i, v);
            const int c = 2 * (u + i);
            *(f32x4*)(lw + 4 * (c ^ (wr & 31))) = f32x4{v[0], v[1], v[2], v[3]};
            *(f32x4*)(lw + 4 * ((c + 1) ^ (wr & 31))) = f32x4{v[4], v[5], v[6], v[7]};
        }
    };
    // stage s's activations: BM rows of 32 chunks (past K: the row's last
    // chunk again, never read)
    auto copy_x = [&](int s) {
        float* lx = smem + (s & 1) * L::BUF + BN * KS;
        const int64_t k0 = (int64_t)min(s, nst - 1) * KS;
        if constexpr (XA) {
#pragma unroll
            for (int i = 0; i < BM * 32 / T; i++) {
                const int c = T * i + t, row = c >> 5;
                const int64_t k = k0 + 4 * ((c ^ row) & 31);
                lds_copy16(x + (int64_t)min(m0 + row, M - 1) * K + (KT == KS ? k : min(k, K - 4)), lx + 4 * (T * i + 64 * wave));
            }
        } else {
#pragma unroll
            for (int i = 0; i < BM * 128 / T; i++) {
                const int f = T * i + t, row = f >> 7;
                const int64_t k = k0 + 4 * (((f >> 2) ^ row) & 31) + (f & 3);
                lds_copy4(x + (int64_t)min(m0 + row, M - 1) * K + (KT == KS ? k : min(k, K - 1)), lx + T * i + 64 * wave);
            }
        }
    };

    v32f acc[4];
#pragma unroll
    for (int r = 0; r < 4; r++)
#pragma unroll
        for (int i = 0; i < 32; i++) acc[r][i] = 0.f;

    VRaw raw[UW], next[UW];
    load_w(0, raw);
    load_w(min(1, nst - 1), next);
    copy_x(0);
    store_w(0, raw);
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
    lds_barrier();
    const int a = l & 31, op = 2 * cw + (l >> 5);
    for (int s = 0; s < nst; s++) {
        const float* lw = smem + (s & 1) * L::BUF + a * KS;
        const float* lx = lw + (BN + 32 * wm) * KS;
        auto step = [&](int g) {
            const int c = 4 * ((8 * g + op) ^ a);
            const f32x4 xa = *(const f32x4*)(lx + c), wb = *(const f32x4*)(lw + c);
#pragma unroll
            for (int i = 0; i < 4; i++) acc[i] = __builtin_amdgcn_mfma_f32_32x32x1f32(xa[i], wb[i], acc[i], 0, 0, 0);
        };
        // stage s + 1 goes to the other buffer, stage s + 2's weight bytes to
        // registers (past the end: the last stage again, not read)
#pragma unroll
        for (int i = 0; i < UW; i++) raw[i] = next[i];
        load_w(min(s + 2, nst - 1), next);
        copy_x(s + 1);
        __builtin_amdgcn_sched_barrier(0);  // the loads are not sunk to the end of the stage
        auto mfmas = [&]() {
            if constexpr (KT == KS) {
#pragma unroll
                for (int g = 0; g < KS / 32; g++) step(g);
            } else {
#pragma unroll 1
                for (int g = 0; g < (int)min((int64_t)KS, K - (int64_t)s * KS) / 32; g++) step(g);
            }
        };
        // one wave of a SIMD decodes while the other runs its MFMAs
        if (!leader) store_w(s + 1, raw);
        __builtin_amdgcn_sched_barrier(0);
        mfmas();
        __builtin_amdgcn_sched_barrier(0);
        if (leader) store_w(s + 1, raw);
        __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): stage s + 1's copies have landed
        lds_barrier();
    }

    // HSUM: T_l = (Y0 + Y1) + (Y2 + Y3) across the four waves of a tile, in
    // four rounds through LDS (chains l = i and i + 4 in round i), each wave
    // adding four of the 16 output registers; c_i = T_i + T_{i+4}, result
    // (c0 + c1) + (c2 + c3).
    float* ex = smem + wm * 4 * 32 * 64;
    float ci[4][4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
#pragma unroll
        for (int j = 0; j < 32; j++) ex[(cw * 32 + j) * 64 + l] = acc[i][j];
        lds_barrier();
#pragma unroll
        for (int q = 0; q < 4; q++) {
            float tt[2];
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const float* e = ex + (16 * h + 4 * cw + q) * 64 + l;
                tt[h] = (e[0] + e[32 * 64]) + (e[64 * 64] + e[96 * 64]);
            }
            ci[i][q] = tt[0] + tt[1];
        }
        lds_barrier();
    }
    const int64_t n = n0 + a;
    if (n >= N) return;
    const float bn = bias ? bias[n] : 0.f;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        float r = (ci[0][q] + ci[1][q]) + (ci[2][q] + ci[3][q]);
        if (bias) r += bn;
        const int m = m0 + 32 * wm + 8 * cw + 4 * (l >> 5) + q;
        if (m < M) y[(int64_t)m * N + n] = r;
    }
}

template <uint32_t DT, int WM, int KT, bool XA>
static hipError_t launch_gemm_k(const DevWeight& w, const float* x, int64_t rows, const float* bias, float* y,
                                hipStream_t stream) {
    const int64_t tn = (w.n + BN - 1) / BN, nwg = tn * ((rows + Tile<WM>::BM - 1) / Tile<WM>::BM);
    if (nwg > 0x7fffffff) return hipErrorInvalidValue;
    hipLaunchKernelGGL((gemm_kernel<DT, WM, KT, XA>), dim3((unsigned)nwg), dim3(256 * WM), 0, stream, w.data, w.row_bytes,
                       w.n, w.k, x, (int)rows, bias, y, tn);
    return hipGetLastError();
}

template <uint32_t DT, int WM>
static hipError_t launch_gemm(const DevWeight& w, const float* x, int64_t rows, const float* bias, float* y,
                              hipStream_t stream) {
    const bool xa = (uintptr_t)x % 16 == 0;
    if constexpr (DT == DT_Q8_0)
        if (w.k % KS) {
            if (xa) return launch_gemm_k<DT, WM, 32, true>(w, x, rows, bias, y, stream);
            return launch_gemm_k<DT, WM, 32, false>(w, x, rows, bias, y, stream);
        }
    if (xa) return launch_gemm_k<DT, WM, KS, true>(w, x, rows, bias, y, stream);
    return launch_gemm_k<DT, WM, KS, false>(w, x, rows, bias, y, stream);
}

// ---- up to 8 activation rows, and chunks of them ------------------------------
//
// A lane per (weight row, chain): the 32 lanes of a half-wave are one row's
// chains, with one accumulator per activation row. A workgroup owns 8 rows
// and takes K in stages of 256: each thread decodes 8 consecutive weights
// (one (sub-block, st): one step of the chains l = 0..7 of one r) into LDS as
// [row][4 l + r][step], where the row's lanes read their 8 steps as two
// float4; the activations sit beside them in the same order. The raw loads
// run PF stages ahead in registers: with two workgroups a CU the bytes in
// flight, not the arithmetic, bound a decode row.
constexpr int VR = 8, VS = 256 + 32;  // rows of 288 floats: the two rows of a wave write to different banks

// Chain r and step of unit v (elements 8 v..8 v + 7) of a stage.
template <uint32_t DT>
__device__ __forceinline__ int2 unit_chain(int v) {
    const int j = v >> 2, st = v & 3;
    if (DT == DT_Q4_K) return int2{2 * (st & 1) + (j & 1), 2 * (j >> 1) + (st >> 1)};
    if (DT == DT_Q6_K) return int2{j & 3, 4 * (j >> 2) + st};
    return int2{st, j};
}

template <uint32_t DT, int M, int PF>
__global__ __launch_bounds__(256) void gemv_kernel(const uint8_t* __restrict__ W, int64_t rb, int64_t N, int64_t K,
                                                   const float* __restrict__ x, int rows,
                                                   const float* __restrict__ bias, float* __restrict__ y) {
    const int m0 = blockIdx.y * M;  // activation rows m0 .. (past the last: the last again, unstored)
    __shared__ __align__(16) float lw[2][VR * VS];
    __shared__ __align__(16) float lx[2][M * 256];
    const int t = threadIdx.x, lane = t & 63;
    const int64_t n0 = (int64_t)blockIdx.x * VR;
    const int lr = t >> 5, v = t & 31;  // this thread's decoded row and unit
    const uint8_t* wrow = W + (int64_t)min(n0 + lr, N - 1) * rb;
    const int2 uc = unit_chain<DT>(v);
    float* const wst = &lw[0][lr * VS + 8 * uc.x + uc.y];  // + 32 l: chain (l, r) step
    const int2 xc = unit_chain<DT>(t >> 3);
    float* const xst = &lx[0][32 * (t & 7) + 8 * xc.x + xc.y];
    const int nst = (int)((K + 255) / 256);
    // Loads are unconditional (a load under a branch would wait for those
    // before it): past the last stage, and past K in a Q8_0 row of
    // K % 256 != 0, they repeat the last element; such steps are never read.
    auto load = [&](int s, VRaw& w, float (&xv)[M]) {
        const int sc = min(s, nst - 1);
        w = vload<DT>(wrow, sc, v, K);
        const float* xp = x + min((int64_t)256 * sc + t, K - 1);
#pragma unroll
        for (int m = 0; m < M; m++) xv[m] = xp[(int64_t)min(m0 + m, rows - 1) * K];
    };
    auto store = [&](int s, const VRaw& w, const float (&xv)[M]) {
        const int buf = s & 1;
        float wv[8];
        vdecode<DT>(w, v, wv);
#pragma unroll
        for (int i = 0; i < 8; i++) wst[buf * VR * VS + 32 * i] = wv[i];
#pragma unroll
        for (int m = 0; m < M; m++) xst[buf * M * 256 + 256 * m] = xv[m];
    };
    float acc[M];
#pragma unroll
    for (int m = 0; m < M; m++) acc[m] = 0.f;
    VRaw wq[PF];
    float xq[PF][M];
#pragma unroll
    for (int p = 0; p < PF; p++) load(p, wq[p], xq[p]);
    for (int s0 = 0; s0 < nst; s0 += PF) {
#pragma unroll
        for (int p = 0; p < PF; p++) {
            const int s = s0 + p;
            if (s >= nst) break;
            store(s, wq[p], xq[p]);
            load(s + PF, wq[p], xq[p]);
            lds_barrier();
            const float* ws = &lw[s & 1][(t >> 5) * VS + 8 * (t & 31)];
            const float* xs = &lx[s & 1][8 * (t & 31)];
            const int64_t left = (K - (int64_t)256 * s) / 32;
            if (DT != DT_Q8_0 || left >= 8) {
                const f32x4 w0 = *(const f32x4*)ws, w1 = *(const f32x4*)(ws + 4);
#pragma unroll
                for (int m = 0; m < M; m++) {
                    const f32x4 x0 = *(const f32x4*)(xs + 256 * m), x1 = *(const f32x4*)(xs + 256 * m + 4);
#pragma unroll
                    for (int i = 0; i < 4; i++) acc[m] = __builtin_fmaf(w0[i], x0[i], acc[m]);
#pragma unroll
                    for (int i = 0; i < 4; i++) acc[m] = __builtin_fmaf(w1[i], x1[i], acc[m]);
                }
            } else {
                for (int i = 0; i < (int)left; i++)
#pragma unroll
                    for (int m = 0; m < M; m++) acc[m] = __builtin_fmaf(ws[i], xs[256 * m + i], acc[m]);
            }
        }
    }
    // HSUM over the row's lanes 4 l + r: T_l, T_l + T_{l+4}, c0 + c1, e0 + e2
    const int64_t n = n0 + lr;
#pragma unroll
    for (int m = 0; m < M; m++) {
        float r = acc[m];
        r += __shfl_xor(r, 1);
        r += __shfl_xor(r, 2);
        r += __shfl_xor(r, 16);
        r += __shfl_xor(r, 4);
        r += __shfl_xor(r, 8);
        if (n < N && m0 + m < rows && (lane & 31) == 0) {
            if (bias) r += bias[n];
            y[(int64_t)(m0 + m) * N + n] = r;
        }
    }
}

template <uint32_t DT, int M>
static hipError_t launch_gemv(const DevWeight& w, const float* x, int64_t rows, const float* bias, float* y,
                              hipStream_t stream) {
    constexpr int PF = M <= 4 ? 4 : 3;
    const int64_t nwg = (w.n + VR - 1) / VR;
    if (nwg > 0x7fffffff) return hipErrorInvalidValue;
    hipLaunchKernelGGL((gemv_kernel<DT, M, PF>), dim3((unsigned)nwg, (unsigned)((rows + M - 1) / M)), dim3(256), 0, stream,
                       w.data, w.row_bytes, w.n, w.k, x, (int)rows, bias, y);
    return hipGetLastError();
}

template <uint32_t DT>
static hipError_t launch(const DevWeight& w, const float* x, int64_t rows, const float* bias, float* y,
                         hipStream_t stream) {
    // The GEMV in chunks of activation rows where its grid is small: of one, two
    // or four rows up to 256 workgroups (Q8_0 512; up to 8 rows only whole
    // chunks), and for Q8_0, whose chains are the same above 8 rows, of eight
    // rows up to 768. Measured on MI355X, us, in chunks / in one pass up to 8
    // rows, in tiles above (10 N from 8 to 8192, 6 K): Q8_0 512 x 2048 at 8 rows
    // 6.7 / 9.9, at 16 7.7 / 21.6, at 64 14.2 / 21.8, 2048 x 4096 at 16 rows
    // 23.2 / 38; 1000 x 256 at 33 rows 6.3 / 7.3; in chunks of eight from 769 to
    // 1024 workgroups at K <= 1024 0.96 to 1.07 of the tiles, up to 1536 1.29 to
    // 1.53 at K <= 512; Q4_K 512 x 2048 at 8 rows 6.2 / 9.9.
    if (rows <= 8 || DT == DT_Q8_0) {
        const int64_t nwg = (w.n + VR - 1) / VR;
        auto takes = [&](int m) {
            return (rows > 8 || rows % m == 0) && nwg * ((rows + m - 1) / m) <= (DT == DT_Q8_0 ? 512 : 256);
        };
        if (takes(1)) return launch_gemv<DT, 1>(w, x, rows, bias, y, stream);
        if (takes(2)) return launch_gemv<DT, 2>(w, x, rows, bias, y, stream);
        if (takes(4)) return launch_gemv<DT, 4>(w, x, rows, bias, y, stream);
        if (rows > 8 && nwg * ((rows + 7) / 8) <= 768) return launch_gemv<DT, 8>(w, x, rows, bias, y, stream);
    }
    switch (rows) {
    case 1: return launch_gemv<DT, 1>(w, x, rows, bias, y, stream);
    case 2: return launch_gemv<DT, 2>(w, x, rows, bias, y, stream);
    case 3: return launch_gemv<DT, 3>(w, x, rows, bias, y, stream);
    case 4: return launch_gemv<DT, 4>(w, x, rows, bias, y, stream);
    case 5: return launch_gemv<DT, 5>(w, x, rows, bias, y, stream);
    case 6: return launch_gemv<DT, 6>(w, x, rows, bias, y, stream);
    case 7: return launch_gemv<DT, 7>(w, x, rows, bias, y, stream);
    case 8: return launch_gemv<DT, 8>(w, x, rows, bias, y, stream);
    }
    // Tiles of 32 x 64 where they give at least three quarters of the CUs a
    // workgroup, else 32 x 32, two workgroups a CU (measured on MI355X: 192
    // workgroups of 64 rows, 2048 x 8192 at 181 rows, 107 against 125 us;
    // 128, 4096 x 4096 at 64 rows, 51 against 35 us).
    if ((w.n + BN - 1) / BN * ((rows + 63) / 64) >= 192) return launch_gemm<DT, 2>(w, x, rows, bias, y, stream);
    return launch_gemm<DT, 1>(w, x, rows, bias, y, stream);
}

}  // namespace lf32

hipError_t launch_linear_f32(const DevWeight& w, const float* x, int64_t rows, const float* bias, float* y,
                             hipStream_t stream) {
    if (rows <= 0 || w.n <= 0) return hipSuccess;
    if (rows > INT32_MAX) return hipErrorInvalidValue;
    switch (w.dt) {
    case DT_Q4_K: return lf32::launch<DT_Q4_K>(w, x, rows, bias, y, stream);
    case DT_Q6_K: return lf32::launch<DT_Q6_K>(w, x, rows, bias, y, stream);
    case DT_Q8_0: return lf32::launch<DT_Q8_0>(w, x, rows, bias, y, stream);
    }
    return hipErrorInvalidValue;
}

}  // namespace mimg
