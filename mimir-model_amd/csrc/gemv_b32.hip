// Q8_0, Q4_K and Q6_K weights x 1..8 rows of 8-bit activations in blocks of
// 32 (dequant_matmul_a8.v1, or v2 with block = 32), in the float order of
// the reference's block-32 kernels dotQ8_0Q8AVX2, dotQ4KQ8AVX2 and
// dotQ6KQ8AVX2 (internal/kernels/kernels_amd64.s:1003-1043, 428-597,
// 760-882), whose x4 variants give the same bits: per output eight SIMD
// lanes ("chains"), chain c owning elements 4c..4c+3 of every run of 32.
// With P_j the exact integer sum of those four products of sub-block j:
//   Q8_0  acc = fma(f32(P_j), f32(dw_j * dx_j), acc)
//   Q4_K, Q6_K, per block of 256: A over the even and B over the odd
//         sub-blocks j in order, fma(f32(sc_j * P_j), dx_j, .) from 0; then
//         tot = fma(d, A + B, tot), and for Q4_K off = fma(dmin * f32(m_c),
//         dbs_c, off) (chain c owns sub-block c's min), result tot - off;
// and the eight chains end in HSUM1. The lane orders are restated from the
// assembly text; no golden output of the reference pins them, so they are
// checked against the oracle's restatement bit for bit and against the spec
// tolerance.
//
// Two forms, bit for bit the same.
//
// Two phases (gemv_b32_kernel), for grids that the latency of a chain's loads
// would bound: the chains are serial over K, the integer sums are not. A
// workgroup owns eight weight rows and takes K in stages of 1024 elements:
// every thread multiplies 32 weights of one row with the M activation rows
// (v_dot4_i32_i8, quants held in LDS) and leaves the eight sums as floats in
// LDS; then a lane per (weight row, chain) of wave m % 4 runs the stage's
// fmas of activation row m, reading them back (rows 4..7 in a second pass).
// The next stage's loads run under the second phase; more stages ahead
// measured slower (4096 x 4096 Q8_0 at one row 8.7, 9.7 and 10.8 us with
// one, two and three).
// Bound: latency at these sizes (a stage's two phases and its memory round
// trip). Measured on MI355X with the quantizer launch, against one group of
// eight lanes per row that loaded its four bytes a block as the chain came
// to them: 4096 x 4096 at 1 / 8 rows Q8_0 31.0 / 50.6 -> 8.7 / 17.5 us,
// Q4_K 12.0 / 37.2 -> 8.8 / 19.1, Q6_K 35.5 / 130 -> 9.5 / 19.7; Q8_0
// 14336 x 4096 at one row 35.5 -> 14.9 us, 2048 x 8192 57 -> 11.1 us.
//
// Direct (direct_kernel), where many weight rows keep the vector units busy by
// themselves: a group of eight lanes per row, lane c running chain c in
// registers, no sum through LDS. direct() below says which form runs.
//
// Rows of W with a non-finite block scale and refused activation rows take
// the float32 path (reference interp/fast.go:323-377).
#include <algorithm>

#include "f32path.hpp"
#include "kquant_lane.hpp"
#include "mimg_device.hpp"
#include "mimg_kernels.hpp"

namespace mimg {
namespace b32v {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int R = 8;        // weight rows a workgroup
constexpr int SE = 1024;    // elements a stage
constexpr int NJ = SE / 32; // sub-blocks of 32 a stage
constexpr int VS = NJ * 8 + 8;  // floats of a row's sums: the rows of a chain read start 8 banks apart
constexpr int DS = NJ + 4;      // floats of a row's scales

struct Args {
    const uint8_t* W;
    int64_t rb;
    int64_t N, K;
    const int8_t* q;       // [rows][K]
    const float* d32;      // [rows][K/32]
    const float* dbs;      // [rows][K/32]
    const int32_t* ok;     // [rows]
    const uint8_t* wref;   // [N]
    const float* x;        // [rows][K]
    const float* bias;
    float* y;
    int fused;
};

// One thread's raw weights of a stage: Q8_0 a block (its quants as the nine
// dwords that hold them, and its scale), Q4_K and Q6_K lane l's share of a block.
template <uint32_t DT>
struct Raw;
template <>
struct Raw<DT_Q8_0> {
    uint32_t v[9], d;
};
template <>
struct Raw<DT_Q4_K> {
    u32x4 hdr, q;
};
template <>
struct Raw<DT_Q6_K> {
    Q6KRaw r;
};

__device__ __forceinline__ void load_raw(const uint8_t* row, int64_t nblk, int s, int i, Raw<DT_Q8_0>& w) {
    const uint8_t* blk = row + min((int64_t)NJ * s + i, nblk - 1) * Q80_BYTES;
    const uint32_t* b = (const uint32_t*)__builtin_align_down(blk + 2, 4);
    const u32x4a4 v0 = *(const u32x4a4*)b, v1 = *(const u32x4a4*)(b + 4);
    w.v[0] = v0.x, w.v[1] = v0.y, w.v[2] = v0.z, w.v[3] = v0.w;
    w.v[4] = v1.x, w.v[5] = v1.y, w.v[6] = v1.z, w.v[7] = v1.w;
    w.v[8] = b[8];
    w.d = load_u16(blk) | ((uint32_t)((uintptr_t)(blk + 2) & 3) << 16);
}
__device__ __forceinline__ void load_raw(const uint8_t* row, int64_t nblk, int s, int i, Raw<DT_Q4_K>& w) {
    const uint8_t* blk = row + min((int64_t)(NJ / 8) * s + (i >> 3), nblk - 1) * Q4K_BYTES;
    w.hdr = *(const u32x4a4*)blk;
    w.q = *(const u32x4a4*)(blk + 16 + 16 * (i & 7));
}
__device__ __forceinline__ void load_raw(const uint8_t* row, int64_t nblk, int s, int i, Raw<DT_Q6_K>& w) {
    w.r = q6k_load(row + min((int64_t)(NJ / 8) * s + (i >> 3), nblk - 1) * Q6K_BYTES, i & 7);
}

template <uint32_t DT, int M>
__global__ __launch_bounds__(256) void gemv_b32_kernel(Args A) {
    constexpr bool KQ = DT != DT_Q8_0;
    constexpr int MH = M < 4 ? M : 4;                   // activation rows a pass
    __shared__ __align__(16) float V[MH * R * VS];      // [m][row][sub-block][chain] of a pass
    __shared__ __align__(16) uint8_t yq[2][M * SE];     // activation quants of a stage
    __shared__ __align__(16) float dx[2][M * NJ];       // their scales
    __shared__ __align__(16) float db[2][DT == DT_Q4_K ? M * NJ : 1];  // and scaled sums
    // Q8_0: dw * dx [m][row][sub-block] of a pass; K-quants: d [row][block], Q4_K also
    // dmin * m [row][sub-block]
    __shared__ __align__(16) float sc[KQ ? R * DS : MH * R * DS];
    __shared__ float dk[KQ ? R * 4 : 1];
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int64_t n0 = (int64_t)blockIdx.x * R;
    const int pr = t >> 5, pi = t & 31;  // phase 1: row, and unit of 32 weights
    const int64_t R32 = A.K / 32, nblk = KQ ? A.K / 256 : R32;
    const uint8_t* wrow = A.W + min(n0 + pr, A.N - 1) * A.rb;
    const int nst = (int)((A.K + SE - 1) / SE);

    // Loads past the row repeat its last bytes (their sums are not used).
    Raw<DT> raw;
    uint32_t aq[M];
    float ad, ab;
    auto load = [&](int s) {
        s = min(s, nst - 1);
        load_raw(wrow, nblk, s, pi, raw);
        const int64_t e = min((int64_t)SE * s + 4 * t, A.K - 4);
#pragma unroll
        for (int m = 0; m < M; m++) aq[m] = *(const uint32_t*)(A.q + m * A.K + e);
        const int64_t j = min(t / NJ, M - 1) * R32 + min((int64_t)NJ * s + t % NJ, R32 - 1);
        ad = A.d32[j];
        if constexpr (DT == DT_Q4_K) ab = A.dbs[j];
    };

    // phase 2: row pr2, chain c of activation row 4 i + wave in pass i
    constexpr int MW = (M + 3) / 4;
    const int pr2 = lane >> 3, c = lane & 7;
    float tot[MW], off[MW];
#pragma unroll
    for (int i = 0; i < MW; i++) tot[i] = off[i] = 0.f;

    load(0);
    for (int s = 0; s < nst; s++) {
#pragma unroll
        for (int m = 0; m < M; m++) *(uint32_t*)(&yq[s & 1][m * SE + 4 * t]) = aq[m];
        if (t < M * NJ) {
            dx[s & 1][t] = ad;
            if constexpr (DT == DT_Q4_K) db[s & 1][t] = ab;
        }
        lds_barrier();  // the stage's activations are in LDS, the last stage's sums read
        const uint8_t* ys = &yq[s & 1][0];
        // the thread's 32 weights as bytes: two runs of 16
        uint32_t lo[4], hi[4];
        int scl = 0, sch = 0;         // K-quants: the runs' scales,
        int vl = 8 * pi, vh = vl + 4; // their sums' places in a row of V
        int yl = 32 * pi, yh = yl + 16;  // and their activations'
        float dw = 0.f;
        if constexpr (DT == DT_Q8_0) {
            dw = f16_to_f32(raw.d & 0xFFFFu);
#pragma unroll
            for (int k = 0; k < 4; k++) {
                lo[k] = __builtin_amdgcn_alignbyte(raw.v[k + 1], raw.v[k], raw.d >> 16);
                hi[k] = __builtin_amdgcn_alignbyte(raw.v[k + 5], raw.v[k + 4], raw.d >> 16);
            }
        } else if constexpr (DT == DT_Q4_K) {
            const int blk = pi >> 3, l = pi & 7;
            const Q4KLane w = q4k_lane(raw.hdr, raw.q, l);
#pragma unroll
            for (int k = 0; k < 4; k++) lo[k] = w.lo[k], hi[k] = w.hi[k];
            scl = w.scl, sch = w.sch;
            vl = 8 * (8 * blk + 2 * (l >> 1)) + 4 * (l & 1), vh = vl + 8;
            yl = 256 * blk + w.yoff, yh = yl + 32;
            sc[pr * DS + 8 * blk + l] = w.dmin * (float)w.mm;
            if (l == 0) dk[pr * 4 + blk] = w.d;
        } else {
            const Q6KRaw& r = raw.r;
            const int blk = pi >> 3, l = pi & 7, h = l >> 2, pp = l & 3;
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const uint32_t ql = __builtin_amdgcn_alignbyte(r.ql[k + 1], r.ql[k], r.shift);
                const uint32_t qh = __builtin_amdgcn_alignbyte(r.qh[k + 1], r.qh[k], r.shift) >> (2 * (pp >> 1));
                // q - 32 per byte, no borrow between bytes
                const uint32_t q0 = (ql & 0x0F0F0F0Fu) | ((qh & 0x03030303u) << 4);
                const uint32_t q1 = ((ql >> 4) & 0x0F0F0F0Fu) | (((qh >> 4) & 0x03030303u) << 4);
                lo[k] = ((q0 | 0x80808080u) - 0x20202020u) ^ 0x80808080u;
                hi[k] = ((q1 | 0x80808080u) - 0x20202020u) ^ 0x80808080u;
            }
            scl = r.scl, sch = r.sch;
            vl = 8 * (8 * blk + 4 * h + (pp >> 1)) + 4 * (pp & 1), vh = vl + 16;
            yl = 256 * blk + 128 * h + 32 * (pp >> 1) + 16 * (pp & 1), yh = yl + 64;
            if (l == 0) dk[pr * 4 + blk] = f16_to_f32(r.dbits);
        }
        load(s + 1);
        const int64_t left = R32 - (int64_t)NJ * s;  // sub-blocks of the row from this stage on
#pragma unroll
        for (int i = 0; i < MW; i++) {
            if (i > 0) lds_barrier();  // the last pass's sums are read
#pragma unroll
            for (int k = 0; k < MH; k++) {
                const int m = 4 * i + k;
                if (m >= M) break;
                const u32x4 ya = *(const u32x4*)(ys + m * SE + yl), yb = *(const u32x4*)(ys + m * SE + yh);
                auto sum = [&](uint32_t w, uint32_t y, int scale) {
                    const int P = sdot4(w, y, 0);
                    return (float)(KQ ? __mul24(scale, P) : P);
                };
                float* v = V + (k * R + pr) * VS;
                *(f32x4*)(v + vl) = f32x4{sum(lo[0], ya.x, scl), sum(lo[1], ya.y, scl), sum(lo[2], ya.z, scl), sum(lo[3], ya.w, scl)};
                *(f32x4*)(v + vh) = f32x4{sum(hi[0], yb.x, sch), sum(hi[1], yb.y, sch), sum(hi[2], yb.z, sch), sum(hi[3], yb.w, sch)};
                if constexpr (!KQ) sc[(k * R + pr) * DS + pi] = dw * dx[s & 1][m * NJ + pi];
            }
            lds_barrier();
            const int m = 4 * i + wave;
            if (m >= M) continue;
            const float* v = V + (wave * R + pr2) * VS + c;
            if constexpr (!KQ) {
                const float* dd = sc + (wave * R + pr2) * DS;
                if (left >= NJ) {
#pragma unroll
                    for (int j = 0; j < NJ; j++) tot[i] = __builtin_fmaf(v[8 * j], dd[j], tot[i]);
                } else {
                    for (int j = 0; j < (int)left; j++) tot[i] = __builtin_fmaf(v[8 * j], dd[j], tot[i]);
                }
            } else {
                const float* dj = &dx[s & 1][m * NJ];
#pragma unroll
                for (int b = 0; b < NJ / 8; b++) {
                    if (8 * b >= left) break;
                    float a = 0.f, o = 0.f;
#pragma unroll
                    for (int j = 0; j < 8; j += 2) {
                        a = __builtin_fmaf(v[8 * (8 * b + j)], dj[8 * b + j], a);
                        o = __builtin_fmaf(v[8 * (8 * b + j + 1)], dj[8 * b + j + 1], o);
                    }
                    tot[i] = __builtin_fmaf(dk[pr2 * 4 + b], a + o, tot[i]);
                    if constexpr (DT == DT_Q4_K)
                        off[i] = __builtin_fmaf(sc[pr2 * DS + 8 * b + c], db[s & 1][m * NJ + 8 * b + c], off[i]);
                }
            }
        }
    }
    const int64_t n = n0 + pr2, nc = min(n, A.N - 1);
    const bool wok = A.wref[nc] == 0;
#pragma unroll
    for (int i = 0; i < MW; i++) {
        const int m = 4 * i + wave;
        if (m >= M) break;
        float r = DT == DT_Q4_K ? tot[i] - off[i] : tot[i];
        // HSUM1: c_l = a_l + a_{l+4}, c0 + c1 and c2 + c3, their sum
        r += __shfl_xor(r, 4);
        r += __shfl_xor(r, 1);
        r += __shfl_xor(r, 2);
        if (!wok || !A.ok[m]) r = f32dot_g8<DT>(A.W + nc * A.rb, A.x + (int64_t)m * A.K, A.K, A.fused != 0);
        if (A.bias) r += A.bias[nc];
        if (c == 0 && n < A.N) A.y[(int64_t)m * A.N + n] = r;
    }
}

// Lane c of a group of eight owns elements 4c..4c+3 of every run of 32 of one
// weight row, and with Q4_K the min of sub-block c; M activation rows.
template <uint32_t DT, int M>
__global__ __launch_bounds__(256) void direct_kernel(Args A) {
    const int g = threadIdx.x >> 3, l = threadIdx.x & 7;
    const int64_t row = (int64_t)blockIdx.x * 32 + g, rowc = min(row, A.N - 1);
    const uint8_t* wrow = A.W + rowc * A.rb;
    const int64_t K = A.K, R32 = K / 32, nb = DT == DT_Q8_0 ? R32 : K / 256;
    float tot[M], off[M];
#pragma unroll
    for (int m = 0; m < M; m++) tot[m] = off[m] = 0.f;
    for (int64_t b = 0; b < nb; b++) {
        if constexpr (DT == DT_Q8_0) {
            const uint8_t* blk = wrow + b * Q80_BYTES;
            const uint32_t* a = (const uint32_t*)__builtin_align_down(blk + 2 + 4 * l, 4);
            const uint32_t wq = __builtin_amdgcn_alignbyte(a[1], a[0], (uint32_t)((uintptr_t)(blk + 2) & 3));
            const float dw = f16_to_f32(load_u16(blk));
#pragma unroll
            for (int m = 0; m < M; m++) {
                const int P = sdot4(wq, *(const uint32_t*)(A.q + m * K + 32 * b + 4 * l), 0);
                tot[m] = __builtin_fmaf((float)P, dw * A.d32[m * R32 + b], tot[m]);
            }
        } else if constexpr (DT == DT_Q4_K) {
            const uint8_t* blk = wrow + b * Q4K_BYTES;
            const u32x4 hdr = *(const u32x4a4*)blk;
            const float d = f16_to_f32(hdr.x & 0xFFFFu), dmin = f16_to_f32(hdr.x >> 16);
            const Q4KScales s = q4k_scales(hdr.y, hdr.z, hdr.w);
            uint32_t qd[4];
#pragma unroll
            for (int c = 0; c < 4; c++) qd[c] = *(const uint32_t*)(blk + 16 + 32 * c + 4 * l);
            const float dm = dmin * (float)byte_of(s.m, l);
#pragma unroll
            for (int m = 0; m < M; m++) {
                const float* dx = A.d32 + m * R32 + 8 * b;
                off[m] = __builtin_fmaf(dm, A.dbs[m * R32 + 8 * b + l], off[m]);
                float a = 0.f, o = 0.f;
#pragma unroll
                for (int c = 0; c < 4; c++) {
                    const int8_t* yc = A.q + m * K + 256 * b + 64 * c + 4 * l;
                    const int lo = sdot4(qd[c] & 0x0F0F0F0Fu, *(const uint32_t*)yc, 0);
                    const int hi = sdot4((qd[c] >> 4) & 0x0F0F0F0Fu, *(const uint32_t*)(yc + 32), 0);
                    a = __builtin_fmaf((float)((int)byte_of(s.sc, 2 * c) * lo), dx[2 * c], a);
                    o = __builtin_fmaf((float)((int)byte_of(s.sc, 2 * c + 1) * hi), dx[2 * c + 1], o);
                }
                tot[m] = __builtin_fmaf(d, a + o, tot[m]);
            }
        } else {
            const uint8_t* blk = wrow + b * Q6K_BYTES;
            const uint32_t sh = (uint32_t)((uintptr_t)blk & 3);  // 2-byte aligned blocks
            auto load4 = [&](const uint8_t* p) {
                const uint32_t* a = (const uint32_t*)__builtin_align_down(p, 4);
                return __builtin_amdgcn_alignbyte(a[1], a[0], sh);
            };
            const float d = f16_to_f32(load_u16(blk + 208));
            uint32_t ql[4], qh[2];
#pragma unroll
            for (int j = 0; j < 4; j++) ql[j] = load4(blk + 64 * (j >> 1) + 32 * (j & 1) + 4 * l);
#pragma unroll
            for (int h = 0; h < 2; h++) qh[h] = load4(blk + 128 + 32 * h + 4 * l);
            int sc[8];
#pragma unroll
            for (int j = 0; j < 8; j++) sc[j] = (int)(int8_t)blk[192 + 8 * (j >> 2) + 2 * (j & 3) + (l >> 2)];
#pragma unroll
            for (int m = 0; m < M; m++) {
                const float* dx = A.d32 + m * R32 + 8 * b;
                float a = 0.f, o = 0.f;
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    const int h = j >> 2, p = j & 3;
                    const uint32_t q6 = ((ql[2 * h + (p & 1)] >> (4 * (p >> 1))) & 0x0F0F0F0Fu) |
                                        (((qh[h] >> (2 * p)) & 0x03030303u) << 4);
                    const uint32_t yv = *(const uint32_t*)(A.q + m * K + 256 * b + 32 * j + 4 * l);
                    const float v = (float)(sc[j] * (sdot4(q6, yv, 0) - 32 * sdot4(0x01010101u, yv, 0)));
                    if (j % 2 == 0) a = __builtin_fmaf(v, dx[j], a);
                    else o = __builtin_fmaf(v, dx[j], o);
                }
                tot[m] = __builtin_fmaf(d, a + o, tot[m]);
            }
        }
    }
    const bool wok = A.wref[rowc] == 0;
#pragma unroll
    for (int m = 0; m < M; m++) {
        float r = DT == DT_Q4_K ? tot[m] - off[m] : tot[m];
        r += __shfl_xor(r, 4);  // HSUM1, as above
        r += __shfl_xor(r, 1);
        r += __shfl_xor(r, 2);
        if (!wok || !A.ok[m]) r = f32dot_g8<DT>(wrow, A.x + m * K, K, A.fused != 0);
        if (A.bias) r += A.bias[rowc];
        if (l == 0 && row < A.N) A.y[(int64_t)m * A.N + row] = r;
    }
}

// The form for N x K weights and M activation rows: direct from the N on at
// which it measured faster on MI355X (both forms timed with the quantizer at
// every M, 13 N from 2048 to 128256 and 9 K from 256 to 8192). The two-phase
// form's LDS traffic grows with N M; the direct form's cost is the latency of
// its loads, which Q8_0's and Q6_K's 4-byte pieces of 2-byte aligned blocks
// make long, so only a short K or many rows pay there. Time of the two-phase
// form over the direct one's at M = 1 / 4 / 8:
//   Q4_K  4096 x 4096 0.80 / 0.70 / 0.51, 11008 x 4096 0.98 / 0.94 / 1.24,
//         14336 x 4096 0.98 / 1.04 / 1.46, 32768 x 2048 1.17 / 1.39 / 1.79,
//         128256 x 2048 1.24 / 1.64 / 2.06, 8192 x 512 1.07 / 1.20 / 1.17
//   Q8_0  14336 x 4096 0.44 / 0.58 / 0.79, 14336 x 1024 0.75 / 0.91 / 1.11,
//         32768 x 2048 0.67 / 0.98 / 1.38, 128256 x 2048 0.52 / 0.86 / 1.50,
//         32768 x 512 1.15 / 1.65 / 2.22
//   Q6_K  32768 x 512 1.18 / 1.10 / 1.05, 22000 x 256 1.39 / 1.36 / 1.27,
//         128256 x 1024 0.70 / 0.79 / 0.81
static bool direct(uint32_t dt, int64_t N, int64_t K, int M) {
    const bool part = K < 2048 && K % 1024 != 0;  // half a stage of the two-phase form is empty
    if (dt == DT_Q4_K) return N >= (K < 512 ? 5000 : part ? 8192 : M >= 7 ? 9000 : M >= 5 ? 8192 : 12000);
    if (dt == DT_Q6_K) return K < 512 ? N >= 12000 : K < 768 && N >= 32768;
    if (M >= 7) return N >= std::min<int64_t>(std::max<int64_t>(12 * K, 6000), 22000);
    if (M >= 5) return K <= 4096 && N >= std::min<int64_t>(std::max<int64_t>(18 * K, 8192), 32768);
    if (M == 4) return K <= 1536 && N >= std::max<int64_t>(20 * K, 8192);
    return K <= (M == 3 ? 768 : 512) && N >= 40 * K;
}

template <uint32_t DT, int M>
static hipError_t launch(const Args& A, hipStream_t stream) {
    const bool dir = direct(DT, A.N, A.K, M);
    const int64_t rows = dir ? 32 : R, nwg = (A.N + rows - 1) / rows;
    if (nwg > 0x7fffffff) return hipErrorInvalidValue;
    if (dir) hipLaunchKernelGGL((direct_kernel<DT, M>), dim3((unsigned)nwg), dim3(256), 0, stream, A);
    else hipLaunchKernelGGL((gemv_b32_kernel<DT, M>), dim3((unsigned)nwg), dim3(256), 0, stream, A);
    return hipGetLastError();
}

template <uint32_t DT>
static hipError_t launch_rows(const Args& A, int rows, hipStream_t stream) {
    switch (rows) {
    case 1: return launch<DT, 1>(A, stream);
    case 2: return launch<DT, 2>(A, stream);
    case 3: return launch<DT, 3>(A, stream);
    case 4: return launch<DT, 4>(A, stream);
    case 5: return launch<DT, 5>(A, stream);
    case 6: return launch<DT, 6>(A, stream);
    case 7: return launch<DT, 7>(A, stream);
    default: return launch<DT, 8>(A, stream);
    }
}

}  // namespace b32v

hipError_t launch_gemv_b32(const DevWeight& w, const ActPtrs& a, int64_t rows, int64_t total_rows, const float* x,
                           const float* bias, float* y, hipStream_t stream) {
    if (w.k % (w.dt == DT_Q8_0 ? 32 : 256) || rows < 1 || rows > 8) return hipErrorInvalidValue;
    b32v::Args A;
    A.W = w.data;
    A.rb = w.row_bytes;
    A.N = w.n;
    A.K = w.k;
    A.q = a.q;
    A.d32 = a.d32;
    A.dbs = a.dbs;
    A.ok = a.ok;
    A.wref = w.wref;
    A.x = x;
    A.bias = bias;
    A.y = y;
    A.fused = total_rows <= 8;
    switch (w.dt) {
    case DT_Q8_0: return b32v::launch_rows<DT_Q8_0>(A, (int)rows, stream);
    case DT_Q4_K: return b32v::launch_rows<DT_Q4_K>(A, (int)rows, stream);
    case DT_Q6_K: return b32v::launch_rows<DT_Q6_K>(A, (int)rows, stream);
    }
    return hipErrorInvalidValue;
}

}  // namespace mimg
