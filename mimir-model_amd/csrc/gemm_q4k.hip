// Prefill GEMM, Q4_K weights x 8-bit activations in blocks of 256
// (dequant_matmul_a8.v2, block = 256), on the int8 matrix cores
// (v_mfma_i32_32x32x32_i8). The result equals the decode GEMV's bit for bit,
// as the reference's AMX/VNNI tile kernels equal its one-row kernel (reference
// internal/kernels/amx.go:194-316, amx_test.go:41-141): per (weight row n,
// activation row m) and block b the exact int32
//   S = sum_k sc_s(k) q_k y_k,   M = sum_k m_s(k) y_k (= sum_s m_s xs_s)
// then serially in block order tot = fma(f32(S), d*dx_b, tot) and off =
// fma(f32(M), dmin*dx_b, off), result tot - off (+ bias), as dotQ8KRef
// (q8k_test.go:38-102).
//
// Exact integer products: sc*q (up to 945) does not fit int8, so it is split
// in two planes, sc = 8 sh + sl with sh*q and sl*q at most 105 (the packed
// nibbles times a small constant), S = 8 H + L. M comes from the activation's
// per-32 sums on one v_mfma_f32_32x32x16_f16: xs = 64 hi + lo against 64 m_s
// and m_s, every operand an exact f16 and every partial sum an integer below
// 2^24. The scale products d*dx and dmin*dx of a 32 x 32 tile are one
// v_mfma_f32_32x32x1_2b_f32 (an outer product added to zero: each rounded as
// the multiplication rounds, measured bit for bit against it over all value
// classes), which leaves the vector unit four instructions an output and
// block (shift-add, conversion, two fmas) where it had six.
//
// Bound: the matrix cores and the vector unit, which a SIMD's two waves keep
// busy only partly at the same time (14336 x 4096 x 2048 rows: vector unit
// busy 59 %, matrix cores 43 % of the cycles). A wave takes 32 weight rows
// (the column operand: lane l holds row l % 32, unpacked in registers from
// the raw block) against MT tiles of 32 activation rows (the row operand).
// The float step runs at raised priority, so that the waves of a SIMD drift
// apart and one's MFMAs run under the other's vector instructions, without
// the barriers that make them do so in gemm_kquant.hip's kernel.
// A workgroup is four such waves on the same activation rows. A wave's raw
// weight blocks are in its own LDS slot: it reads a block into registers and
// issues the next one's copies at once, so that one buffer does. The int8
// activation rows (16-byte chunks XOR-swizzled by row), their scales and
// per-32 sums are double-buffered; all by global_load_lds, one barrier a block.
//
// Measured on MI355X against the 128 x 128 ping-pong tiles and the 16 x 16 x
// 64 tiles that ran these before, us with quantizing: 14336 x 4096 by 2048
// rows 371 -> 344, 512 rows 100 -> 89, 256 rows 70.8 -> 47.9, 64 rows 24.9 ->
// 22.9; 4096 x 4096 by 768 rows 72.6 -> 48.0, 384 rows 44 -> 32.7, 256 rows
// 25 -> 23; 11008 x 4096 by 2048 rows 310 -> 273.
//
// Rows of x the quantizer refused and weight rows with a non-finite block
// scale take the float32 path (reference interp/fast.go:323-377) at the end.
#include "f32path.hpp"
#include "mimg_device.hpp"
#include "mimg_kernels.hpp"

namespace mimg {
namespace gq4 {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v32f __attribute__((ext_vector_type(32)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));

template <int MT_, int NW_>
struct Cfg {
    static constexpr int MT = MT_, NW = NW_;
    static constexpr int T = 64 * NW, BN = 32 * NW, BM = 32 * MT;
    static constexpr int WCH = 9;  // 16-byte chunks of a block
    static constexpr int WSLOT = 16 * WCH;
    // A wave's own 32 rows: copied, read and overwritten by that wave alone.
    static constexpr int WDMA = (32 * WCH + 63) / 64;
    static constexpr int WWAVE = WDMA * 1024;      // incl. slack for the last copy
    static constexpr int WBYTES = NW * WWAVE;
    // The activations of a block, two stages.
    static constexpr int ADMA = BM * 16 / T;
    static constexpr int ABYTES = BM * 256;
    static constexpr int RDMA = (BM + T - 1) / T;  // copies of a row's scale (and sums) per thread
    static constexpr int XBYTES = RDMA * T * 16;
    static constexpr int DBYTES = RDMA * T * 4;
    static constexpr int BUF = ABYTES + XBYTES + DBYTES;
    static_assert(ADMA * T == BM * 16 && WBYTES + 2 * BUF <= 160 * 1024, "GEMM tile shape");
};

struct Args {
    const uint8_t* W;
    const uint8_t* wref;   // [N]
    const float* bias;     // [N] or null
    float* y;              // [M][N]
    int64_t rb;            // bytes per weight row
    int N, M, nb;
    int64_t K;
    const int8_t* q;       // [M][K]
    const float* d32;      // [M][K/32]
    const int16_t* xs;     // [M][K/32]
    const int32_t* ok;     // [M]
    const float* x;        // [M][K] f32 (fallback)
    int fused;             // float32 fallback order (rows of the whole call <= 8)
    int tiles_m;           // row tiles of BM activation rows
};

// s_waitcnt with vmcnt <= n (n < 64), the other counters unconstrained.
#define GQ4_WAIT_VMCNT(n) __builtin_amdgcn_s_waitcnt(((n) & 0xF) | (((n) >> 4) << 14) | (0x7 << 4) | (0xF << 8))

// The copies of a thread: block 0's sources; block b adds a constant step.
template <class C>
struct Copies {
    const uint8_t *w[C::WDMA], *a[C::ADMA], *x[C::RDMA], *d[C::RDMA];
    uint32_t wave;
    __device__ __forceinline__ void init(const Args& A, int n0, int m0) {
        const int t = threadIdx.x, l = t & 63;
        wave = __builtin_amdgcn_readfirstlane(t >> 6);
#pragma unroll
        for (int i = 0; i < C::WDMA; i++) {
            const int c = min(64 * i + l, 32 * C::WCH - 1), r = c / C::WCH, j = c - C::WCH * r;
            w[i] = A.W + (int64_t)min(n0 + 32 * (int)wave + r, A.N - 1) * A.rb + 16 * j;
        }
#pragma unroll
        for (int i = 0; i < C::ADMA; i++) {
            const int c = C::T * i + t, r = c >> 4, s = c & 15;
            a[i] = (const uint8_t*)A.q + (int64_t)min(m0 + r, A.M - 1) * A.K + 16 * (s ^ (r & 15));
        }
#pragma unroll
        for (int i = 0; i < C::RDMA; i++) {
            const int64_t row = (int64_t)min(m0 + min(C::T * i + t, C::BM - 1), A.M - 1) * (A.K / 32);
            x[i] = (const uint8_t*)(A.xs + row);
            d[i] = (const uint8_t*)(A.d32 + row);
        }
    }
    __device__ __forceinline__ void weights(int b, uint32_t lds) const {
#pragma unroll
        for (int i = 0; i < C::WDMA; i++) lds_copy16(w[i] + (int64_t)b * Q4K_BYTES, lds + C::WWAVE * wave + 1024 * i);
    }
    __device__ __forceinline__ void activations(int b, uint32_t lds) const {
#pragma unroll
        for (int i = 0; i < C::ADMA; i++) lds_copy16(a[i] + 256 * (int64_t)b, lds + 1024 * wave + 16 * C::T * i);
#pragma unroll
        for (int i = 0; i < C::RDMA; i++) lds_copy16(x[i] + 16 * (int64_t)b, lds + 1024 * wave + C::ABYTES + 16 * C::T * i);
#pragma unroll
        for (int i = 0; i < C::RDMA; i++)
            lds_copy4(d[i] + 32 * (int64_t)b, lds + 256 * wave + C::ABYTES + C::XBYTES + 4 * C::T * i);
    }
};

// One block of a wave's 32 weight rows: the lane's raw bytes, from which the
// two planes of a k step are built.
struct Block {
    u32x4 q[4];
    Q4KScales s;
    float d, dmin;
    __device__ __forceinline__ void read(const uint8_t* wr, int g) {
        const u32x4 h = *(const u32x4*)wr;
        d = f16_to_f32(h.x & 0xFFFFu);
        dmin = f16_to_f32(h.x >> 16);
        s = q4k_scales(h.y, h.z, h.w);
#pragma unroll
        for (int c = 0; c < 4; c++) q[c] = *(const u32x4*)(wr + 16 + 32 * c + 16 * g);
    }
    __device__ __forceinline__ void planes(int ks, v4i& H, v4i& L) const {
        const uint32_t sc = byte_of(s.sc, ks);
        const short sh = (short)(sc >> 3), sl = (short)(sc & 7);
        const s16x2 shp = {sh, sh}, slp = {sl, sl};
        const u32x4 qd = q[ks >> 1];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const s16x2 nib = as_s16x2((qd[k] >> (4 * (ks & 1))) & 0x0F0F0F0Fu);
            H[k] = (int)as_u32(nib * shp);
            L[k] = (int)as_u32(nib * slp);
        }
    }
};
template <class C>
__global__ __launch_bounds__(C::T, 2) void gemm_kernel(Args A) {
    constexpr int MT = C::MT;
    __shared__ __align__(16) uint8_t smem[C::WBYTES + 2 * C::BUF];  // weights, then two activation stages
    __shared__ int flags[1];
    const int t = threadIdx.x, l = t & 63;
    const int a = l & 31, g = l >> 5;
    const int ntn = (A.N + C::BN - 1) / C::BN;
    const int nwg = ntn * A.tiles_m;
    int wg = blockIdx.x;
    if (nwg % 8 == 0) wg = (wg % 8) * (nwg / 8) + wg / 8;  // row tiles of a weight tile on one XCD
    const int n0 = wg / A.tiles_m * C::BN, m0 = wg % A.tiles_m * C::BM;
    const int nb = A.nb;

    Copies<C> cp;
    cp.init(A, n0, m0);
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)smem);
    const int wr0 = 32 * (int)cp.wave;  // this wave's first weight row
    cp.weights(0, lds0);
    cp.activations(0, lds0 + C::WBYTES);
    if (t == 0) flags[0] = 0;
    lds_barrier();
    {
        int f = 0;
        for (int i = t; i < C::BN; i += C::T) f |= n0 + i < A.N && A.wref[n0 + i] != 0;
        for (int i = t; i < C::BM; i += C::T) f |= m0 + i < A.M && A.ok[m0 + i] == 0;
        if (f) flags[0] = 1;
    }
    float tot[MT][16], off[MT][16];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int i = 0; i < 16; i++) tot[mt][i] = off[mt][i] = 0.f;
    const int asw = (a & 15) ^ g;  // chunk 2 ks + g of row a: slot 2 ks ^ asw
    for (int b = 0; b < nb; b++) {
        GQ4_WAIT_VMCNT(0);
        lds_barrier();  // block b's copies have landed, block b - 1's activations are read
        const uint8_t* buf = smem + C::WBYTES + (b & 1) * C::BUF;
        const uint8_t* al = buf + a * 256;
        Block blk;
        blk.read(smem + C::WWAVE * cp.wave + a * C::WSLOT, g);
        if (b + 1 < nb) {
            cp.activations(b + 1, lds0 + C::WBYTES + ((b + 1) & 1) * C::BUF);
            __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the wave's weight slot is read
            cp.weights(b + 1, lds0);
        }
        v16i H[MT], L[MT];
        v4i av[MT];
#pragma unroll
        for (int i = 0; i < MT; i++) av[i] = *(const v4i*)(al + i * 8192 + 16 * asw);
        __builtin_amdgcn_s_setprio(0);
#pragma unroll
        for (int ks = 0; ks < 8; ks++) {
            v4i pH, pL;
            blk.planes(ks, pH, pL);
            v4i nx[MT];
#pragma unroll
            for (int i = 0; i < MT; i++)
                if (ks < 7) nx[i] = *(const v4i*)(al + i * 8192 + 16 * ((2 * ks + 2) ^ asw));
            const v16i z = {};
#pragma unroll
            for (int i = 0; i < MT; i++) {
                H[i] = __builtin_amdgcn_mfma_i32_32x32x32_i8(av[i], pH, ks ? H[i] : z, 0, 0, 0);
                L[i] = __builtin_amdgcn_mfma_i32_32x32x32_i8(av[i], pL, ks ? L[i] : z, 0, 0, 0);
            }
#pragma unroll
            for (int i = 0; i < MT; i++) av[i] = nx[i];
        }
        __builtin_amdgcn_s_setprio(1);
        const float* dl = (const float*)(buf + C::ABYTES + C::XBYTES);
        const float pb = g ? blk.dmin : blk.d;
        v8h bm;
        {
            const uint32_t mw[2] = {(uint32_t)blk.s.m, (uint32_t)(blk.s.m >> 32)};
            const h2 mul = g ? h2{(_Float16)1.0f, (_Float16)1.0f} : h2{(_Float16)64.0f, (_Float16)64.0f};
            const h2 c1024 = {(_Float16)1024.0f, (_Float16)1024.0f};
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const uint32_t u = __builtin_amdgcn_perm(0u, mw[j >> 1], (j & 1) ? 0x0C030C02u : 0x0C010C00u);
                const h2 f = (__builtin_bit_cast(h2, u | 0x64006400u) - c1024) * mul;
                bm[2 * j] = f.x;
                bm[2 * j + 1] = f.y;
            }
        }
#pragma unroll
        for (int i = 0; i < MT; i++) {
            // d*dx and dmin*dx of the tile (lanes g = 0 hold d, g = 1 dmin)
            const v32f z = {};
            const v32f dd = __builtin_amdgcn_mfma_f32_32x32x1f32(dl[32 * i + a], pb, z, 0, 0, 0);
            v16f Mm = {};
            {
                const u32x4 xw = *(const u32x4*)(buf + C::ABYTES + 16 * (32 * i + a));
                const uint32_t xd[4] = {xw.x, xw.y, xw.z, xw.w};
                const short sh = g ? 0 : 6;
                const s16x2 sh2 = {sh, sh};
                const uint32_t msk = g ? 0x003F003Fu : 0xFFFFFFFFu;
                const h2 cf = g ? h2{(_Float16)1024.0f, (_Float16)1024.0f} : h2{(_Float16)1088.0f, (_Float16)1088.0f};
                const s16x2 cadd = g ? s16x2{0x6400, 0x6400} : s16x2{0x6440, 0x6440};
                v8h v;
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const uint32_t u = as_u32(as_s16x2(xd[j]) >> sh2) & msk;
                    const h2 f = __builtin_bit_cast(h2, as_u32(as_s16x2(u) + cadd)) - cf;
                    v[2 * j] = f.x;
                    v[2 * j + 1] = f.y;
                }
                Mm = __builtin_amdgcn_mfma_f32_32x32x16_f16(v, bm, Mm, 0, 0, 0);
            }
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int S = (H[i][r] << 3) + L[i][r];
                tot[i][r] = __builtin_fmaf((float)S, dd[r], tot[i][r]);
                off[i][r] = __builtin_fmaf(Mm[r], dd[16 + r], off[i][r]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }

    // Outputs: lane l holds weight row n against activation rows m.
    const int n = n0 + wr0 + a;
    const int refused = flags[0];
    if (n < A.N && !(refused && A.wref[n] != 0)) {
        const float bn = A.bias ? A.bias[n] : 0.f;
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const int m = m0 + 32 * mt + 8 * (i >> 2) + 4 * g + (i & 3);
                if (m >= A.M) continue;
                if (refused && A.ok[m] == 0) continue;
                float res = tot[mt][i] - off[mt][i];
                if (A.bias) res += bn;
                A.y[(int64_t)m * A.N + n] = res;
            }
        }
    }
    if (!refused) return;
    // Refused pairs of the tile: the float32 path, one group of eight lanes
    // per (row, activation row).
    for (int pidx = t >> 3; pidx < C::BN * C::BM; pidx += C::T / 8) {
        const int nn = n0 + pidx % C::BN, m = m0 + pidx / C::BN;
        if (nn >= A.N || m >= A.M) continue;
        if (A.wref[nn] == 0 && A.ok[m] != 0) continue;
        float res = f32dot_g8<DT_Q4_K>(A.W + (int64_t)nn * A.rb, A.x + (int64_t)m * A.K, A.K, A.fused != 0);
        if (A.bias) res += A.bias[nn];
        if ((t & 7) == 0) A.y[(int64_t)m * A.N + nn] = res;
    }
}

template <class C>
static hipError_t launch(Args A, hipStream_t stream) {
    A.tiles_m = (A.M + C::BM - 1) / C::BM;
    const int64_t nwg = (int64_t)((A.N + C::BN - 1) / C::BN) * A.tiles_m;
    if (nwg > 0x7fffffff) return hipErrorInvalidValue;
    hipLaunchKernelGGL(gemm_kernel<C>, dim3((unsigned)nwg), dim3(C::T), 0, stream, A);
    return hipGetLastError();
}

}  // namespace gq4

// 128 weight rows by 64 activation rows a workgroup where that gives more
// than 256 workgroups, else by 32 rows where that gives at least 96; fewer:
// not taken (the 16 x 16 x 64 tiles, gemm_kquant16.hip). Nor above 16 rows up to
// 128 of them at one to three blocks a row, where the prologue weighs, if the other
// tiles' grid is a full one. Measured on MI355X,
// us with quantizing, 64-row tiles / 32-row tiles / 16 x 16 x 64 tiles:
// 14336 x 4096 by 512 rows (896 workgroups of 64 rows) 89 / 95 / -, 4096 x
// 4096 by 768 (384) 48.0 / 48.6, by 512 (256) 35.5 / 35.3, by 256 33 / 23.0 /
// 25, by 96 (96 workgroups of 32 rows) - / 22.5 / 23.4, by 64 (64) - / 22.5 /
// 19.5, 512 x 2048 by 181 (24) - / 14.7 / 14.9; 8192 x 512 by 48 (128) - / 9.9 /
// 9.2, 4096 x 256 by 128 (128) - / 9.1 / 8.5, but 6144 x 512 by 64 (96; 192 of
// the others) - / 9.9 / 12.8, 12288 x 512 by 64 (192) - / 10.3 / 10.9, 3072 x
// 1024 by 181 (144) - / 12.2 / 13.3, 16384 x 512 by 16 (128) - / 8.8 / 9.3.
bool launch_gemm_q4k(const DevWeight& w, const ActPtrs& a, int64_t rows, int64_t total_rows, const float* x,
                     const float* bias, float* y, hipStream_t stream, hipError_t* err) {
    const int64_t ntn = (w.n + 127) / 128;
    const int64_t nwg = ntn * ((rows + 31) / 32);
    if (nwg < 96) return false;
    if (w.k < 1024 && rows > 16 && nwg <= 128 && (w.n + 31) / 32 * ((rows + 63) / 64) >= (rows <= 64 ? 256 : 192)) return false;
    gq4::Args A;
    A.W = w.data;
    A.wref = w.wref;
    A.bias = bias;
    A.y = y;
    A.rb = w.row_bytes;
    A.N = (int)w.n;
    A.M = (int)rows;
    A.nb = (int)(w.k / 256);
    A.K = w.k;
    A.q = a.q;
    A.d32 = a.d32;
    A.xs = a.xs;
    A.ok = a.ok;
    A.x = x;
    A.fused = total_rows <= 8;
    *err = ntn * ((rows + 63) / 64) > 256 ? gq4::launch<gq4::Cfg<2, 4>>(A, stream) : gq4::launch<gq4::Cfg<1, 4>>(A, stream);
    return true;
}

}  // namespace mimg
