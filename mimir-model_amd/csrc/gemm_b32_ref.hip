// Q8_0 weights x 8-bit activations in blocks of 32 (dequant_matmul_a8.v1 and
// .v2 with block = 32, reference interp/fast.go:246-379) for many activation
// rows, in the float order of dotQ8_0Q8AVX2 (reference
// internal/kernels/kernels_amd64.s:1003-1043), bit for bit the GEMV
// (gemv_b32.hip): per output eight chains, chain c over the blocks j
// in order
//   P = sum of elements 4c..4c+3 of w_j * y_j   (an exact integer)
//   acc_c = fma(f32(P), f32(dw_j * dx_j), acc_c)
// and HSUM1 of the eight.
//
// P comes from v_mfma_f32_16x16x4_4b_f16: its four blocks are four chains of
// a 16 x 16 tile, its k = 4 one chain's elements, and with the int8 values as
// f16 the sum of four products (below 2^16) is an exact f32, so the vector
// unit is left with one fma per chain and block and a quarter of a product
// of scales. (The int8 form would need a conversion of each sum: twice the
// vector instructions.) That fma is the bound: 32 of a 16 x 16 tile's 36
// vector instructions per block and wave.
//
// Tiling: a wave owns 16 weight rows and MT tiles of 16 activation rows with
// all eight chains (CS = 1), or with four of them (CS = 2, for few rows: two
// waves share a tile). The four waves of a workgroup share the activation
// rows and hold 64 / CS weight rows. K runs in stages of SB blocks: each
// thread loads its share of the raw bytes a stage ahead, converts it to f16
// (0x6400 | (q + 128) is f16(1152 + q)) and writes it to LDS, double-buffered,
// a row's 16-byte chunks permuted by row so that the lanes of a 16-row
// operand read meet each bank once. Small tiles take longer stages: there a
// stage is a memory round trip (4096 x 4096 at 16 rows 46 us with stages of
// two blocks, 27 with eight).
// Measured on MI355X with the quantizer launch, against the GEMV in chunks
// of eight rows: 14336 x 4096 at 181 rows 1361 -> 164 us, 2048 x 8192 at
// 512 rows 5247 -> 160 us, 1024 x 4096 at 64 rows 347 -> 27 us.
//
// Rows the quantizer refused and weight rows with a non-finite block scale
// take the float32 path at the end, as in the GEMV.
#include "f32path.hpp"
#include "mimg_device.hpp"
#include "mimg_kernels.hpp"

namespace mimg {
namespace b32r {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

struct Args {
    const uint8_t* W;
    const uint8_t* wref;   // [N]
    const float* bias;     // [N] or null
    float* y;              // [M][N]
    int64_t rb, K;
    int64_t N;
    int M, nblk;           // nblk = K / 32
    const int8_t* q;       // [M][K]
    const float* d32;      // [M][K/32]
    const int32_t* ok;     // [M]
    const float* x;        // [M][K] (float32 path)
    int fused;
    int tiles_m;
};

template <int MT_, int CS_, int SB_>
struct Cfg {
    static constexpr int MT = MT_, CS = CS_;
    static constexpr int BN = 64 / CS, BM = 16 * MT;
    static constexpr int SB = SB_;                      // blocks a stage
    static constexpr int ROW = SB * 64;                 // LDS bytes of a row: 32 SB f16
    static constexpr int WB = BN * ROW, AB = BM * ROW;
    static constexpr int DB = (BN + BM) * SB * 4;       // dw [SB][BN], dx [SB][BM]
    static constexpr int BUF = WB + AB + DB;
    static constexpr int WU = BN * 2 * SB, AU = BM * 2 * SB;      // units of 16 elements a stage
    static constexpr int WT = (WU + 255) / 256, AT = (AU + 255) / 256;
    static constexpr int RT = 256 / (2 * SB);           // rows of 256 units
    static constexpr int XT = (BM * SB + 255) / 256;    // activation scales a thread copies
    // the 16-byte chunk of a row where its chunk c sits
    static __device__ __forceinline__ int slot(int c, int r) { return SB >= 4 ? c ^ (r & 15) : c ^ ((r >> 1) & 7); }
};

// Four int8 as four f16: bytes q + 128 under 0x64 are f16(1024 + 128 + q).
__device__ __forceinline__ u32x2 cvt4(uint32_t q) {
    const uint32_t u = q ^ 0x80808080u;
    const h2 c = {(_Float16)1152.0f, (_Float16)1152.0f};
    const h2 lo = __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, u, 0x07010700u)) - c;
    const h2 hi = __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, u, 0x07030702u)) - c;
    return u32x2{__builtin_bit_cast(uint32_t, lo), __builtin_bit_cast(uint32_t, hi)};
}

// A unit's raw bytes: 16 elements of a weight block (with its scale) or of
// an activation row.
struct WUnit {
    uint32_t v[5], d;
};

template <class C>
__global__ __launch_bounds__(256, 2) void gemm_q8_0_kernel(Args A) {
    constexpr int MT = C::MT, CS = C::CS, BN = C::BN, BM = C::BM, SB = C::SB;
    __shared__ __align__(16) uint8_t smem[2 * C::BUF];
    __shared__ int flags[1];
    const int t = threadIdx.x, l = t & 63, wave = t >> 6;
    const int wn = wave / CS, ch = wave % CS;
    const int a = l & 15, g = l >> 4;
    const int nwg = (int)gridDim.x;
    int wg = blockIdx.x;
    if (nwg % 8 == 0) wg = (wg % 8) * (nwg / 8) + wg / 8;  // row tiles of a weight tile on one XCD
    const int64_t n0 = (int64_t)(wg / A.tiles_m) * BN;
    const int m0 = wg % A.tiles_m * BM;

    if (t == 0) flags[0] = 0;
    __syncthreads();
    {
        int f = 0;
        if (t < BN && n0 + t < A.N) f |= A.wref[n0 + t] != 0;
        if (t < BM && m0 + t < A.M) f |= A.ok[m0 + t] == 0;
        if (f) flags[0] = 1;
    }

    // unit i of this thread: row RT i + t / (2 SB), 16 elements t % (2 SB) of
    // the stage; units past the tile repeat its last row
    const int u = t % (2 * SB), ur = t / (2 * SB);
    const uint8_t* wp[C::WT];
    const int8_t* ap[C::AT];
#pragma unroll
    for (int i = 0; i < C::WT; i++) wp[i] = A.W + min(n0 + min(C::RT * i + ur, BN - 1), A.N - 1) * A.rb;
#pragma unroll
    for (int i = 0; i < C::AT; i++) ap[i] = A.q + (int64_t)min(m0 + min(C::RT * i + ur, BM - 1), A.M - 1) * A.K;
    // the activation scales this thread copies: row t / SB + .., block t % SB
    const int xj = t % SB, xr = t / SB;

    WUnit wu[C::WT];
    u32x4 au[C::AT];
    float xd[C::XT];
    auto load = [&](int s) {
        // past the last block: the last block again, with an activation scale of 0
        const int j = min(SB * s + (u >> 1), A.nblk - 1);
#pragma unroll
        for (int i = 0; i < C::WT; i++) {
            const uint8_t* blk = wp[i] + (int64_t)j * Q80_BYTES;
            const uint8_t* p = blk + 2 + 16 * (u & 1);
            const uint32_t* b = (const uint32_t*)__builtin_align_down(p, 4);
            const u32x4a4 v = *(const u32x4a4*)b;
            wu[i].v[0] = v.x, wu[i].v[1] = v.y, wu[i].v[2] = v.z, wu[i].v[3] = v.w, wu[i].v[4] = b[4];
            wu[i].d = load_u16(blk) | ((uint32_t)((uintptr_t)p & 3) << 16);
        }
#pragma unroll
        for (int i = 0; i < C::AT; i++) au[i] = *(const u32x4*)(ap[i] + (int64_t)j * 32 + 16 * (u & 1));
        // (a scale of 0 leaves every chain as it is: acc is never -0, P finite)
#pragma unroll
        for (int i = 0; i < C::XT; i++) {
            const int m = min(m0 + min(256 / SB * i + xr, BM - 1), A.M - 1);
            const float d = A.d32[(int64_t)m * A.nblk + min(SB * s + xj, A.nblk - 1)];
            xd[i] = SB * s + xj < A.nblk ? d : 0.f;
        }
    };
    auto put = [&](uint8_t* rows, int r, const uint32_t (&v)[4]) {
        const int c = 2 * u;
        const u32x2 e0 = cvt4(v[0]), e1 = cvt4(v[1]), e2 = cvt4(v[2]), e3 = cvt4(v[3]);
        *(u32x4*)(rows + r * C::ROW + 16 * C::slot(c, r)) = u32x4{e0.x, e0.y, e1.x, e1.y};
        *(u32x4*)(rows + r * C::ROW + 16 * C::slot(c + 1, r)) = u32x4{e2.x, e2.y, e3.x, e3.y};
    };
    auto store = [&](int s) {
        uint8_t* wl = smem + (s & 1) * C::BUF;
        uint8_t* al = wl + C::WB;
        float* dl = (float*)(al + C::AB);
#pragma unroll
        for (int i = 0; i < C::WT; i++) {
            const int r = C::RT * i + ur;
            const uint32_t sh = wu[i].d >> 16;
            uint32_t v[4];
#pragma unroll
            for (int k = 0; k < 4; k++) v[k] = __builtin_amdgcn_alignbyte(wu[i].v[k + 1], wu[i].v[k], sh);
            if (C::WU % 256 == 0 || r < BN) {
                put(wl, r, v);
                if ((u & 1) == 0) dl[(u >> 1) * BN + r] = f16_to_f32(wu[i].d & 0xFFFFu);
            }
        }
#pragma unroll
        for (int i = 0; i < C::AT; i++) {
            const int r = C::RT * i + ur;
            const uint32_t v[4] = {au[i].x, au[i].y, au[i].z, au[i].w};
            if (C::AU % 256 == 0 || r < BM) put(al, r, v);
        }
#pragma unroll
        for (int i = 0; i < C::XT; i++) {
            const int r = 256 / SB * i + xr;
            if (BM * SB % 256 == 0 || r < BM) dl[SB * BN + xj * BM + r] = xd[i];
        }
    };

    // acc[mt][h][4 b + r]: chain 2 b + h of (activation row 16 mt + 4 g + r,
    // weight row a); CS = 2: h = ch only
    constexpr int NH = 2 / CS;
    float acc[MT][NH][16];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int h = 0; h < NH; h++)
#pragma unroll
            for (int i = 0; i < 16; i++) acc[mt][h][i] = 0.f;

    const int nst = (A.nblk + SB - 1) / SB;
    load(0);
    store(0);
    load(min(1, nst - 1));
    lds_barrier();
    for (int s = 0; s < nst; s++) {
        const uint8_t* wl = smem + (s & 1) * C::BUF;
        const uint8_t* al = wl + C::WB;
        const float* dl = (const float*)(al + C::AB);
        store(s + 1);
        load(min(s + 2, nst - 1));
        __builtin_amdgcn_sched_barrier(0);  // the loads are not sunk to the end of the stage
        // Steps of one block and one 16-row tile: the operands of step k + 1
        // are read, and its first product issued, before the fmas of step k
        // (pinned, so that two products are live and not all of them).
        struct Ops {
            u32x4 xa, wb;
            f32x4 dx;
            float dw;
        };
        const int wr = 16 * wn + a;
        auto read = [&](int k, Ops& o) {
            const int j = k / MT, r = 16 * (k % MT) + a;
            if (k % MT == 0) {  // chunk 4 j + g of a row: chains 2 g and 2 g + 1
                o.wb = *(const u32x4*)(wl + wr * C::ROW + 16 * C::slot(4 * j + g, wr));
                o.dw = dl[j * BN + wr];
            }
            o.xa = *(const u32x4*)(al + r * C::ROW + 16 * C::slot(4 * j + g, r));
            o.dx = *(const f32x4*)(dl + SB * BN + j * BM + 16 * (k % MT) + 4 * g);
        };
        auto product = [&](const Ops& o, int h) {
            const bool hi = CS == 1 ? h == 1 : ch == 1;
            const h4 av = __builtin_bit_cast(h4, hi ? u32x2{o.xa.z, o.xa.w} : u32x2{o.xa.x, o.xa.y});
            const h4 bv = __builtin_bit_cast(h4, hi ? u32x2{o.wb.z, o.wb.w} : u32x2{o.wb.x, o.wb.y});
            const v16f z = {};
            return __builtin_amdgcn_mfma_f32_16x16x4f16(av, bv, z, 0, 0, 0);
        };
        constexpr int NK = SB * MT;
        Ops o;
        read(0, o);
        v16f P = product(o, 0);
#pragma unroll
        for (int k = 0; k < NK; k++) {
            const int mt = k % MT;
            float dd[4];
#pragma unroll
            for (int r = 0; r < 4; r++) dd[r] = o.dw * o.dx[r];
            v16f Q;
            if constexpr (NH == 2) {
                Q = product(o, 1);
                if (k + 1 < NK) read(k + 1, o);
#pragma unroll
                for (int i = 0; i < 16; i++) acc[mt][0][i] = __builtin_fmaf(P[i], dd[i & 3], acc[mt][0][i]);
                __builtin_amdgcn_sched_barrier(0);
                if (k + 1 < NK) P = product(o, 0);
#pragma unroll
                for (int i = 0; i < 16; i++) acc[mt][1][i] = __builtin_fmaf(Q[i], dd[i & 3], acc[mt][1][i]);
            } else {
                if (k + 1 < NK) {
                    read(k + 1, o);
                    Q = product(o, 0);
                }
#pragma unroll
                for (int i = 0; i < 16; i++) acc[mt][0][i] = __builtin_fmaf(P[i], dd[i & 3], acc[mt][0][i]);
                P = Q;
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        lds_barrier();
    }

    // HSUM1: c_l = a_l + a_{l+4}, (c0 + c1) + (c2 + c3); chain 2 b + h
    const int refused = flags[0];
    const int64_t n = n0 + 16 * wn + a;
    float* ex = (float*)smem;
    float res[MT][4];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            float c[NH][2];
#pragma unroll
            for (int h = 0; h < NH; h++)
#pragma unroll
                for (int b = 0; b < 2; b++) c[h][b] = acc[mt][h][4 * b + r] + acc[mt][h][8 + 4 * b + r];
            if constexpr (CS == 1) {
                res[mt][r] = (c[0][0] + c[1][0]) + (c[0][1] + c[1][1]);
            } else {
                // the wave of h = 1 hands c1 and c3 over
                float2* e = (float2*)ex + ((wn * MT + mt) * 4 + r) * 64 + l;
                if (ch == 1) *e = float2{c[0][0], c[0][1]};
                res[mt][r] = c[0][0];
                acc[mt][0][r] = c[0][1];
            }
        }
    if constexpr (CS == 2) {
        lds_barrier();
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const float2 o = ((const float2*)ex)[((wn * MT + mt) * 4 + r) * 64 + l];
                res[mt][r] = (res[mt][r] + o.x) + (acc[mt][0][r] + o.y);
            }
    }
    if (n < A.N && (CS == 1 || ch == 0) && !(refused && A.wref[n] != 0)) {
        const float bn = A.bias ? A.bias[n] : 0.f;
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int m = m0 + 16 * mt + 4 * g + r;
                if (m >= A.M) continue;
                if (refused && A.ok[m] == 0) continue;
                float v = res[mt][r];
                if (A.bias) v += bn;
                A.y[(int64_t)m * A.N + n] = v;
            }
    }
    if (!refused) return;
    // Refused pairs of the tile: the reference's float32 path.
    for (int pidx = t >> 3; pidx < BN * BM; pidx += 32) {
        const int64_t nn = n0 + pidx % BN;
        const int m = m0 + pidx / BN;
        if (nn >= A.N || m >= A.M) continue;
        if (A.wref[nn] == 0 && A.ok[m] != 0) continue;
        float v = f32dot_g8<DT_Q8_0>(A.W + nn * A.rb, A.x + (int64_t)m * A.K, A.K, A.fused != 0);
        if (A.bias) v += A.bias[nn];
        if ((t & 7) == 0) A.y[(int64_t)m * A.N + nn] = v;
    }
}

template <class C>
static hipError_t launch(Args A, hipStream_t stream) {
    A.tiles_m = (A.M + C::BM - 1) / C::BM;
    const int64_t nwg = (A.N + C::BN - 1) / C::BN * A.tiles_m;
    if (nwg > 0x7fffffff) return hipErrorInvalidValue;
    hipLaunchKernelGGL(gemm_q8_0_kernel<C>, dim3((unsigned)nwg), dim3(256), 0, stream, A);
    return hipGetLastError();
}

}  // namespace b32r

hipError_t launch_gemm_q8_0_ref(const DevWeight& w, const ActPtrs& a, int64_t rows, int64_t total_rows, const float* x,
                                const float* bias, float* y, hipStream_t stream) {
    using namespace b32r;
    if (w.dt != DT_Q8_0 || w.k % 32 || rows <= 0 || rows > (1 << 30) || w.k / 32 > (1 << 30)) return hipErrorInvalidValue;
    Args A;
    A.W = w.data;
    A.wref = w.wref;
    A.bias = bias;
    A.y = y;
    A.rb = w.row_bytes;
    A.K = w.k;
    A.N = w.n;
    A.M = (int)rows;
    A.nblk = (int)(w.k / 32);
    A.q = a.q;
    A.d32 = a.d32;
    A.ok = a.ok;
    A.x = x;
    A.fused = total_rows <= 8;
    A.tiles_m = 1;
    auto wgs = [&](int bn, int bm) { return (w.n + bn - 1) / bn * ((rows + bm - 1) / bm); };
    // the largest tile that gives every CU a workgroup (measured: 4096 x 4096
    // at 64 rows 38 us in 256 tiles of 16 rows, 52 in 64 of 64)
    if (rows > 32 && wgs(64, 64) >= 256) return launch<Cfg<4, 1, 4>>(A, stream);
    if (rows > 16 && wgs(64, 32) >= 256) return launch<Cfg<2, 1, 4>>(A, stream);
    if (wgs(64, 16) >= 256) return launch<Cfg<1, 1, 4>>(A, stream);
    return launch<Cfg<1, 2, 8>>(A, stream);
}

}  // namespace mimg
