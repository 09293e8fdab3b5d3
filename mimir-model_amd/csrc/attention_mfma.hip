// Attention for many query rows on the matrix cores (attention.v1/.v2 in the
// reference's attendRow order, interp/fast.go:728-751 with attn_amd64.s), bit
// for bit: v_mfma_f32_{32x32x1,16x16x1,4x4x1}_f32 adds one product to each
// output as one fused multiply-add (measured equal to fmaf over every value
// class, NaN payloads included), so a chain of them is the reference's chain
// of fmas.
//
// Rows: the G = H / Hkv query heads of a kv head read the same keys and
// values, so a row tile holds rows rho = t * G + g of one kv head; the tiles
// are full at any number of query heads. The launch is two kernels, the
// scores in between in the workspace, [T][H][maxk].
//
// scores_kernel: a wave owns 32 keys (in registers), a workgroup 128 and 32
// rows (in LDS). The reference's eight chains of a score, l_c = fma(q[8m + c],
// k[8m + c], l_c), are four v_mfma_f32_32x32x1_2b a step m: the instruction's
// two blocks hold chains i and 4 + i, lane l giving row (key) l % 32 and
// q[8m + 4 (l/32) + i], one 16-byte read a step. A lane ends with all eight
// chains of 16 (row, key) pairs and adds them as the reference does
// (((l0+l1)+(l2+l3))+((l4+l5)+(l6+l7)) for keys in the groups of four,
// ((l0+l4)+(l1+l5))+((l2+l6)+(l3+l7)) for the last n % 4), times the scale.
//
// wsum_kernel: a workgroup per 2 RT rows; each wave takes RT rows and 64 dims
// and runs acc = fma(e_j, v_j[d], acc) over the keys in order, one
// v_mfma_f32_16x16x1_4b (RT = 16) or 4x4x1_16b (RT = 4) a key: lane l gives
// the weight of row l % RT and the value of dim l, read straight from the
// value cache (16 bytes: eight keys of the dim). The weights of a chunk of keys
// are made by all waves into LDS (double-buffered): Cephes exp of s - max
// for the first n & ~7 keys, the f64 exp for the rest; the eight stride-8 lane
// sums follow them in key order. Keys that only some rows of a wave see keep
// the other rows' sums. Rows with different first keys (several sequences)
// run one first key at a time.
//
// EACH, for calls whose sequences may have few rows each (decode batches of
// many sequences, few query heads a kv head): a 32-row tile of scores and a
// pass over a first key would mostly work for rows that don't see the keys. A
// scores wave whose keys at most eight rows see takes those rows, four at a
// time, on the 4x4x1_16b (an eighth of the matrix time, the same operands);
// wsum has workgroups of four rows, one per first key of the four, which skip
// the weights of rows of other passes. A prompt's waves take the 32-row tile
// as before. These are instances of their own: the branches in the others'
// code cost a prompt 3 to 10 %.
//
// Bound: the matrix cores' f32 rate (measured 18 ns a 16x16x1_4b and 32 ns a
// 32x32x1_2b, 2x the vector unit's fmas) and, in wsum, a wave's serial chain
// over the keys (6.9 ns a key with RT = 4, 18 with 16); below a few hundred
// rows the chain of loads and reductions before the first product.
// Measured on MI355X, us, against a key a lane for the scores and eight chains
// a lane for the sum on the vector unit (32 heads, 8 kv heads, D = 128, f16):
// 512 rows 125 -> 53 (each kernel by itself: scores 65 -> 24, sum 63 -> 32),
// 2000 rows 3197 -> 510, 64 rows 37.7 -> 14.9, 16 rows 16.7 -> 13.9; D = 64: 256
// rows 51 -> 36, 512 rows 93 -> 62 (f16), 94 -> 70 (f32), 1000 rows 346 -> 130;
// there, and with float32 values at D = 128, wsum's 16-row instances spill (33
// registers for D = 64 f16, 73 f32, 11 for D = 128 f32). Loading the next tile's keys ahead in scores_kernel cost a
// wave a SIMD and measured 61 us at 512 rows.
#include <type_traits>

#include "decoder_math.hpp"
#include "mimg_device.hpp"
#include "mimg_kernels.hpp"

namespace mimg {
namespace am {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v32f __attribute__((ext_vector_type(32)));

struct Args {
    const float* q;       // [T][H][D]
    const void *kc, *vc;  // [Hkv][C][D]; blocked by eight keys (vcache_at)
    const int64_t *kend, *kstart;
    int T, H, Hkv, G;
    int64_t C, maxk;
    float* ws;            // [T][H][maxk]
    float* out;           // [T][H][D]
};

__device__ __forceinline__ int wave_min_i32(int v) {
    v = min(v, lane_xor<32>(v));
    v = min(v, lane_xor<16>(v));
    v = min(v, lane_xor<8>(v));
    v = min(v, lane_xor<4>(v));
    v = min(v, lane_xor<2>(v));
    v = min(v, lane_xor<1>(v));
    return __builtin_amdgcn_readfirstlane(v);
}
__device__ __forceinline__ int wave_max_i32(int v) { return -wave_min_i32(-v); }

// Row rho of kv head hk: the keys it sees (none past the last query), and
// t * H + h (past the last query: the last row's). Fewer than 2^32 rows; keys
// below 2^30 (the launcher's rule).
struct Row {
    int k0, n;
    uint32_t head;
};
__device__ __forceinline__ Row row_of(const Args& A, int hk, uint32_t rho) {
    const uint32_t rc = min(rho, (uint32_t)A.T * (uint32_t)A.G - 1), t = rc / (uint32_t)A.G;
    const AttRange a = att_range(A.kend, A.kstart, (int)t, A.C, A.maxk);
    return {(int)a.k0, rc == rho ? (int)a.n : 0, t * (uint32_t)A.H + (uint32_t)(hk * A.G) + (rc - t * (uint32_t)A.G)};
}

constexpr int SROWS = 32, SKEYS = 128;

template <bool F16, int D, bool EACH>
__global__ __launch_bounds__(256, 2) void scores_kernel(Args A) {
    constexpr int DM = D / 8, QS = D + 4;  // a row in LDS, padded by four banks
    __shared__ __align__(16) float qs[SROWS * QS];
    __shared__ int4 rinfo[SROWS];  // first key, keys, workspace offset (two words)
    __shared__ uint32_t rhead[SROWS];
    const int hk = blockIdx.x % (uint32_t)A.Hkv, t = threadIdx.x, l = t & 63, w = t >> 6;
    // the last rows (the most keys of a prompt) first
    const uint32_t rho0 = (gridDim.x / (uint32_t)A.Hkv - 1 - blockIdx.x / (uint32_t)A.Hkv) * SROWS;
    const int a32 = l & 31, g = l >> 5;
    const Row r = row_of(A, hk, rho0 + a32);  // every lane: row l % 32
    // the cache entries the rows see: [kmin, kfin)
    const int kmin = wave_min_i32(r.n > 0 ? r.k0 : 0x7fffffff), kfin = wave_max_i32(r.n > 0 ? r.k0 + r.n : 0);
    const int kt0 = kmin + SKEYS * (int)blockIdx.y;
    if (kfin == 0 || kt0 >= kfin) return;  // uniform in the workgroup
    if (t < SROWS) {
        const uint64_t o = (uint64_t)r.head * (uint64_t)A.maxk;
        rinfo[t] = int4{r.k0, r.n, (int)(uint32_t)o, (int)(uint32_t)(o >> 32)};
        rhead[t] = rho0 + t < (uint32_t)A.T * (uint32_t)A.G ? r.head : 0xFFFFFFFFu;
    }
    lds_barrier();
    for (int i = t; i < SROWS * D / 4; i += 256) {
        const int row = i / (D / 4), d4 = i - row * (D / 4);
        const uint32_t hd = rhead[row];  // rows past the last: zeros
        const float4 v = hd != 0xFFFFFFFFu ? *(const float4*)(A.q + (int64_t)hd * D + 4 * d4) : float4{0.f, 0.f, 0.f, 0.f};
        *(float4*)(qs + row * QS + 4 * d4) = v;
    }
    lds_barrier();
    const float scale = (float)(1.0 / sqrt((double)D));
    for (int kt = kt0; kt < kfin; kt += SKEYS * (int)gridDim.y) {
        const int kb = kt + 32 * w;  // this wave's first key
        // the rows that see any of its keys
        uint32_t seen = (uint32_t)__ballot(r.n > 0 && r.k0 < kb + 32 && r.k0 + r.n > kb);
        if (seen == 0) continue;
        const int a = kb + a32;
        const int64_t ac = a < A.C ? a : A.C - 1;  // past the cache: its last key, unstored
        using KT = typename std::conditional<F16, uint2, float4>::type;
        KT kw[DM];
        const uint8_t* kp = (const uint8_t*)A.kc + (((int64_t)hk * A.C + ac) * D + 4 * g) * (F16 ? 2 : 4);
#pragma unroll
        for (int m = 0; m < DM; m++) kw[m] = *(const KT*)(kp + m * (F16 ? 16 : 32));
        auto key4 = [&](int m, float (&kv)[4]) {
            if constexpr (F16) {
                const uint32_t wd[2] = {kw[m].x, kw[m].y};
#pragma unroll
                for (int i = 0; i < 4; i++)
                    kv[i] = (float)__builtin_bit_cast(_Float16, (uint16_t)((i & 1) ? wd[i / 2] >> 16 : wd[i / 2] & 0xFFFF));
            } else {
                kv[0] = kw[m].x, kv[1] = kw[m].y, kv[2] = kw[m].z, kv[3] = kw[m].w;
            }
        };
        if (EACH && __popc(seen) <= 8) {
            // four rows a turn on the 4x4x1_16b: lane l gives the (l % 4)th
            // row's q and gets all four's chains 4 g + i against its own key
            while (seen) {
                int sel[4], nsel = 0;
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    sel[i] = seen ? __builtin_ctz(seen) : sel[i > 0 ? i - 1 : 0];
                    nsel += seen != 0;
                    seen &= seen - 1;
                }
                const float* qr = qs + (l & 2 ? (l & 1 ? sel[3] : sel[2]) : (l & 1 ? sel[1] : sel[0])) * QS + 4 * g;
                v4f acc[4];
#pragma unroll
                for (int m = 0; m < DM; m++) {
                    const float4 q4 = *(const float4*)(qr + 8 * m);
                    const float qv[4] = {q4.x, q4.y, q4.z, q4.w};
                    float kv[4];
                    key4(m, kv);
                    const v4f z = {};
#pragma unroll
                    for (int i = 0; i < 4; i++) acc[i] = __builtin_amdgcn_mfma_f32_4x4x1f32(qv[i], kv[i], m ? acc[i] : z, 0, 0, 0);
                }
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    if (i >= nsel) break;
                    const int4 ri = rinfo[sel[i]];
                    const int j = a - ri.x, n = ri.y, n4 = n & ~3;
                    const float h = (acc[0][i] + acc[1][i]) + (acc[2][i] + acc[3][i]);
                    float p = h + lane_xor_f32<32>(h);
                    if (__any(j >= n4)) {
                        const float e0 = acc[0][i] + lane_xor_f32<32>(acc[0][i]), e1 = acc[1][i] + lane_xor_f32<32>(acc[1][i]);
                        const float e2 = acc[2][i] + lane_xor_f32<32>(acc[2][i]), e3 = acc[3][i] + lane_xor_f32<32>(acc[3][i]);
                        p = j >= n4 ? (e0 + e1) + (e2 + e3) : p;
                    }
                    if (g == 0 && j >= 0 && j < n)
                        A.ws[(int64_t)(((uint64_t)(uint32_t)ri.w << 32) | (uint32_t)ri.z) + j] = p * scale;
                }
            }
            continue;
        }
        const float* qr = qs + a32 * QS + 4 * g;
        v32f acc[4];
#pragma unroll
        for (int m = 0; m < DM; m++) {
            const float4 q4 = *(const float4*)(qr + 8 * m);
            const float qv[4] = {q4.x, q4.y, q4.z, q4.w};
            float kv[4];
            key4(m, kv);
            const v32f z = {};
#pragma unroll
            for (int i = 0; i < 4; i++) acc[i] = __builtin_amdgcn_mfma_f32_32x32x1f32(qv[i], kv[i], m ? acc[i] : z, 0, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const int row = 8 * (i >> 2) + 4 * g + (i & 3);
            const int4 ri = rinfo[row];
            const int j = a - ri.x, n = ri.y, n4 = n & ~3;
            const float l0 = acc[0][i], l1 = acc[1][i], l2 = acc[2][i], l3 = acc[3][i];
            const float l4 = acc[0][16 + i], l5 = acc[1][16 + i], l6 = acc[2][16 + i], l7 = acc[3][16 + i];
            float p = ((l0 + l1) + (l2 + l3)) + ((l4 + l5) + (l6 + l7));
            if (j >= n4) p = ((l0 + l4) + (l1 + l5)) + ((l2 + l6) + (l3 + l7));
            if (j >= 0 && j < n) A.ws[(int64_t)(((uint64_t)(uint32_t)ri.w << 32) | (uint32_t)ri.z) + j] = p * scale;
        }
    }
}

// RT rows x 64 dims of a wave: the accumulators and where they lie.
template <int RT>
struct Tile;
template <>
struct Tile<16> {
    static constexpr int NA = 16;
    typedef v16f acc_t;
    static __device__ __forceinline__ acc_t step(float e, float v, acc_t c) {
        return __builtin_amdgcn_mfma_f32_16x16x1f32(e, v, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int i, int l) { return 4 * (l >> 4) + (i & 3); }
    static __device__ __forceinline__ int dim(int i, int l) { return 16 * (i >> 2) + (l & 15); }
};
template <>
struct Tile<4> {
    static constexpr int NA = 4;
    typedef v4f acc_t;
    static __device__ __forceinline__ acc_t step(float e, float v, acc_t c) {
        return __builtin_amdgcn_mfma_f32_4x4x1f32(e, v, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int i, int) { return i; }
    static __device__ __forceinline__ int dim(int, int l) { return l; }
};

template <bool F16, int D, int RT, bool EACH>
__global__ __launch_bounds__((EACH ? 1 : 2) * D, 2) void wsum_kernel(Args A) {
    using TL = Tile<RT>;
    constexpr int RG = EACH ? 1 : 2, R = RG * RT, DH = D / 64, NT = RG * D, NW = NT / 64;
    // keys of a chunk (64 for RT = 16: 128 measured the same with 30 more
    // registers); a row's weights in LDS, padded by four banks
    constexpr int KC = RT == 16 ? 64 : D, ES = KC + 4;
    constexpr int EPT = R * KC / NT;              // weights of a chunk per thread
    constexpr int SPT = (R * 8 + NT - 1) / NT;    // lane sums per thread
    constexpr int RPW = R / NW, MU = 32 / RPW;    // rows per wave of the max, loads in flight per row
    // value blocks of a segment (two segments in registers): what a wave's
    // chains cover of a load's latency
    constexpr int HB = RT == 16 ? 4 : KC / (F16 ? 16 : 32), SEG = KC / 8 / HB;  // value blocks of a segment, segments of a chunk
    using VT = typename std::conditional<F16, _Float16, float>::type;
    __shared__ __align__(16) float ew[2][R * ES];
    __shared__ float lsum[R][8], tail[R][8], rsum[R], rmx[R];
    __shared__ uint32_t rhead[R];
    __shared__ int rn[R], rbad[R];
    const int hk = blockIdx.x % (uint32_t)A.Hkv, t = threadIdx.x, l = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
    // the last rows (the most keys of a prompt) first, then the first ones, so
    // that two workgroups of a CU share long and short
    const uint32_t nt = gridDim.x / (uint32_t)A.Hkv, tb = blockIdx.x / (uint32_t)A.Hkv;
    const uint32_t rho0 = (2 * tb < nt ? nt - 1 - tb : tb - (nt + 1) / 2) * R;
    const int dh = w % DH, rg = w / DH, d = 64 * dh + l;  // this lane's dim, this wave's rows
    Row r = row_of(A, hk, rho0 + l % R);  // lane l: row l
    if (l >= R) r.n = 0;
    if (t < R) rhead[t] = r.head;
    const uint32_t rows = (uint32_t)A.T * (uint32_t)A.G;

    uint64_t live = __ballot(r.n > 0);
    // rows that see no key: zeros
    if ((!EACH || blockIdx.y == 0) && (~live & ((1ull << R) - 1))) {
        lds_barrier();
        for (int i = t; i < R * D; i += NT) {
            const int row = i / D;
            if (!((live >> row) & 1) && rho0 + row < rows) A.out[(int64_t)rhead[row] * D + i % D] = 0.f;
        }
    }
    for (uint32_t pass = 0; live; pass++) {
        // the rows that share the first live row's first key
        const int k0 = __builtin_amdgcn_readlane(r.k0, __builtin_ctzll(live));
        const uint64_t in = __ballot(r.n > 0 && r.k0 == k0);
        live &= ~in;
        if (EACH && pass % gridDim.y != blockIdx.y) continue;  // another workgroup's
        const bool mine = (in >> l) & 1;
        const int nl = mine ? r.n : 0;
        const int nall = wave_max_i32(nl);
        const bool wr = mine && l / RT == rg;  // the rows of this wave's chains
        const int nmin = wave_min_i32(wr ? nl : 0x7fffffff), nmax = wave_max_i32(wr ? nl : 0);
        lds_barrier();  // the pass before is done with LDS
        if (t < R) rn[t] = nl;
        lds_barrier();
        // The keys go in chunks of KC from the value block that holds k0: slot
        // s of the chunks is key s - off of the rows. Everything that needs no
        // maximum is loaded first.
        const int off = k0 & 7, kbeg = k0 - off;
        const int nch = (off + nall + KC - 1) / KC, nblk = (off + nall + 7) >> 3;
        // the rows of this thread's weights (uniform in the wave)
        int un[EPT];
        float sv[EPT];
        uint32_t uh[EPT];
#pragma unroll
        for (int u = 0; u < EPT; u++) {
            const int row = (t + NT * u) / KC;
            un[u] = __builtin_amdgcn_readfirstlane(rn[row]);
            uh[u] = __builtin_amdgcn_readfirstlane(rhead[row]);
        }
        const int us = t % KC - off;  // this thread's key of chunk 0
        auto load_scores = [&](int ch) {
#pragma unroll
            for (int u = 0; u < EPT; u++) {
                // past the row's scores: the last one (of no row: its first word), unused
                sv[u] = A.ws[(int64_t)uh[u] * A.maxk + max(min(KC * ch + us, un[u] - 1), 0)];
            }
        };
        uint4 va[HB * (F16 ? 1 : 2)], vb[HB * (F16 ? 1 : 2)];
        auto vload = [&](uint4* v, int sg) {  // segment sg: its HB value blocks (past the last: the last)
#pragma unroll
            for (int i = 0; i < HB; i++) {
                const int b = min(HB * sg + i, nblk - 1);
                const VT* vp = (const VT*)A.vc + vcache_at(hk, (int64_t)kbeg + 8 * b, d, D, A.C);
                if constexpr (F16) {
                    v[i] = *(const uint4*)vp;
                } else {
                    v[2 * i] = ((const uint4*)vp)[0];
                    v[2 * i + 1] = ((const uint4*)vp)[1];
                }
            }
        };
        float tv[SPT];  // the scores of each row's last n % 8 keys: thread 8 row + c
#pragma unroll
        for (int u = 0; u < SPT; u++) {
            const int p = t + NT * u, row = (p >> 3) % R, n = rn[row], j = (n & ~7) + (p & 7);
            tv[u] = A.ws[(int64_t)rhead[row] * A.maxk + max(min(j, n - 1), 0)];
        }
        load_scores(0);
        vload(va, 0);
        // 1. each row's largest score, NaN check (a wave: rows w, w + NW, ..)
        {
            float mx[RPW];
            int bad[RPW];
#pragma unroll
            for (int i = 0; i < RPW; i++) mx[i] = -INFINITY, bad[i] = 0;
            for (int j0 = l; j0 < nall; j0 += 64 * MU) {
                float v[RPW][MU];
#pragma unroll
                for (int i = 0; i < RPW; i++) {
                    const int n = rn[w + NW * i];
                    const float* sr = A.ws + (int64_t)rhead[w + NW * i] * A.maxk;
#pragma unroll
                    for (int u = 0; u < MU; u++) v[i][u] = sr[max(min(j0 + 64 * u, n - 1), 0)];
                }
#pragma unroll
                for (int i = 0; i < RPW; i++)
#pragma unroll
                    for (int u = 0; u < MU; u++) {
                        bad[i] |= v[i][u] != v[i][u];
                        mx[i] = fmaxf(mx[i], v[i][u]);
                    }
            }
#pragma unroll
            for (int i = 0; i < RPW; i++) {
                const float m = wave_max_f32(mx[i]);
                const bool b = __any(bad[i]) || __builtin_isinf(m);
                if (l == 0) {
                    rmx[w + NW * i] = m;
                    rbad[w + NW * i] = b;
                }
            }
        }
        lds_barrier();
        // 2. the exps of the last n % 8 keys
#pragma unroll
        for (int u = 0; u < SPT; u++) {
            const int p = t + NT * u, row = (p >> 3) % R;
            if (p < 8 * R && (p & 7) < rn[row] % 8) tail[row][p & 7] = (float)exp((double)(tv[u] - rmx[row]));
        }
        float um[EPT];
#pragma unroll
        for (int u = 0; u < EPT; u++) um[u] = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(rmx[(t + NT * u) / KC])));
        lds_barrier();
        auto exps = [&](int ch) {
            float* eb = ew[ch & 1] + t % KC;
            const int j = KC * ch + us;
            auto one = [&](int u) {
                const int row = (t + NT * u) / KC, nv = un[u] & ~7;
                const float e = cephes_exp(sv[u] - um[u]), et = tail[row][j & 7];
                eb[row * ES] = (uint32_t)j < (uint32_t)nv ? e : ((uint32_t)j < (uint32_t)un[u] ? et : 0.f);
            };
            if (!EACH || in == (1ull << R) - 1) {
#pragma unroll
                for (int u = 0; u < EPT; u++) {
                    one(u);
                    if (u % 4 == 3) __builtin_amdgcn_sched_barrier(0);  // four exps at a time: registers
                }
                return;
            }
#pragma unroll
            for (int u = 0; u < EPT; u++)
                if (un[u] > 0) one(u);  // rows of other passes: what LDS holds, for sums that are dropped
        };
        float sl[SPT];
#pragma unroll
        for (int u = 0; u < SPT; u++) sl[u] = 0.f;
        int nr[4];  // the counts of this lane's rows
#pragma unroll
        for (int i = 0; i < 4; i++) nr[i] = rn[RT * rg + TL::row(i, l)];
        typename TL::acc_t acc = {};
        auto vget = [&](const uint4* v, int i, int k) -> float {
            if constexpr (F16) {
                const uint32_t x[4] = {v[i].x, v[i].y, v[i].z, v[i].w};
                return (float)__builtin_bit_cast(_Float16, (uint16_t)((k & 1) ? x[k / 2] >> 16 : x[k / 2] & 0xFFFF));
            } else {
                const uint4 y = v[2 * i + k / 4];
                const uint32_t x[4] = {y.x, y.y, y.z, y.w};
                return __uint_as_float(x[k & 3]);
            }
        };
        auto chain = [&](const uint4* v, int ch, int sg) {  // segment sg of the chunk's
            const float* er = ew[ch & 1] + (RT * rg + l % RT) * ES + 8 * HB * sg;
            const int js = KC * ch + 8 * HB * sg - off;
            if (js >= 0 && js + 8 * HB <= nmin) {  // every row of the pass sees the segment
#pragma unroll
                for (int i0 = 0; i0 < HB; i0 += 4) {
                    float4 e4[8];
#pragma unroll
                    for (int i = 0; i < 8; i++)
                        if (i0 + i / 2 < HB) e4[i] = *(const float4*)(er + 8 * i0 + 4 * i);
#pragma unroll
                    for (int i = 0; i < 8; i++) {
                        if (i0 + i / 2 >= HB) break;
                        const float e[4] = {e4[i].x, e4[i].y, e4[i].z, e4[i].w};
#pragma unroll
                        for (int k = 0; k < 4; k++) acc = TL::step(e[k], vget(v, i0 + i / 2, 4 * (i & 1) + k), acc);
                    }
                }
                return;
            }
#pragma unroll
            for (int i = 0; i < HB; i++) {
                const int s0 = KC * ch + 8 * (HB * sg + i), j0 = s0 - off;
                if (j0 >= nmax) break;
                const float4 ea = *(const float4*)(er + 8 * i), eb = *(const float4*)(er + 8 * i + 4);
                const float e[8] = {ea.x, ea.y, ea.z, ea.w, eb.x, eb.y, eb.z, eb.w};
                if (j0 >= 0 && j0 + 8 <= nmin) {
#pragma unroll
                    for (int k = 0; k < 8; k++) acc = TL::step(e[k], vget(v, i, k), acc);
                } else {
#pragma unroll
                    for (int k = 0; k < 8; k++) {
                        if (j0 + k < 0 || j0 + k >= nmax) continue;
                        const typename TL::acc_t nx = TL::step(e[k], vget(v, i, k), acc);
#pragma unroll
                        for (int c = 0; c < TL::NA; c++) acc[c] = j0 + k < nr[c & 3] ? nx[c] : acc[c];
                    }
                }
            }
        };
        exps(0);
        lds_barrier();
        for (int ch = 0; ch < nch; ch++) {
            const bool more = ch + 1 < nch;
            if (more) load_scores(ch + 1);
            // the lane sums: thread 8 row + c, keys j = c mod 8 below n & ~7
#pragma unroll
            for (int u = 0; u < SPT; u++) {
                const int p = t + NT * u;
                if (p < 8 * R) {
                    const int row = p >> 3, c = p & 7, n = rn[row], nv = n & ~7;
                    const int s0 = (c + off) & 7;  // the chain's slots: s0 mod 8
                    const float* eb = ew[ch & 1] + row * ES + s0;
                    float ev[KC / 8];
#pragma unroll
                    for (int i = 0; i < KC / 8; i++) ev[i] = eb[8 * i];
#pragma unroll
                    for (int i = 0; i < KC / 8; i++) {
                        const int j = KC * ch + s0 + 8 * i - off;
                        if (j >= 0 && j < nv) sl[u] = sl[u] + ev[i];
                    }
                }
            }
#pragma unroll 1
            for (int sg = 0; sg < SEG; sg += 2) {
                vload(vb, SEG * ch + sg + 1);
                chain(va, ch, sg);
                vload(va, SEG * ch + sg + 2);
                chain(vb, ch, sg + 1);
            }
            __builtin_amdgcn_sched_barrier(0);
            if (more) exps(ch + 1);
            lds_barrier();
        }
#pragma unroll
        for (int u = 0; u < SPT; u++)
            if (t + NT * u < 8 * R) lsum[(t + NT * u) >> 3][(t + NT * u) & 7] = sl[u];
        lds_barrier();
        if (t < R) {
            const float* s = lsum[t];
            float sum = ((s[0] + s[4]) + (s[1] + s[5])) + ((s[2] + s[6]) + (s[3] + s[7]));
            const int n = rn[t], nv = n & ~7;
            for (int j = nv; j < n; j++) sum = sum + tail[t][j - nv];
            rsum[t] = sum;
        }
        lds_barrier();
#pragma unroll
        for (int i = 0; i < TL::NA; i++) {
            const int row = RT * rg + TL::row(i, l);
            if (!((in >> row) & 1)) continue;
            A.out[(int64_t)rhead[row] * D + 64 * dh + TL::dim(i, l)] = rbad[row] ? __builtin_nanf("") : acc[i] / rsum[row];
        }
    }
}

// Scores of few queries (decode), a wave per (64 keys, kv head, query): a key
// per lane, the query heads of the kv head in fours, one v_mfma_f32_4x4x1_16b
// a dim: lane l gives head l % 4's q and its own key's element and gets the
// chains of four heads against its key. The keys come through LDS (16-byte
// pieces, XOR-swizzled by key), so that global memory is read in whole lines.
// Bound: the key bytes (33 MB at 8 queries x 8 kv heads x 2048 keys, f16).
// Measured on MI355X, us, the whole attention, against a workgroup per 64 keys
// with eight lanes a key on the vector unit: that size 33.9 -> 32.4; 64 heads
// of 8 kv heads, 300 keys 23.2 -> 20.5; 24 of 4, D = 64, 2000 keys 22.8 -> 19.6.

template <bool F16, int D, int NG>
__global__ __launch_bounds__(64) void decode_scores_kernel(Args A) {
    constexpr int DM = D / 8, PC = D * (F16 ? 2 : 4) / 16, QS = D + 4;  // pieces of a key; a q row in LDS
    __shared__ __align__(16) uint8_t keys[64 * PC * 16];
    __shared__ __align__(16) float qs[4 * NG * QS];
    const int hk = blockIdx.y, t = blockIdx.z, l = threadIdx.x, j0 = 64 * blockIdx.x;
    const AttRange r = att_range(A.kend, A.kstart, t, A.C, A.maxk);
    const int n = (int)r.n;
    if (j0 >= n) return;
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)keys);
    const uint8_t* kb = (const uint8_t*)A.kc + ((int64_t)hk * A.C + r.k0) * (16 * PC);
#pragma unroll
    for (int i = 0; i < PC; i++) {  // keys past the last: the last one, unstored
        const int c = 64 * i + l, k = c / PC, p = (c % PC) ^ (k & (PC - 1) & 15);
        lds_copy16(kb + (int64_t)min(j0 + k, n - 1) * (16 * PC) + 16 * p, lds0 + 1024 * i);
    }
    const int64_t head0 = (int64_t)t * A.H + (int64_t)hk * A.G;
    for (int i = l; i < 4 * NG * (D / 4); i += 64) {  // heads past the group's: the last one, unstored
        const int g = i / (D / 4), d4 = i % (D / 4);
        *(float4*)(qs + g * QS + 4 * d4) = *(const float4*)(A.q + (head0 + min(g, A.G - 1)) * D + 4 * d4);
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the copies have landed
    asm volatile("" ::: "memory");
    v4f acc[NG][8];
#pragma unroll
    for (int m = 0; m < DM; m++) {
        float kv[8];
        const uint8_t* kr = keys + l * (16 * PC);
        if constexpr (F16) {
            const uint4 w = *(const uint4*)(kr + 16 * (m ^ (l & (PC - 1) & 15)));
            const uint32_t x[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
            for (int c = 0; c < 8; c++)
                kv[c] = (float)__builtin_bit_cast(_Float16, (uint16_t)((c & 1) ? x[c / 2] >> 16 : x[c / 2] & 0xFFFF));
        } else {
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const float4 w = *(const float4*)(kr + 16 * ((2 * m + h) ^ (l & (PC - 1) & 15)));
                kv[4 * h] = w.x, kv[4 * h + 1] = w.y, kv[4 * h + 2] = w.z, kv[4 * h + 3] = w.w;
            }
        }
#pragma unroll
        for (int g = 0; g < NG; g++) {
            const float* qr = qs + (4 * g + (l & 3)) * QS + 8 * m;
            const float4 qa = *(const float4*)qr, qb = *(const float4*)(qr + 4);
            const float qv[8] = {qa.x, qa.y, qa.z, qa.w, qb.x, qb.y, qb.z, qb.w};
            const v4f z = {};
#pragma unroll
            for (int c = 0; c < 8; c++) acc[g][c] = __builtin_amdgcn_mfma_f32_4x4x1f32(qv[c], kv[c], m ? acc[g][c] : z, 0, 0, 0);
        }
    }
    const float scale = (float)(1.0 / sqrt((double)D));
    const int j = j0 + l;
    if (j >= n) return;
    const bool four = j < (n & ~3);
#pragma unroll
    for (int g = 0; g < NG; g++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            if (4 * g + i >= A.G) break;
            const float l0 = acc[g][0][i], l1 = acc[g][1][i], l2 = acc[g][2][i], l3 = acc[g][3][i];
            const float l4 = acc[g][4][i], l5 = acc[g][5][i], l6 = acc[g][6][i], l7 = acc[g][7][i];
            const float pf = ((l0 + l1) + (l2 + l3)) + ((l4 + l5) + (l6 + l7));
            const float pn = ((l0 + l4) + (l1 + l5)) + ((l2 + l6) + (l3 + l7));
            A.ws[(head0 + 4 * g + i) * A.maxk + j] = (four ? pf : pn) * scale;
        }
}

template <bool F16, int D>
static hipError_t launch_decode_scores(const Args& A, hipStream_t s) {
    const dim3 grid((unsigned)((A.maxk + 63) / 64), (unsigned)A.Hkv, (unsigned)A.T);
    if (A.G <= 4) hipLaunchKernelGGL((decode_scores_kernel<F16, D, 1>), grid, dim3(64), 0, s, A);
    else hipLaunchKernelGGL((decode_scores_kernel<F16, D, 2>), grid, dim3(64), 0, s, A);
    return hipGetLastError();
}

template <bool F16, int D>
static hipError_t launch(const Args& A, hipStream_t s) {
    const int64_t rows = (int64_t)A.T * A.G, xt = (rows + SROWS - 1) / SROWS * A.Hkv;
    // key tiles: those the rows can see (several sequences: the whole cache),
    // walked by as many workgroups as give about four a CU
    const int64_t kt = ((A.kstart ? A.C : A.maxk) + SKEYS - 1) / SKEYS, yt = 1024 / xt;
    const dim3 g1((unsigned)xt, (unsigned)(yt < 1 ? 1 : (yt < kt ? yt : kt)));
    // Up to four rows (query, head) a sequence on average (the cache holds
    // C / maxk sequences): EACH. Measured on MI355X, f16, us, with it / without /
    // on the vector unit, a query a sequence: 32 heads of 32 kv heads, D = 128,
    // 16 sequences of 700 keys 52 / 175 / 112, 64 of 700 176 / 305 / 213, 128 of
    // 64 58 / 85 / 46; D = 64, 64 of 700 92 / 267 / 158; 16 kv heads 95 / 167 /
    // 181 (64 of 700); 8 kv heads 58 / 78 / 160; 4 kv heads (eight rows a
    // sequence) 53 / 47 / 158. Two queries a sequence of 700 keys, 64 sequences,
    // D = 64, 32 kv heads 98 / 211 / 175, 16 61 / 107 / 162; four queries, 16
    // sequences, 32 kv heads 43 / 71 / 68, 16 (eight rows) 41 / 39 / 69. A prompt
    // of 64 rows in a cache of 64 sequences 16.8 / 16.1 / 32.5.
    if (A.kstart && A.G <= 4 && (int64_t)A.T * A.G * A.maxk <= 4 * A.C) {
        hipLaunchKernelGGL((scores_kernel<F16, D, true>), g1, dim3(256), 0, s, A);
        // four rows are of at most (G + 2) / G + 1 queries, each with its first key
        const dim3 g2((unsigned)((rows + 3) / 4 * A.Hkv), (unsigned)((A.G + 2) / A.G + 1));
        hipLaunchKernelGGL((wsum_kernel<F16, D, 4, true>), g2, dim3(D), 0, s, A);
        return hipGetLastError();
    }
    hipLaunchKernelGGL((scores_kernel<F16, D, false>), g1, dim3(256), 0, s, A);
    // 16 rows a wave where that gives every CU a workgroup, else four (a
    // quarter of the rows a workgroup, and a key of the chain in 6.9 ns, not
    // 18). The line was measured at D = 128 f16; at D = 64, whose 16-row
    // instances spill, 181 rows of 32 heads (four) take 18 us and 256 (16) 36.
    const int64_t wt = (rows + 31) / 32 * A.Hkv;
    if (wt >= 256) hipLaunchKernelGGL((wsum_kernel<F16, D, 16, false>), dim3((unsigned)wt), dim3(2 * D), 0, s, A);
    else hipLaunchKernelGGL((wsum_kernel<F16, D, 4, false>), dim3((unsigned)((rows + 7) / 8 * A.Hkv)), dim3(2 * D), 0, s, A);
    return hipGetLastError();
}

}  // namespace am

static am::Args am_args(const float* q, const void* kc, const void* vc, const int64_t* kend, const int64_t* kstart,
                        int T, int H, int Hkv, int64_t C, int64_t maxk, float* out, float* ws) {
    am::Args A;
    A.q = q;
    A.kc = kc;
    A.vc = vc;
    A.kend = kend;
    A.kstart = kstart;
    A.T = T;
    A.H = H;
    A.Hkv = Hkv;
    A.G = H / Hkv;
    A.C = C;
    A.maxk = maxk;
    A.ws = ws;
    A.out = out;
    return A;
}

hipError_t launch_attention_mfma(const float* q, const void* kc, const void* vc, const int64_t* kend,
                                 const int64_t* kstart, int T, int H, int Hkv, int D, int64_t C, int64_t maxk, int f16,
                                 float* out, float* ws, hipStream_t s) {
    const am::Args A = am_args(q, kc, vc, kend, kstart, T, H, Hkv, C, maxk, out, ws);
    if (D == 128) return f16 ? am::launch<true, 128>(A, s) : am::launch<false, 128>(A, s);
    if (D == 64) return f16 ? am::launch<true, 64>(A, s) : am::launch<false, 64>(A, s);
    return hipErrorInvalidValue;
}

hipError_t launch_att_scores_mfma(const float* q, const void* kc, const int64_t* kend, const int64_t* kstart, int T, int H,
                                  int Hkv, int D, int64_t C, int64_t maxk, int f16, float* ws, hipStream_t s) {
    const am::Args A = am_args(q, kc, nullptr, kend, kstart, T, H, Hkv, C, maxk, nullptr, ws);
    if (A.G > 8) return hipErrorInvalidValue;
    if (D == 128) return f16 ? am::launch_decode_scores<true, 128>(A, s) : am::launch_decode_scores<false, 128>(A, s);
    if (D == 64) return f16 ? am::launch_decode_scores<true, 64>(A, s) : am::launch_decode_scores<false, 64>(A, s);
    return hipErrorInvalidValue;
}

}  // namespace mimg
