// Dequant GEMM for large batches (q4t_matmat / q4tp_matmat with b > 16,
// qtensor.rs:5830-5960 / 5422-5680, and the prefill's dense contractions):
// Y[b][n] = sum_k X[b][k] W[n][k] for b < M (any M), W in the q4t / q4tp
// device layout of the GEMV kernels.
//
// Tiling (MFMA f32 32x32x16 f16): a workgroup of 4 waves owns 64 batch rows
// x 128 RN weight rows (wave w holds 32 RN of them) and walks K in stages of
// two tiles (64 columns):
//   - a stage's operand (hi / lo f16 planes of 64 rows, 16 KiB) goes straight
//     from global memory into one of three LDS slots, two stages ahead;
//   - the weights and scales of the next group of four tiles are requested
//     into registers a group ahead, each wave its own rows;
//   - the nibbles become the f16 integers n - 8 (dq_signed), so a tile needs
//     no bias; a block of 32 x 32 outputs takes four MFMAs per tile, the lo
//     plane's two and then the hi plane's two in one f32 accumulator started
//     at zero; the tile scale multiplies the sum in f32 as q4t_row_exact does
//     (qtensor.rs:4418-4432).  The lo sum is exact; each of the two hi MFMAs
//     rounds the whole to 24 bits, where an exact accumulator per plane and an
//     add rounded once.  That is the price of the shared accumulator: relative
//     L2 from an f64 product 2.952e-7 -> 2.958e-7 at 512x512 m = 17, 3.123e-7
//     -> 3.127e-7 at 2048x1024 m = 200, 0.05 to 0.2 % more wherever K has as
//     many parts as before (3.78e-7 -> 3.73e-7 at 1024x4096 m = 200, which
//     has more).
// Bound by issue: per tile and block 4 MFMAs (128 cycles of the matrix
// pipe) stand beside 16 FMAs (the tile scale) and 9 VALU ops that unpack
// weights (100 cycles), and the clock falls to ~1.85 GHz under this load.
// Measured on MI355X (the GEMM and the sum of its parts): q4t 12288x4096 m =
// 2048 604 -> 381 us, 6144x1024 106 -> 70, 1024x3072 64 -> 49, 12288x4096 m =
// 256 110 -> 77, m = 64 48 -> 34; q4tp 12288x4096 m = 2048 947 -> 395 (the
// 16x16x32 form with an accumulator per plane and tile biases from LDS took
// 8 FMAs and adds per two MFMAs, and as many LDS as matrix cycles).
#include <mutex>
#include <set>

#include "gemv_kern.h"
#include "runtime.h"

namespace cmf {

struct GemmArgs {
    const void* w;        // [rb][group of 4 tiles][lane][16 B]   (q8: [rb][64-column chunk][lane][16 B])
    const void* scale;    // q4t f16 [rb][group][16][4]; q4tp u32 codes; q8 f32 row scales
    const float2* rowp;   // q4tp (2^lo, 2^step) per row
    const uint8_t* planes;  // hi [item][Mp], lo [item][Mp] (16 B) (q8: q0 q1 q2 [item][Mp])
    const float* xs;      // [Mp] 2^-e per batch row (q8: amax / 127)
    float* y;
    int ldy, M, Mp, N, ntg, nrb, resid;
    // split K: workgroup z takes K steps [z gsteps, (z + 1) gsteps) and
    // writes its partial sums to part [z][M][N] (part == nullptr: one part,
    // y written directly)
    int gsteps;
    float* part;
    // grouped (MoE experts): batch tile y holds tiles[y].y <= 64 rows of
    // expert tiles[y].x, whose weight is desc[tiles[y].x] (tiles == nullptr:
    // one weight for all rows)
    const int2* tiles;
    const GemvDesc* desc;
};

constexpr int G4_NB = 3;           // k_gemm_q4: operand stages in LDS
constexpr size_t GEMM_AT_BYTES = (size_t)G4_NB * 16 * 1024;  // its dynamic LDS
constexpr int GB = 64;             // batch rows per workgroup

// s_waitcnt lgkmcnt(0) + s_barrier: an LDS-only workgroup barrier (the
// weight loads in flight are not waited for, as __syncthreads would)
__device__ __forceinline__ void lds_sync() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

typedef float float16v __attribute__((ext_vector_type(16)));
typedef uint32_t uint4r __attribute__((ext_vector_type(4)));

// Four nibble bytes as the f16 integers n - 8, in-slot order
// {0,4,2,6,1,5,3,7}: a nibble or-ed into 1024.0's mantissa is 1024 + n (low
// nibble of a byte) or 1024 + 16 n (high nibble); both become n - 8 exactly
// by one packed f16 op.
__device__ __forceinline__ half8 dq_signed(uint32_t w) {
    constexpr uint32_t LO = 0x000F000Fu, HI = 0x00F000F0u, M = 0x64006400u;
    const half2v k1 = {(_Float16)-1032.f, (_Float16)-1032.f}, k2 = {(_Float16)0.0625f, (_Float16)0.0625f},
                 k3 = {(_Float16)-72.f, (_Float16)-72.f};
    const uint32_t w8 = w >> 8;
    auto mo = [](uint32_t x, uint32_t mask) __attribute__((always_inline)) {
        uint32_t y;  // (x & mask) | M, one instruction: the mask an SGPR, M a VGPR
        asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(y) : "v"(x), "s"(mask), "v"(M));
        return __builtin_bit_cast(half2v, y);
    };
    const half2v a = mo(w, LO) + k1;    // elements 0, 4
    const half2v b = mo(w8, LO) + k1;   // 2, 6
    const half2v c = __builtin_elementwise_fma(mo(w, HI), k2, k3);   // 1, 5
    const half2v d = __builtin_elementwise_fma(mo(w8, HI), k2, k3);  // 3, 7
    return half8{a.x, a.y, b.x, b.y, c.x, c.y, d.x, d.y};
}

// RN: 32-row weight blocks per wave.
template <int FMT, int RN>
__global__ __launch_bounds__(256, 2) void k_gemm_q4(GemmArgs a) {
    constexpr bool TP = FMT == DT_Q4TP;
    constexpr int MB = 2, BM = GB;  // 32-row batch blocks, batch rows per workgroup
    constexpr int TPS = 2;          // tiles per stage (a stage's operand: 16 KiB)
    constexpr int SPG = 4 / TPS;    // stages per group of 4 tiles
    constexpr int NB = G4_NB;       // operand stages in LDS
    constexpr int NCH = 4;         // 1 KiB operand chunks per wave and stage
    constexpr int NW = 3 * RN;     // weight and scale loads per group
    // the operand ring [NB][plane][4 TPS items][BM rows] x 16 B, filled by
    // direct global -> LDS loads (dynamic LDS: with a static array as the
    // load target the compiler waits for every load in flight before each
    // LDS read)
    extern __shared__ __align__(16) uint4 gemm_at[];
    if (a.tiles) {  // (uniform)
        const int2 t = a.tiles[blockIdx.y];
        if (t.y == 0) return;
        const GemvDesc d = a.desc[t.x];
        a.w = d.w;
        a.scale = d.scale;
        a.rowp = d.rowp;
        a.M = GB * (int)blockIdx.y + t.y;
    }
    // q4tp: the 32 rungs of every row, rung c of row i in word c ^ (i % 32)
    // (rows' equal rungs in different banks)
    __shared__ float lad[TP ? 4 * RN * 32 * 32 : 1];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int c32 = lane & 31, h = lane >> 5, r = lane & 15, rsel = (lane >> 4) & 1;
    const int by = blockIdx.y, rbw = (blockIdx.x * 4 + wave) * 2 * RN;  // first 16-row block of this wave
    const int ntg = a.ntg, Mp = a.Mp;
    const size_t items = (size_t)ntg * 16;  // operand items (4 per tile)
    const int gs0 = blockIdx.z * a.gsteps, gs1 = min(ntg, gs0 + a.gsteps);  // this part's K steps

    // the 16-byte words of group g: lane -> weight row (block 2 q + rsel, row
    // r), k-slots h and 2 + h of its four tiles; blocks past the matrix
    // repeat the last one
    const uint4* wp[RN];
    const uint8_t* sp[RN];
#pragma unroll
    for (int q = 0; q < RN; q++) {
        const size_t t = (size_t)min(rbw + 2 * q + rsel, a.nrb - 1) * ntg;
        wp[q] = (const uint4*)a.w + t * 64 + 16 * h + r;
        sp[q] = (const uint8_t*)a.scale + (t * 16 + r) * (TP ? 4 : 8);
    }
    auto load_w = [&](uint4 (*wv)[2], uint2* sv, int g) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < RN; q++) {
            wv[q][0] = wp[q][(size_t)g * 64];
            wv[q][1] = wp[q][(size_t)g * 64 + 32];
            if constexpr (TP) sv[q].x = *(const uint32_t*)(sp[q] + (size_t)g * 64);
            else sv[q] = *(const uint2*)(sp[q] + (size_t)g * 128);
        }
    };
    // the operand of stage i (of the whole K: tiles TPS i ..) into ring slot
    // buf: chunk c = plane, item, 64 rows
    auto dma = [&](int i, int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < NCH; j++) {
            const int c = wave * NCH + j;
            const int rh = c % (BM / 64), it = (c / (BM / 64)) % (4 * TPS), pl = c / (4 * TPS * (BM / 64));
            const uint4* src = (const uint4*)a.planes +
                               ((size_t)pl * items + 4 * TPS * i + it) * Mp + BM * by + 64 * rh + lane;
            uint4* dst = gemm_at + ((size_t)buf * 8 * TPS + pl * 4 * TPS + it) * BM + 64 * rh;
            __builtin_amdgcn_global_load_lds((const void*)src, (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
        }
    };
    const int i0 = gs0 * SPG, i1 = gs1 * SPG;  // stages
    uint4 wv[RN][2];
    uint2 sv[RN];
#pragma unroll
    for (int k = 0; k < NB - 1; k++) dma(min(i0 + k, i1 - 1), (i0 + k) % NB);
    load_w(wv, sv, gs0);
    if constexpr (TP) {  // 32-rung ladders of the wave's rows (quant.rs:399-410)
#pragma unroll
        for (int q = 0; q < RN; q++) {
            if (h == 0) {
                const float2 p = a.rowp[min(rbw + 2 * q + rsel, a.nrb - 1) * 16 + r];
                float* row = lad + ((wave * RN + q) * 32 + c32) * 32;
                float tv = p.x;
                row[c32] = tv;
                for (int c = 1; c < 32; c++) {
                    tv = tv * p.y;
                    row[c ^ c32] = tv;
                }
            }
        }
    }
    float16v acc[RN][MB];
#pragma unroll
    for (int q = 0; q < RN; q++)
#pragma unroll
        for (int mb = 0; mb < MB; mb++) acc[q][mb] = float16v{};
    wait_vmcnt<0>();
    __syncthreads();

    // tile tt of a group (its words and scales in registers): the weights of
    // 32-row block q, k half j, and its scale
    auto wword = [&](const uint4& w4, int tt) __attribute__((always_inline)) -> uint32_t {
        return tt == 0 ? w4.x : tt == 1 ? w4.y : tt == 2 ? w4.z : w4.w;
    };
    auto tscale = [&](const uint2& s2, int tt, int q) __attribute__((always_inline)) -> float {
        float f;
        if constexpr (TP) {
            f = lad[((wave * RN + q) * 32 + c32) * 32 + (((s2.x >> (5 * tt)) & 31) ^ c32)];
        } else {
            const uint32_t u = tt < 2 ? s2.x : s2.y;
            f = f16_bits_to_f32((tt & 1) == 0 ? u & 0xffffu : u >> 16);
        }
        asm("" : "+v"(f));  // (an f32 register: plain FMAs)
        return f;
    };
    half8 bw[2][RN][2];
    float sc[2][RN];
#pragma unroll
    for (int q = 0; q < RN; q++) {
        sc[0][q] = tscale(sv[q], 0, q);
#pragma unroll
        for (int j = 0; j < 2; j++) bw[0][q][j] = dq_signed(wword(wv[q][j], 0));
    }
#pragma unroll
    for (int q = 0; q < RN; q++) sc[1][q] = 0.f;
    float16v d[2] = {};
    // Stage i: the operand of stage i + NB - 1 goes out (into the slot that
    // stage i - 1 has left), in a group's first stage also the next group's
    // weights, then stage i's MFMAs; the wait covers stage i + 1's operand
    // and leaves the loads issued after it in flight.  Past the last stage
    // the loads repeat it into slots no one reads.
    // The outputs go in blocks of 32 x 32; a block's four MFMAs (lo then hi,
    // one accumulator) run while the block before it is scaled into its f32
    // sums, the next operand rows are read and the next tile's weights
    // unpacked, some of that beside each MFMA (the scheduling barriers keep
    // the compiler from moving it in front of them).
    constexpr int NBLK = TPS * MB * RN;
    for (int g = gs0; g < gs1; g++) {
        uint4 wn[RN][2];
        uint2 sn[RN];
#pragma unroll
        for (int st = 0; st < SPG; st++) {
            const int i = g * SPG + st;
            const uint4* A = gemm_at + (size_t)(i % NB) * 8 * TPS * BM + h * BM + c32;
            // operand fragment k (lo0, lo1, hi0, hi1) of rows mb, tile t
            auto frag = [&](int t, int mb, int k) __attribute__((always_inline)) {
                return __builtin_bit_cast(half8, A[(4 * t + 2 * (k & 1) + (k < 2 ? 4 * TPS : 0)) * BM + 32 * mb]);
            };
            half8 xa[2][4];
#pragma unroll
            for (int k = 0; k < 4; k++) xa[0][k] = frag(0, 0, k);
            dma(min(i + NB - 1, i1 - 1), (i + NB - 1) % NB);
            // (the wait below counts the weights as issued after the operand)
            __builtin_amdgcn_sched_barrier(0);
            if (st == 0) load_w(wn, sn, min(g + 1, gs1 - 1));
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int n = 0; n < NBLK; n++) {
                const int q = n % RN, mb = (n / RN) % MB, t = n / (RN * MB), tt = TPS * st + t;
                // the block before (n = 0: the last of the stage before)
                const int np = n + NBLK - 1, pq = np % RN, pm = (np / RN) % MB, pt = tt - (n % (RN * MB) == 0);
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    d[n & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
                        xa[(n / RN) & 1][k], bw[tt & 1][q][k & 1], k == 0 ? float16v{} : d[n & 1], 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                    // the next rows' fragments, during the last block of these
                    const int e = n / RN + 1;
                    if (q == RN - 1 && e < TPS * MB) xa[e & 1][k] = frag(e / MB, e % MB, k);
                    // the next tile's weight words, one per block, then its scales
                    const int bi = n % (RN * MB), sq = bi - RN * MB + RN;
                    if (k == 0 && bi < 2 * RN)
                        bw[(tt + 1) & 1][bi / 2][bi & 1] =
                            dq_signed(tt < 3 ? wword(wv[bi / 2][bi & 1], tt + 1) : wword(wn[bi / 2][bi & 1], 0));
                    if (k == 3 && sq >= 0)
                        sc[(tt + 1) & 1][sq] = tt < 3 ? tscale(sv[sq], tt + 1, sq) : tscale(sn[sq], 0, sq);
                    if (k > 0) {
                        const int v0 = k == 1 ? 0 : k == 2 ? 5 : 10, v1 = k == 1 ? 5 : k == 2 ? 10 : 16;
#pragma unroll
                        for (int v = 0; v < 16; v++)
                            if (v >= v0 && v < v1)
                                acc[pq][pm][v] = fmaf(d[np & 1][v], sc[pt & 1][pq], acc[pq][pm][v]);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            // loads issued after stage i + 1's operand: the NB - 2 stages
            // after it and one group's weights
            wait_vmcnt<(NB - 2) * NCH + NW>();
            lds_sync();
        }
#pragma unroll
        for (int q = 0; q < RN; q++) {
            wv[q][0] = wn[q][0];
            wv[q][1] = wn[q][1];
            sv[q] = sn[q];
        }
    }
    wait_vmcnt<0>();  // (no load into this workgroup's LDS outlives it)
#pragma unroll
    for (int v = 0; v < 16; v++)  // the last block (tile 3 of a group)
        acc[RN - 1][MB - 1][v] = fmaf(d[(NBLK - 1) & 1][v], sc[1][RN - 1], acc[RN - 1][MB - 1][v]);
#pragma unroll
    for (int q = 0; q < RN; q++) {
        const int n = (rbw + 2 * q) * 16 + c32;
        if (n >= a.N) continue;
#pragma unroll
        for (int mb = 0; mb < MB; mb++)
#pragma unroll
            for (int v = 0; v < 16; v++) {
                const int b = BM * by + 32 * mb + 8 * (v >> 2) + 4 * h + (v & 3);
                if (b < a.M) {
                    const float val = acc[q][mb][v] * a.xs[b];
                    if (a.part) {
                        a.part[((size_t)blockIdx.z * a.M + b) * a.N + n] = val;
                    } else {
                        float* yp = a.y + (size_t)b * a.ldy + n;
                        *yp = a.resid ? *yp + val : val;
                    }
                }
            }
    }
}

// ---------------------------------------------------------------------------
// q8 (qmatvec's exact arm in batches, qtensor.rs:9980-10047): int8 weights
// times the operand carried as three int8 planes x ~= sx (q0 + q1/128 +
// q2/16384) (prep8_row), on v_mfma_i32_16x16x64_i8.  A workgroup of 4 waves
// owns 64 batch rows x 64 Q8RB weight rows and walks K in steps of two
// 64-column chunks: the step's operand (3 planes x 2 chunks x 64 rows x
// 64 B = 24 KiB) is staged one step ahead through registers into a
// double-buffered LDS tile, the next step's weights are requested before the
// current MFMAs.  Each plane keeps its own int32 accumulators over the whole
// K (exact: |sum| <= 127 * 127 * K < 2^31 for K <= 16384), combined in f32
// at the end as the GEMV does: ((s0 + s1/128 + s2/16384) * sx) * rs.
// ---------------------------------------------------------------------------
constexpr int Q8CH = 24;              // 1 KiB operand chunks per step
constexpr int Q8J = Q8CH / 4;         // per wave
constexpr size_t GEMM_Q8_AT_BYTES = (size_t)2 * Q8CH * 64 * 16;  // k_gemm_q8's dynamic LDS
template <int Q8RB>
__global__ __launch_bounds__(256) void k_gemm_q8(GemmArgs a) {
    // double-buffered operand tile [2][Q8CH chunks][64 lanes] x 16 B, filled
    // by direct global -> LDS loads (as k_gemm_q4)
    extern __shared__ __align__(16) int4v gemm_at8[];
    if (a.tiles) {  // (uniform)
        const int2 t = a.tiles[blockIdx.y];
        if (t.y == 0) return;
        const GemvDesc d = a.desc[t.x];
        a.w = d.w;
        a.scale = d.scale;
        a.rowp = d.rowp;
        a.M = GB * (int)blockIdx.y + t.y;
    }
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15, s = lane >> 4;
    const int by = blockIdx.y, rbw = (blockIdx.x * 4 + wave) * Q8RB;
    const int nk = a.ntg, Mp = a.Mp;
    const int4v* P = (const int4v*)a.planes;  // plane p, item (kc * 4 + s): P[(p * nk * 4 + item) * Mp + row]
    // operand chunk c of step g: plane c / 8, chunk 2g + (c / 4) % 2, quarter c % 4
    auto src_a = [&](int j, int g) __attribute__((always_inline)) -> const int4v* {
        const int c = wave + 4 * j;
        const int p = c >> 3, kc = min(2 * g + ((c >> 2) & 1), nk - 1), q = c & 3;
        return P + ((size_t)p * nk * 4 + kc * 4 + q) * Mp + GB * by + lane;
    };
    auto load_w = [&](int4v (*wv)[2], int g) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < Q8RB; q++)
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const size_t t = (size_t)min(rbw + q, a.nrb - 1) * nk + min(2 * g + h, nk - 1);
                wv[q][h] = ld_stream((const int4v*)a.w + t * 64 + lane);
            }
    };
    int4v acc[Q8RB][4][3];
#pragma unroll
    for (int q = 0; q < Q8RB; q++)
#pragma unroll
        for (int mb = 0; mb < 4; mb++)
#pragma unroll
            for (int p = 0; p < 3; p++) acc[q][mb][p] = int4v{0, 0, 0, 0};
    int4v wA[Q8RB][2], wB[Q8RB][2];
    const int nst = (nk + 1) / 2;
    const int gs0 = blockIdx.z * a.gsteps, gs1 = min(nst, gs0 + a.gsteps);  // this part's K steps
    auto dma_a = [&](int g, int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < Q8J; j++) {
            int4v* dst = gemm_at8 + ((size_t)buf * Q8CH + wave + 4 * j) * 64;
            __builtin_amdgcn_global_load_lds((const void*)src_a(j, g), (__attribute__((address_space(3))) void*)dst,
                                             16, 0, 0);
        }
    };
    dma_a(gs0, 0);
    load_w(wA, gs0);
    wait_vmcnt<0>();
    __syncthreads();

    auto compute = [&](int buf, int4v (*wv)[2], int g) __attribute__((always_inline)) {
        const int4v* A = gemm_at8 + (size_t)buf * Q8CH * 64;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            if (2 * g + h >= nk) break;  // uniform: an odd chunk count's last step
#pragma unroll
            for (int mb = 0; mb < 4; mb++) {
                const int4v x0 = A[(0 * 8 + h * 4 + s) * 64 + 16 * mb + r];
                const int4v x1 = A[(1 * 8 + h * 4 + s) * 64 + 16 * mb + r];
                const int4v x2 = A[(2 * 8 + h * 4 + s) * 64 + 16 * mb + r];
#pragma unroll
                for (int q = 0; q < Q8RB; q++) {
                    acc[q][mb][0] = __builtin_amdgcn_mfma_i32_16x16x64_i8(x0, wv[q][h], acc[q][mb][0], 0, 0, 0);
                    acc[q][mb][1] = __builtin_amdgcn_mfma_i32_16x16x64_i8(x1, wv[q][h], acc[q][mb][1], 0, 0, 0);
                    acc[q][mb][2] = __builtin_amdgcn_mfma_i32_16x16x64_i8(x2, wv[q][h], acc[q][mb][2], 0, 0, 0);
                }
            }
        }
    };
    // as k_gemm_q4: the next step's operand straight into the other buffer,
    // a wait for those loads only, an LDS-only barrier
    for (int g = gs0; g < gs1; g += 2) {
        {
            const int gn = min(g + 1, gs1 - 1);
            dma_a(gn, 1);
            load_w(wB, gn);
            compute(0, wA, g);
            wait_vmcnt<2 * Q8RB>();
        }
        lds_sync();
        if (g + 1 >= gs1) break;
        {
            const int gn = min(g + 2, gs1 - 1);
            dma_a(gn, 0);
            load_w(wA, gn);
            compute(1, wB, g + 1);
            wait_vmcnt<2 * Q8RB>();
        }
        lds_sync();
    }
#pragma unroll
    for (int q = 0; q < Q8RB; q++) {
        const int n = (rbw + q) * 16 + r;
        if (rbw + q >= a.nrb || n >= a.N) continue;
        const float rs = ((const float*)a.scale)[n];
#pragma unroll
        for (int mb = 0; mb < 4; mb++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int b = GB * by + 16 * mb + 4 * s + v;
                if (b < a.M) {
                    const float tt = (float)acc[q][mb][0][v] + (float)acc[q][mb][1][v] * 0.0078125f +
                                     (float)acc[q][mb][2][v] * 6.103515625e-05f;
                    const float val = (tt * a.xs[b]) * rs;
                    if (a.part) {
                        a.part[((size_t)blockIdx.z * a.M + b) * a.N + n] = val;
                    } else {
                        float* yp = a.y + (size_t)b * a.ldy + n;
                        *yp = a.resid ? *yp + val : val;
                    }
                }
            }
    }
}

// y = (resid ? y : 0) + sum over the parts in part order (split K).
__global__ __launch_bounds__(256) void k_gemm_reduce(const float* __restrict__ part, int nz, int M, int N,
                                                     float* __restrict__ y, int ldy, int resid) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= M * N) return;
    const int b = i / N, n = i - b * N;
    float acc = part[i];
    for (int z = 1; z < nz; z++) acc += part[(size_t)z * M * N + i];
    float* yp = y + (size_t)b * ldy + n;
    *yp = resid ? *yp + acc : acc;
}

// Operand planes of the GEMM (grown on demand).
// operand planes, row scales and split-K partial sums, grown on demand, per
// host thread (each thread runs on its own stream); a GEMM is never part of
// a captured graph (the decode rounds' batches are <= 16 rows)
static thread_local uint8_t* g_gemm_planes = nullptr;
static thread_local size_t g_gemm_cap = 0;
static thread_local float* g_gemm_xs = nullptr;
static thread_local size_t g_gemm_xs_cap = 0;
static thread_local float* g_gemm_part = nullptr;  // split-K partial sums
static thread_local size_t g_gemm_part_cap = 0;

// K parts for a grid of base workgroups over nsteps K steps: doubled while
// the grid is below one workgroup per CU (256), at least 4 steps a part.
// Measured on MI355X: q4t 1024x3072 m = 2048 (128 workgroups unsplit) 77 us
// in one part, 68 in two, 74 in four; q4tp 2048x6144 m = 200 (64) 90 / 61 /
// 46 us in 1 / 2 / 4; q4t 12288x4096 m = 64 (96) 62 / 46 / 42; a grid of
// 256 or more loses (2048x6144 m = 2048 161 -> 162, 6144x1024 88 -> 125).
static int gemm_kparts(long base, int nsteps) {
    static const int env = [] {
        const char* e = getenv("CMF_GEMM_SPLITK");
        return e ? atoi(e) : -1;
    }();
    if (env == 0) return 1;
    int z = 1;
    while (base * z < 256 && nsteps / (z * 2) >= 4) z *= 2;
    return z;
}

// Allows kernel kf its dynamic LDS (once a kernel).
static int gemm_lds(const void* kf, size_t bytes) {
    static std::mutex mu;
    static std::set<const void*> done;
    std::lock_guard<std::mutex> g(mu);
    if (!done.count(kf)) {
        CMF_HIP(hipFuncSetAttribute(kf, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes));
        done.insert(kf);
    }
    return CMF_OK;
}

// y[row][n] (ldy) of the rows of every tile, planes and xs prepared for
// ntiles * 64 rows (proto: an expert's weight, for the shape and codec).
// 64 weight rows a wave: the tiles alone fill the CUs.
int gemm_grouped(const DevWeight& proto, const GemvDesc* desc, const int2* tiles, int ntiles, const uint8_t* planes,
                 const float* xs, float* y, int ldy, hipStream_t st) {
    if (ntiles < 1 || ntiles > 65535 || !desc || !tiles) return fail("gemm: bad tile list");
    GemmArgs a{};
    a.planes = planes;
    a.xs = xs;
    a.y = y;
    a.ldy = ldy;
    a.Mp = ntiles * GB;
    a.N = proto.rows;
    a.ntg = proto.kchunks;
    a.nrb = proto.rows_pad / 16;
    a.tiles = tiles;
    a.desc = desc;
    void* args[] = {&a};
    if (proto.dtype == DT_Q8ROW) {
        a.gsteps = (a.ntg + 1) / 2;
        CMF_HIP(hipLaunchKernel((const void*)k_gemm_q8<2>, dim3((a.nrb + 7) / 8, ntiles), dim3(256), args,
                                GEMM_Q8_AT_BYTES, st));
        return CMF_OK;
    }
    a.gsteps = a.ntg;
    const void* kf = proto.dtype == DT_Q4T ? (const void*)k_gemm_q4<DT_Q4T, 2> : (const void*)k_gemm_q4<DT_Q4TP, 2>;
    if (gemm_lds(kf, GEMM_AT_BYTES) != CMF_OK) return CMF_ERR;
    CMF_HIP(hipLaunchKernel(kf, dim3((a.nrb + 15) / 16, ntiles), dim3(256), args, GEMM_AT_BYTES, st));
    return CMF_OK;
}

size_t gemm_planes_bytes(const DevWeight& w, int mp) {
    // q8: three planes of nk * 64 * Mp B; q4: hi + lo 2 * items * Mp * 16 B
    if (w.dtype == DT_Q8ROW) return (size_t)w.kchunks * 64 * mp * 3;
    return (size_t)w.kchunks * 16 * mp * 32;
}

int gemm(const DevWeight& w, const XSrc& src, int m, float* y, int ldy, bool resid, hipStream_t st, bool prepared) {
    if (w.dtype != DT_Q4T && w.dtype != DT_Q4TP && w.dtype != DT_Q8ROW) return fail("gemm: q8 / q4t / q4tp weights");
    if (m < 1 || m > 65535) return fail("gemm: batch must be 1..65535");
    const int mp = (m + GB - 1) / GB * GB;
    const size_t pb = gemm_planes_bytes(w, mp);
    if (g_gemm_cap < pb) {
        (void)hipStreamSynchronize(st);
        if (g_gemm_planes) (void)hipFree(g_gemm_planes);
        g_gemm_planes = nullptr;
        g_gemm_cap = 0;
        CMF_HIP(hipMalloc(&g_gemm_planes, pb));
        g_gemm_cap = pb;
    }
    if (g_gemm_xs_cap < (size_t)mp) {
        (void)hipStreamSynchronize(st);
        if (g_gemm_xs) (void)hipFree(g_gemm_xs);
        g_gemm_xs = nullptr;
        g_gemm_xs_cap = 0;
        CMF_HIP(hipMalloc(&g_gemm_xs, (size_t)mp * sizeof(float)));
        g_gemm_xs_cap = mp;
    }
    if (!prepared) {
        const int rc = launch_prep_src_gemm(w, src, m, mp, g_gemm_planes, g_gemm_xs, st);
        if (rc != CMF_OK) return rc;
    }
    GemmArgs a;
    a.w = w.w;
    a.scale = w.scale;
    a.rowp = w.rowp;
    a.planes = g_gemm_planes;
    a.xs = g_gemm_xs;
    a.y = y;
    a.ldy = ldy;
    a.M = m;
    a.Mp = mp;
    a.N = w.rows;
    a.ntg = w.kchunks;
    a.nrb = w.rows_pad / 16;
    a.resid = resid ? 1 : 0;
    a.part = nullptr;
    a.tiles = nullptr;
    a.desc = nullptr;
    // split K (nz parts into the partial buffer, then k_gemm_reduce)
    auto split = [&](long base, int nsteps) -> int {
        const int nz = gemm_kparts(base, nsteps);
        a.gsteps = (nsteps + nz - 1) / nz;
        if (nz == 1) return 1;
        const size_t need = (size_t)nz * m * w.rows;
        if (g_gemm_part_cap < need) {
            (void)hipStreamSynchronize(st);
            if (g_gemm_part) (void)hipFree(g_gemm_part);
            g_gemm_part = nullptr;
            g_gemm_part_cap = 0;
            if (hipMalloc(&g_gemm_part, need * sizeof(float)) != hipSuccess) return -1;
            g_gemm_part_cap = need;
        }
        a.part = g_gemm_part;
        return (nsteps + a.gsteps - 1) / a.gsteps;
    };
    auto reduce = [&](int nz) -> int {
        if (nz > 1)
            hipLaunchKernelGGL(k_gemm_reduce, dim3((m * w.rows + 255) / 256), dim3(256), 0, st, g_gemm_part, nz, m,
                               w.rows, y, ldy, a.resid);
        CMF_HIP(hipGetLastError());
        return CMF_OK;
    };
    if (w.dtype == DT_Q8ROW) {
        // two row blocks per wave once that still leaves ~4 workgroups per CU
        const bool big = (long)((a.nrb + 7) / 8) * (mp / GB) >= 1024;
        const int rbwg = big ? 8 : 4;
        const int gx = (a.nrb + rbwg - 1) / rbwg, nz = split((long)gx * (mp / GB), (a.ntg + 1) / 2);
        if (nz < 0) return fail("gemm: split-K buffer");
        const dim3 grid(gx, mp / GB, nz);
        if (big) hipLaunchKernelGGL((k_gemm_q8<2>), grid, dim3(256), GEMM_Q8_AT_BYTES, st, a);
        else hipLaunchKernelGGL((k_gemm_q8<1>), grid, dim3(256), GEMM_Q8_AT_BYTES, st, a);
        return reduce(nz);
    }
    // 64 rows a wave (half the operand reads of 32) where that gives a
    // workgroup to every CU, or to half of them and K is long enough (3072
    // columns) for its parts to fill the rest; else 32.  Measured on MI355X, us
    // at 64 / 32 rows: q4t 12288x4096 m = 2048 379 / 457, 4096x4096 m = 512 (128
    // workgroups) 57 / 63, 4096x12288 m = 700 (176) 185 / 208; but 2048x2048
    // m = 1024 (128) 40 / 35, 6144x2048 m = 512 (192) 52 / 43, 4096x1024 m = 512
    // (128) 30 / 21; q4tp 6144x2048 m = 200 (96) 50 / 40.
    const long wide = (long)((a.nrb + 15) / 16) * (mp / GB);
    const int rn = wide >= 256 || (wide >= 128 && a.ntg >= 24) ? 2 : 1;
    const int rbwg = 8 * rn;
    const int gx = (a.nrb + rbwg - 1) / rbwg;
    // up to 11 groups of K are split only where that leaves 64 workgroups or
    // fewer: the partial sums' launch takes 4 us (8 groups, in one part / two:
    // q4t 3072x1024 m = 128 (48 workgroups) 19.3 / 18.7 us, 4096x1024 m = 320
    // (160) 20 / 26, 6144x1024 m = 256 (192) 20 / 28)
    const long base = (long)gx * (mp / GB);
    const int nz = split(a.ntg < 12 && base > 64 ? 256 : base, a.ntg);
    if (nz < 0) return fail("gemm: split-K buffer");
    const dim3 grid(gx, mp / GB, nz);
    const bool q4t = w.dtype == DT_Q4T;
    const void* kf = rn == 2 ? (q4t ? (const void*)k_gemm_q4<DT_Q4T, 2> : (const void*)k_gemm_q4<DT_Q4TP, 2>)
                             : (q4t ? (const void*)k_gemm_q4<DT_Q4T, 1> : (const void*)k_gemm_q4<DT_Q4TP, 1>);
    if (gemm_lds(kf, GEMM_AT_BYTES) != CMF_OK) return CMF_ERR;
    void* args[] = {&a};
    CMF_HIP(hipLaunchKernel(kf, grid, dim3(256), args, GEMM_AT_BYTES, st));
    return reduce(nz);
}

int gemm_q4(const DevWeight& w, const float* x, int ldx, int m, float* y, int ldy, hipStream_t st) {
    XSrc r{};
    r.mode = XS_ROWS;
    r.x = x;
    r.ldx = ldx;
    return gemm(w, r, m, y, ldy, false, st);
}

}  // namespace cmf
