// Causal attention of a prefill chunk (head_dim 128) for gfx950.
//
// The chunk's rows sit at positions p0 .. p0 + cnt - 1 (p0 known to the
// host).  Three launches per chunk and layer:
//   - k_prefill_qk: q-norm + RoPE of the queries (into a scratch buffer),
//     k-norm + RoPE of the new K rows, K and V appended to the cache
//     (attention.rs:606-624, 818-890; kv_cache.rs:366-505), as the decode
//     kernels do it;
//   - k_prefill_fakv: the cache's K / V rows [0, p0 + cnt) rearranged into
//     32-key tiles of the attention's MFMA fragments (f16 hi / lo halves);
//   - k_prefill_fa: 128 query rows per block, two blocks per two workgroups
//     (contexts of at most FA64_KEYS: k_prefill_fa64, 64 rows per block, two
//     blocks per workgroup), each tile in LDS once per workgroup, with a
//     running (online) softmax: scores on the f16 MFMA (q.k = qh.kh + qh.kl + ql.kh, 22-bit
//     operands, f32 sums), causal limit the row's position
//     (kv_cache.rs:521-690), values ph.vh + ph.vl + pl.vh on the f16 MFMA.
// Rows of a block past the chunk see no keys and write nothing.
#include <math.h>

#include "common.h"
#include "layers.h"
#include "wave.h"
#include "xlayer.h"

namespace cmf {

namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float float2v __attribute__((ext_vector_type(2)));
typedef float float4v __attribute__((ext_vector_type(4)));
typedef float float16v __attribute__((ext_vector_type(16)));
typedef int int4v __attribute__((ext_vector_type(4)));

constexpr int HD = 128;
constexpr int KT2 = 128;      // the K / V scratch's padding unit (keys)

__device__ __forceinline__ void wait_vmcnt0() { __builtin_amdgcn_s_waitcnt((7 << 4) | (15 << 8)); }  // vmcnt(0) only
__device__ __forceinline__ void wait_vmcnt4() { __builtin_amdgcn_s_waitcnt(4 | (7 << 4) | (15 << 8)); }  // vmcnt(4) only
__device__ __forceinline__ void wait_all() { __builtin_amdgcn_s_waitcnt(7 << 4); }  // vmcnt(0) lgkmcnt(0)

// the LDS reads before the last N are in
template <int N>
__device__ __forceinline__ void wait_lds() {
    __builtin_amdgcn_s_waitcnt(15 | (7 << 4) | (N << 8) | (3 << 14));
    __builtin_amdgcn_sched_barrier(0);  // (before what uses them)
}

__device__ __forceinline__ uint32_t xcc_id() {
    uint32_t v;
    asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID, 0, 4)" : "=s"(v));
    return v;
}

// max / sum over the four lanes l, l ^ 16, l ^ 32, l ^ 48 (one MFMA output
// column) by the gfx950 row-swap permutes: each returns the value and its
// partner's, so op(first, second) is the pairwise result in every lane
__device__ __forceinline__ float lanes4_max(float v) {
    auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
    auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float lanes4_sum(float v) {
    auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
    auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// max / sum over the lanes l, l ^ 32 (one column of a 32x32 MFMA output) by
// the gfx950 row-swap permute: it returns the value and its partner's
__device__ __forceinline__ float lanes2_max(float v) {
    auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float lanes2_sum(float v) {
    auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

__device__ __forceinline__ void split16(float x, _Float16& hi, _Float16& lo) {
    hi = (_Float16)x;
    lo = (_Float16)(x - (float)hi);
}

// grid (cnt, hq + nkv), 64 threads: block y < hq: query head y of chunk row
// x into qbuf [cnt][nh][128]; else kv head y - hq: K (normed, rotated) and V
// of the row appended at position p0 + x.
__global__ __launch_bounds__(64) void k_prefill_qk(const float* __restrict__ qkv, int ldq,
                                                   const float* __restrict__ qn, const float* __restrict__ kn,
                                                   const float2* __restrict__ rope, float* __restrict__ kc,
                                                   float* __restrict__ vc, int max_seq, int p0, int nh, int nkv,
                                                   double eps, float* __restrict__ qbuf, int hq) {
    const int i = blockIdx.x, h = blockIdx.y, lane = threadIdx.x;
    const int pos = p0 + i;
    const float* row = qkv + (size_t)i * ldq;
    const float2 cs = rope[(size_t)pos * 64 + lane];
    if (h < hq) {
        const float* qr = row + (size_t)h * HD;
        const float2 o = norm_rope(qr[lane], qr[lane + 64], qn[lane], qn[lane + 64], cs, eps);
        float* q = qbuf + ((size_t)i * nh + h) * HD;
        q[lane] = o.x;
        q[lane + 64] = o.y;
    } else {
        const int g = h - hq;
        const float* kr = row + (size_t)(nh + g) * HD;
        const float* vr = row + (size_t)(nh + nkv + g) * HD;
        const float2 k = norm_rope(kr[lane], kr[lane + 64], kn[lane], kn[lane + 64], cs, eps);
        float* kd = kc + ((size_t)g * max_seq + pos) * HD;
        float* vd = vc + ((size_t)g * max_seq + pos) * HD;
        kd[lane] = k.x;
        kd[lane + 64] = k.y;
        vd[lane] = vr[lane];
        vd[lane + 64] = vr[lane + 64];
    }
}

// ---------------------------------------------------------------------------
// Scores are computed transposed, S^T = K Q^T (32x32x16 MFMA, 32 keys of a
// tile by the wave's 32 queries), so that each lane (query r = lane & 31,
// h = lane >> 5) ends up holding the weights of its own query for the keys
// 8 b + 4 h + c: exactly the B operand of O^T = V^T P^T when the V tile's
// k-slots hold the same keys, so the weights never go through LDS, and the
// output's lanes hold their own query's dims.  q.k = qh.kh + (qh.kl + ql.kh)
// (f16 hi / lo halves, f32 sums; the two small products share an accumulator,
// which k_prefill_fa64 does not: a rounding 2^-11 of the score's), exp2 of log2-scaled scores with a running
// maximum, values ph.vh + ph.vl + pl.vh.
// ---------------------------------------------------------------------------
constexpr int FT = 32;                // keys per tile
constexpr int FT_BYTES = 32 * 1024;   // one tile of one kv head: K then V fragments
constexpr int FQ = 128;               // query rows per block
constexpr int FRA = 4;                // fragment pairs read ahead
// contexts of at most this many keys take the 64-row blocks of 16-row waves
// (k_prefill_fa64): us a layer, 64 rows / 128 rows, of 16 query heads on 8 KV
// heads: 64 keys 8.7 / 13.8, 128 12 / 21, 256 16 / 23, 512 25.6 / 27.4, 640
// 30.7 / 29.7, 1024 45 / 36, 2048 86 / 59 (8 on 8, 4 on 4: 512 25.6 / 27,
// 640 30 / 29 and 31.9 / 29)
constexpr int FA64_KEYS = 576;

// The cached K / V rows [0, n) of every kv head as 32-key tiles of MFMA
// fragments, [nkv][npad / 32][32 fragments][64 lanes] x 16 B (keys past n
// zero).  W32 (k_prefill_fa):
//   K fragment 2 ks + plane: lane 32 h + r holds dims 16 ks + 8 h .. + 7 of
//     key r (A operand of S^T, f16 hi / lo);
//   V fragment 16 + 4 db + 2 t + plane: lane 32 h + r holds dim 32 db + r of
//     the keys 16 t + 4 h + j (j < 4) and 16 t + 8 + 4 h + j - 4 (j >= 4) (A
//     operand of O^T = V^T P^T).
// else (k_prefill_fa64):
//   K fragment 8 kb + 2 ks + plane: lane 16 s + r holds dims 32 ks + 8 s .. + 7
//     of key 16 kb + r;
//   V fragment 16 + 2 db + plane: lane 16 s + r holds dim 16 db + r of the
//     keys 4 s + j (j < 4) and 16 + 4 s + j - 4 (j >= 4).
// grid (npad / 32, nkv), 256 threads.
template <bool W32>
__global__ __launch_bounds__(256) void k_prefill_fakv(const float* __restrict__ kc, const float* __restrict__ vc,
                                                      int max_seq, int n, int npad, int4v* __restrict__ op) {
    const int t = threadIdx.x, tile = blockIdx.x, g = blockIdx.y;
    __shared__ float KS[FT][HD + 4], VS[FT][HD + 1];
    for (int e = t; e < FT * 32; e += 256) {
        const int k = e >> 5, c4 = 4 * (e & 31), key = FT * tile + k;
        float4v kv = {0.f, 0.f, 0.f, 0.f}, vv = kv;
        if (key < n) {
            kv = *(const float4v*)(kc + ((size_t)g * max_seq + key) * HD + c4);
            vv = *(const float4v*)(vc + ((size_t)g * max_seq + key) * HD + c4);
        }
        *(float4v*)&KS[k][c4] = kv;
#pragma unroll
        for (int i = 0; i < 4; i++) VS[k][c4 + i] = vv[i];
    }
    __syncthreads();
    int4v* dst = op + ((size_t)g * (npad / FT) + tile) * (FT_BYTES / 16);
    for (int e = t; e < 32 * 64; e += 256) {
        const int l = e & 63, f = e >> 6, r = W32 ? l & 31 : l & 15, sl = W32 ? l >> 5 : l >> 4, plane = f & 1;
        half8 h;
        if (f < 16) {
            const int k = W32 ? r : 16 * (f >> 3) + r, d0 = W32 ? 16 * (f >> 1) + 8 * sl : 32 * ((f >> 1) & 3) + 8 * sl;
#pragma unroll
            for (int j = 0; j < 8; j++) {
                _Float16 hh, ll;
                split16(KS[k][d0 + j], hh, ll);
                h[j] = plane ? ll : hh;
            }
        } else {
            const int d = W32 ? 32 * ((f - 16) >> 2) + r : 16 * ((f - 16) >> 1) + r;
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const int k = W32 ? 16 * ((f >> 1) & 1) + 8 * (j >> 2) + 4 * sl + (j & 3) : 16 * (j >> 2) + 4 * sl + (j & 3);
                _Float16 hh, ll;
                split16(VS[k][d], hh, ll);
                h[j] = plane ? ll : hh;
            }
        }
        dst[f * 64 + l] = __builtin_bit_cast(int4v, h);
    }
}

// grid (16 np) (XCD: kv head = the workgroup's XCD, unit = blockIdx / 8) or
// (2 np, nkv), np = ceil(nqb / 2); 512 threads.  A 128-row query block's
// eight waves are 4 row groups of 32 query rows (PPW = 32 / HPK positions
// times the HPK query heads of kv head g: row r of group w is chunk row
// PPW (4 qb + w) + r % PPW, query head g HPK + r / PPW) by the even and the
// odd 32-key tiles of a step; the two tiles of a step are fetched into LDS
// while the last two are used, and each is read by four waves.  Causal
// blocks see different numbers of tiles, so blocks are paired, i with z =
// nqb - 1 - i, and a pair's tiles dealt to two workgroups evenly: unit 2 i
// takes the first half of them (all block z's, the longer), unit 2 i + 1 the
// rest of z's and then block i's.  The halves of z meet through pt / pml: every
// wave waits until its sums are in L2, thread 0 writes that back (the other
// unit may be on another XCD; a release by each wave instead costs 15 us at
// 2048 positions) and exchanges the launch's tag into mcell; the unit that ends
// second (it finds the tag there) takes the first one's sums and writes the
// rows; none waits.
//
// The floor is the MFMA's (48 of 32x32x16 a wave and tile: 25 us at 2048
// positions of 16 heads at 2 GHz).  Against k_prefill_fa64 (86 -> 59 us): 32
// rows a wave halve the LDS reads per MFMA, both waves of a SIMD have work to
// the end (the pair's short block left four of the eight waves idle past its
// keys), and the tiles cross L2 8448 times instead of 12416.  What is left
// beside the MFMA is spread: without the tile fetch, the LDS reads or the
// softmax (timing only, of a build that took 63 us) it takes 57 to 61 us each;
// about 13 us are the rows' loads, the two merges and the stores.  Not better
// than that build: the last tile's values in the shadow of the next softmax
// (65 us), rows staged through LDS (63).
//
// XCD: the kv head is the XCD the workgroup runs on (its K / V stays in that
// XCD's L2), which covers each (unit, head) once only while the dispatcher
// deals workgroups to the 8 XCDs in turn; each workgroup therefore swaps the
// launch's tag into its cell [unit][g] first, and finding the tag already
// there sets *perr: the host then re-runs the prefill on the grid-indexed
// variant.
template <int HPK, bool XCD>
__global__ __launch_bounds__(512) void k_prefill_fa(const float* __restrict__ qbuf, const int4v* __restrict__ op,
                                                    int npad, int cnt, int p0, int nh, int nqb, float* __restrict__ out,
                                                    unsigned long long* cells, int* perr, unsigned long long* mcell,
                                                    unsigned long long tag, float4v* pt, float2v* pml) {
    constexpr int PPW = 32 / HPK;
    extern __shared__ __align__(16) uint8_t fsm[];  // two steps of two tiles (direct-load targets)
    __shared__ float2v sml[8][64];
    __shared__ int s_second;
    const int unit = XCD ? (int)(blockIdx.x >> 3) : (int)blockIdx.x;
    const int g = XCD ? (int)(xcc_id() & 7) : (int)blockIdx.y;
    const int nkv = nh / HPK;
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    if constexpr (XCD) {
        if (t == 0 && atomicExch(cells + unit * 8 + g, tag) == tag) atomicOr(perr, 1);
    }
    const int pi = unit >> 1, upper = unit & 1;
    const int qz = nqb - 1 - pi, qi = pi;  // the pair (qz == qi: one block)
    auto tiles_of = [&](int qb) { return (p0 + min((qb + 1) * 4 * PPW, cnt) - 1) / FT + 1; };
    const int nz = tiles_of(qz), ni = qi == qz ? 0 : tiles_of(qi);
    const int cut = min((nz + ni + 1) / 2, nz);  // (ni <= nz: the first half is z's)
    const bool split = cut < nz;
    // this unit's one or two runs of tiles [b, e) of a block
    const int b0 = upper ? cut : 0, e0 = upper ? nz : cut, e1 = upper ? ni : 0;
    const int ns0 = (e0 - b0 + 1) >> 1, ns = ns0 + ((e1 + 1) >> 1);  // steps
    const int r = lane & 31, h = lane >> 5, rg = wave & 3, par = wave >> 2;
    const uint8_t* src = (const uint8_t*)(op + (size_t)g * (npad / FT) * (FT_BYTES / 16));
    // step st's two tiles into buffer st & 1: waves 0-3 the even one, 4-7 the odd one
    auto fetch = [&](int st) {
        const int tt = (st < ns0 ? b0 + 2 * st : 2 * (st - ns0)) + par;
        if (tt >= (st < ns0 ? e0 : e1)) return;  // (uniform per wave)
        const uint8_t* from = src + __builtin_amdgcn_readfirstlane(tt * FT_BYTES + rg * 8192);  // (below 2 GiB: 65536 tiles)
#pragma unroll
        for (int c = 0; c < 8; c++) {
            const int ch = 8 * rg + c;
            __builtin_amdgcn_global_load_lds((const void*)(from + c * 1024 + lane * 16),
                                             (__attribute__((address_space(3))) void*)(fsm + (2 * (st & 1) + par) * FT_BYTES + ch * 1024),
                                             16, 0, 0);
        }
    };
    const float scale = 1.4426950408889634f / sqrtf((float)HD);
    if (ns > 0) fetch(0);
    int st = 0;
#pragma unroll 1
    for (int run = 0; run < 2; run++) {
        const int tb = run ? 0 : b0, te = run ? e1 : e0, qb = run ? qi : qz;
        if (tb >= te) continue;  // (uniform per workgroup)
        const int i0 = (4 * qb + rg) * PPW;   // this wave's first chunk row
        const int row = i0 + r % PPW, head = g * HPK + r / PPW, qpos = p0 + row;  // query r
        const bool qv = row < cnt;
        // tiles any row of the wave sees; of them, the tiles all of its rows see whole
        const int wt = i0 < cnt ? (p0 + min(i0 + PPW, cnt) - 1) / FT + 1 : 0, wfull = (p0 + i0 + 1) / FT;
        // the queries (the B operand of S^T), f16 hi / lo
        half8 qh[HD / 16], ql[HD / 16];
        {
            const float* qrow = qbuf + ((size_t)(qv ? row : 0) * nh + head) * HD;
#pragma unroll
            for (int ks = 0; ks < HD / 16; ks++) {
                const float4v a0 = *(const float4v*)(qrow + 16 * ks + 8 * h);
                const float4v a1 = *(const float4v*)(qrow + 16 * ks + 8 * h + 4);
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    _Float16 hh, ll;
                    split16(qv ? (j < 4 ? a0[j] : a1[j - 4]) : 0.f, hh, ll);
                    qh[ks][j] = hh;
                    ql[ks][j] = ll;
                }
            }
        }
        float m = -INFINITY, l = 0.f;  // query r: raw score maximum (both lanes), this lane's share of the sum
        float16v o[4];                 // dims 32 db + 8 (e >> 2) + 4 h + (e & 3)
#pragma unroll
        for (int db = 0; db < 4; db++)
#pragma unroll
            for (int e = 0; e < 16; e++) o[db][e] = 0.f;
        for (int ti = tb; ti < te; ti += 2, st++) {
            wait_all();  // this wave's share of the step is in
            asm volatile("s_barrier" ::: "memory");  // every wave's; the other buffer is free
            const int tt = ti + par;
            if (tt >= te || tt >= wt) {  // (uniform per wave)
                if (st + 1 < ns) fetch(st + 1);
                continue;
            }
            const int4v* F = (const int4v*)(fsm + (2 * (st & 1) + par) * FT_BYTES) + lane;
            // the tile's fragments in sixteen pairs (hi, lo), each read FRA pairs
            // of three MFMAs ahead of its use (left alone the compiler reads a
            // pair and waits for it)
            half8 f[FRA + 1][2];
            auto read = [&](int gr) {
                f[gr % (FRA + 1)][0] = __builtin_bit_cast(half8, F[(2 * gr) * 64]);
                f[gr % (FRA + 1)][1] = __builtin_bit_cast(half8, F[(2 * gr + 1) * 64]);
                __builtin_amdgcn_sched_barrier(0);
            };
#pragma unroll
            for (int gr = 0; gr < FRA; gr++) read(gr);
            // S^T: dh + dl [e] = key 8 (e >> 2) + 4 h + (e & 3), query r
            float16v dh, dl;
#pragma unroll
            for (int e = 0; e < 16; e++) dh[e] = dl[e] = 0.f;
#pragma unroll
            for (int ks = 0; ks < HD / 16; ks++) {
                read(ks + FRA);
                wait_lds<2 * FRA>();
                const half8 kh = f[ks % (FRA + 1)][0], kl = f[ks % (FRA + 1)][1];
                dl = __builtin_amdgcn_mfma_f32_32x32x16_f16(kl, qh[ks], dl, 0, 0, 0);
                dh = __builtin_amdgcn_mfma_f32_32x32x16_f16(kh, qh[ks], dh, 0, 0, 0);
                dl = __builtin_amdgcn_mfma_f32_32x32x16_f16(kh, ql[ks], dl, 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
            // (after the K fragments' waits: with direct loads in flight the
            // compiler waits for all LDS reads where it would count them)
            if (st + 1 < ns) fetch(st + 1);
            // causal mask where the tile crosses it, the running softmax of query r
            float sv[16];
#pragma unroll
            for (int e = 0; e < 16; e++) sv[e] = dh[e] + dl[e];
            if (tt >= wfull) {
#pragma unroll
                for (int e = 0; e < 16; e++)
                    if (FT * tt + 8 * (e >> 2) + 4 * h + (e & 3) > qpos) sv[e] = -INFINITY;
            }
            float mt = sv[0];
#pragma unroll
            for (int e = 1; e < 16; e++) mt = fmaxf(mt, sv[e]);
            const float mn = fmaxf(m, lanes2_max(mt));
            // the weights are relative to a maximum at most 2^8 behind (f16
            // holds them, hi + lo keep their 22 bits): every new maximum of
            // any row would have all sums rescaled at most tiles
            if (__any((mn - m) * scale > 8.f)) {  // (wave-uniform)
                const float al = __builtin_amdgcn_exp2f((m - (mn == -INFINITY ? 0.f : mn)) * scale);
                l *= al;
#pragma unroll
                for (int db = 0; db < 4; db++)
#pragma unroll
                    for (int e = 0; e < 16; e++) o[db][e] *= al;
                m = mn;
            }
            const float ms = (m == -INFINITY ? 0.f : m) * scale;  // (no key yet: every weight exp2(-inf))
            half8 ph[2], pl[2];
#pragma unroll
            for (int e = 0; e < 16; e += 2) {
                const float2v pv = {__builtin_amdgcn_exp2f(__builtin_fmaf(sv[e], scale, -ms)),
                                    __builtin_amdgcn_exp2f(__builtin_fmaf(sv[e + 1], scale, -ms))};
                l += pv[0] + pv[1];
                const half2v hh = __builtin_convertvector(pv, half2v);
                const float2v rest = {pv[0] - (float)hh[0], pv[1] - (float)hh[1]};
                const half2v ll = __builtin_convertvector(rest, half2v);
                ph[e >> 3][e & 7] = hh[0];
                ph[e >> 3][(e & 7) + 1] = hh[1];
                pl[e >> 3][e & 7] = ll[0];
                pl[e >> 3][(e & 7) + 1] = ll[1];
            }
            // O^T += V^T P^T (the same registers as operands the other way
            // round): a lane holds dims of its own query
#pragma unroll
            for (int db = 0; db < 4; db++) {
#pragma unroll
                for (int k = 0; k < 2; k++) {
                    const int gr = 8 + 2 * db + k;
                    if (gr + FRA < 16) read(gr + FRA);
                    const int left = 15 - gr;  // pairs read after this one, FRA of them at most
                    if (left >= FRA) wait_lds<2 * FRA>();
                    else if (left == 3) wait_lds<6>();
                    else if (left == 2) wait_lds<4>();
                    else if (left == 1) wait_lds<2>();
                    else wait_lds<0>();
                    const half8 vh = f[gr % (FRA + 1)][0], vl = f[gr % (FRA + 1)][1];
                    o[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vh, ph[k], o[db], 0, 0, 0);
                    o[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vl, ph[k], o[db], 0, 0, 0);
                    o[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vh, pl[k], o[db], 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
        // the even and odd tiles' sums meet in the buffer just read: wave rg
        // takes dims 0..63, wave rg + 4 dims 64..127
        l = lanes2_sum(l);
        sml[wave][lane] = float2v{m, l};
        __syncthreads();
        float4v* X = (float4v*)(fsm + 2 * ((st - 1) & 1) * FT_BYTES);
#pragma unroll
        for (int i = 0; i < 8; i++) {
            float4v x;
#pragma unroll
            for (int c = 0; c < 4; c++) x[c] = par ? o[i >> 2][4 * (i & 3) + c] : o[2 + (i >> 2)][4 * (i & 3) + c];
            X[(wave * 8 + i) * 64 + lane] = x;
        }
        __syncthreads();
        const float2v oml = sml[wave ^ 4][lane];
        float M = fmaxf(m, oml[0]);
        // the sums of keys a (even tiles, lower half) and b in that order, whichever wave or unit adds them
        auto weight = [&](float x) { return __builtin_amdgcn_exp2f((x - (M == -INFINITY ? 0.f : M)) * scale); };
        float fm = weight(m), fo = weight(oml[0]);
        float L = par ? __builtin_fmaf(l, fm, oml[1] * fo) : __builtin_fmaf(oml[1], fo, l * fm);
        float4v res[8];  // dims 64 par + 8 i + 4 h ..
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const float4v x = X[((wave ^ 4) * 8 + i) * 64 + lane];
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const float own = par ? o[2 + (i >> 2)][4 * (i & 3) + c] : o[i >> 2][4 * (i & 3) + c];
                res[i][c] = par ? __builtin_fmaf(own, fm, x[c] * fo) : __builtin_fmaf(x[c], fo, own * fm);
            }
        }
        if (!run && split) {  // (uniform per workgroup) the other unit has the other half of these rows' keys
            const size_t cell = (size_t)pi * nkv + g;
            int ln = lane;
            asm volatile("" : "+v"(ln));  // (these addresses are not worth registers across the tiles)
            float4v* mine = pt + (2 * cell + upper) * (FQ * HD / 4) + wave * 512 + ln;
            float2v* ml = pml + 2 * cell * 256 + wave * 64 + ln;  // (both halves' waves hold them)
            const auto seen = [&](bool first) {
                if (t == 0) {
                    if (!first) {  // write the XCD's L2 back; the exchange goes out after that
                        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
                        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                    }
                    s_second = (first ? __hip_atomic_load(mcell + cell, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT)
                                      : __hip_atomic_exchange(mcell + cell, tag, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT)) == tag;
                }
                __syncthreads();
                return s_second != 0;
            };
            bool second = seen(true);
            if (!second) {
#pragma unroll
                for (int i = 0; i < 8; i++) mine[i * 64] = res[i];
                if (par == 0) ml[upper * 256] = float2v{M, L};
                // (every wave's own sums are in L2 before the barrier that lets
                // thread 0 release and publish them: the barrier alone waits
                // for no store)
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                __syncthreads();
                second = seen(false);
                if (!second) continue;
            }
            const float4v* its = pt + (2 * cell + (upper ^ 1)) * (FQ * HD / 4) + wave * 512 + ln;
            const float2v iml = pml[(2 * cell + (upper ^ 1)) * 256 + rg * 64 + ln];
            const float own = M;
            M = fmaxf(M, iml[0]);
            fm = weight(own);
            fo = weight(iml[0]);
            L = upper ? __builtin_fmaf(L, fm, iml[1] * fo) : __builtin_fmaf(iml[1], fo, L * fm);
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const float4v x = its[i * 64];
#pragma unroll
                for (int c = 0; c < 4; c++)
                    res[i][c] = upper ? __builtin_fmaf(res[i][c], fm, x[c] * fo) : __builtin_fmaf(x[c], fo, res[i][c] * fm);
            }
        }
        if (qv) {
            float* dst = out + (size_t)row * nh * HD + (size_t)head * HD + 64 * par + 4 * h;
#pragma unroll
            for (int i = 0; i < 8; i++) *(float4v*)(dst + 8 * i) = res[i] / L;
        }
    }
}

// ---------------------------------------------------------------------------
// Short contexts: blocks of 64 query rows in four waves of 16 (16x16x32 MFMA),
// S^T and O^T as above with lane (query r = lane & 15, k-slot s = lane >> 4)
// holding the weights of the keys 4 s .. + 3 and 16 + 4 s .. + 3.  Half the
// rows and keys of a step and nothing to merge: where there are few tiles the
// fixed costs of k_prefill_fa (two merges, wider rows) outweigh its rate.  Bound
// by latency: a chain of one fetch, two products and a softmax a tile.
// grid (8 np) (XCD: kv head = the workgroup's XCD, pair index i =
// blockIdx / 8) or (np, nkv), np = ceil(nqb / 2); 512 threads.  The
// workgroup serves two 64-row query blocks that see about as many keys
// together as any other pair: waves 0-3 block i, waves 4-7 block nqb - 1 -
// i (none when that is block i again), sharing one fetch of every K / V
// tile the short block needs.  Wave w of a block holds 16 query rows, PPW =
// 16 / HPK positions times the HPK query heads of kv head g (row q: chunk
// row PPW (4 qb + w % 4) + q % PPW, query head g HPK + q / PPW).  XCD: the
// kv head is the XCD the workgroup runs on (its K / V stays in that XCD's
// L2), which covers each (query block, head) once only while the
// dispatcher deals workgroups to the 8 XCDs in turn; each workgroup
// therefore swaps the launch's tag into its blocks' cells [qb][g] first,
// and finding the tag already there sets *perr: the host then re-runs the
// prefill on the grid-indexed variant.
template <int HPK, bool XCD>
__global__ __launch_bounds__(512) void k_prefill_fa64(const float* __restrict__ qbuf, const int4v* __restrict__ op,
                                                    int npad, int cnt, int p0, int nh, int nqb, float* __restrict__ out,
                                                    unsigned long long* cells, int* perr, unsigned long long tag) {
    constexpr int PPW = 16 / HPK;
    extern __shared__ __align__(16) uint8_t fsm[];  // three tiles (direct-load targets)
    const int pi = XCD ? (int)(blockIdx.x >> 3) : (int)blockIdx.x;
    const int g = XCD ? (int)(xcc_id() & 7) : (int)blockIdx.y;
    const int qa = pi, qz = nqb - 1 - pi;  // the pair (qz == qa: one block)
    if constexpr (XCD) {
        if (threadIdx.x == 0 && atomicExch(cells + qa * 8 + g, tag) == tag) atomicOr(perr, 1);
        if (threadIdx.x == 64 && qz != qa && atomicExch(cells + qz * 8 + g, tag) == tag) atomicOr(perr, 1);
    }
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int r = lane & 15, s = lane >> 4;
    const bool second = wave >= 4;
    const bool live = !second || qz != qa;                 // (uniform per wave)
    const int qb = second ? qz : qa;
    const int i0 = (4 * qb + (wave & 3)) * PPW;           // this wave's first chunk row
    const int lastrow = min((4 * qb + 4) * PPW, cnt) - 1; // its block's last chunk row
    const int lastz = min((4 * max(qa, qz) + 4) * PPW, cnt) - 1;  // the pair's
    // the queries of column r (the B operand of S^T), f16 hi / lo
    const bool qv = live && i0 + r % PPW < cnt;
    const int qpos = p0 + i0 + r % PPW;                 // position of query r
    half8 qh[HD / 32], ql[HD / 32];
    {
        const float* qrow = qbuf + ((size_t)(qv ? i0 + r % PPW : 0) * nh + g * HPK + r / PPW) * HD;
#pragma unroll
        for (int ks = 0; ks < HD / 32; ks++) {
            const float4v a0 = *(const float4v*)(qrow + 32 * ks + 8 * s);
            const float4v a1 = *(const float4v*)(qrow + 32 * ks + 8 * s + 4);
#pragma unroll
            for (int j = 0; j < 8; j++) {
                _Float16 hh, ll;
                split16(qv ? (j < 4 ? a0[j] : a1[j - 4]) : 0.f, hh, ll);
                qh[ks][j] = hh;
                ql[ks][j] = ll;
            }
        }
    }
    // tiles of the pair (the fetch loop) and of this wave's block
    const int ntiles = lastz < 0 ? 0 : (p0 + lastz) / FT + 1;
    const int mytiles = !live || lastrow < 0 ? 0 : (p0 + lastrow) / FT + 1;
    const uint8_t* src = (const uint8_t*)(op + (size_t)g * (npad / FT) * (FT_BYTES / 16));
    // tile tt into buffer b: 32 KiB as 32 chunks of 1 KiB, 4 per wave
    auto fetch = [&](int tt, int b) {
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const int ch = 4 * wave + c;
            __builtin_amdgcn_global_load_lds((const void*)(src + (size_t)tt * FT_BYTES + ch * 1024 + lane * 16),
                                             (__attribute__((address_space(3))) void*)(fsm + b * FT_BYTES + ch * 1024),
                                             16, 0, 0);
        }
    };
    const float scale = 1.4426950408889634f / sqrtf((float)HD);
    float m = -INFINITY, l = 0.f;   // of query r (the same in the four lanes of column r)
    float4v o[8];                   // rows 4 s + e, dims 16 db + r
#pragma unroll
    for (int db = 0; db < 8; db++) o[db] = float4v{0.f, 0.f, 0.f, 0.f};
    // three buffers: tile tt + 2 is requested while tile tt is used
    if (ntiles > 0) fetch(0, 0);
    if (ntiles > 1) fetch(1, 1);
    for (int tt = 0; tt < ntiles; tt++) {
        const int b = tt % 3;
        if (tt + 1 < ntiles) wait_vmcnt4();  // tile tt's share is in (tile tt + 1's may not be)
        else wait_vmcnt0();
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // every wave's share is in; tile tt - 1's buffer is free
        if (tt + 2 < ntiles) fetch(tt + 2, (tt + 2) % 3);
        if (tt >= mytiles) continue;  // (uniform per wave: past this block's keys)
        const int4v* F = (const int4v*)(fsm + b * FT_BYTES) + lane;
        // S^T for the two key blocks: d[kb][e] = key 16 kb + 4 s + e, query r
        float4v d[2];
#pragma unroll
        for (int kb = 0; kb < 2; kb++) {
            float4v d0 = {0.f, 0.f, 0.f, 0.f}, d1 = d0, d2 = d0;
#pragma unroll
            for (int ks = 0; ks < HD / 32; ks++) {
                const half8 kh = __builtin_bit_cast(half8, F[(8 * kb + 2 * ks) * 64]);
                const half8 kl = __builtin_bit_cast(half8, F[(8 * kb + 2 * ks + 1) * 64]);
                d0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(kh, qh[ks], d0, 0, 0, 0);
                d1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(kl, qh[ks], d1, 0, 0, 0);
                d2 = __builtin_amdgcn_mfma_f32_16x16x32_f16(kh, ql[ks], d2, 0, 0, 0);
            }
            d[kb] = d0 + (d1 + d2);
        }
        // causal mask, log2 scale, the running softmax of query r
        float sv[8];
        float mt = -INFINITY;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int key = FT * tt + (j < 4 ? 4 * s + j : 16 + 4 * s + (j - 4));
            const float x = j < 4 ? d[0][j] : d[1][j - 4];
            sv[j] = qv && key <= qpos ? x * scale : -INFINITY;
            mt = fmaxf(mt, sv[j]);
        }
        mt = lanes4_max(mt);
        const float mn = fmaxf(m, mt);
        const float al = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - mn);
        float ps = 0.f;
        half8 ph, pl;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const float pv = mn == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(sv[j] - mn);
            ps += pv;
            _Float16 hh, ll;
            split16(pv, hh, ll);
            ph[j] = hh;
            pl[j] = ll;
        }
        ps = lanes4_sum(ps);
        l = l * al + ps;
        m = mn;
        // O^T += V^T P^T (the same registers as operands the other way
        // round): lane (query r, s) holds dims 16 db + 4 s + e of its own
        // query, so the rescale needs no exchange
#pragma unroll
        for (int db = 0; db < 8; db++) {
            float4v acc = o[db] * al;
            const half8 vh = __builtin_bit_cast(half8, F[(16 + 2 * db) * 64]);
            const half8 vl = __builtin_bit_cast(half8, F[(16 + 2 * db + 1) * 64]);
            acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(vh, ph, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(vl, ph, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(vh, pl, acc, 0, 0, 0);
            o[db] = acc;
        }
    }
    // out = o / l of query r: dims 16 db + 4 s .. + 3
    const int row = i0 + r % PPW, head = g * HPK + r / PPW;
    if (live && row < cnt) {
        float* dst = out + (size_t)row * nh * HD + (size_t)head * HD + 4 * s;
#pragma unroll
        for (int db = 0; db < 8; db++) *(float4v*)(dst + 16 * db) = o[db] / l;
    }
}

}  // namespace

bool prefill_attention_fits(int nh, int nkv, int hd) {
    if (hd != HD || nkv < 1 || nh % nkv) return false;
    const int hpk = nh / nkv;
    return hpk == 1 || hpk == 2 || hpk == 4 || hpk == 8 || hpk == 16;
}

size_t prefill_attention_cells(int cnt, int nh, int nkv) {
    const int ppb = FQ / (nh / nkv);
    return (size_t)(((cnt + ppb - 1) / ppb + 1) / 2) * nkv;
}

size_t prefill_attention_scratch(int cnt, int nh, int nkv) {
    return prefill_attention_cells(cnt, nh, nkv) * 2 * (FQ * HD * sizeof(float) + 256 * sizeof(float2v));
}

int launch_prefill_attention(const PrefillAttnArgs& a, hipStream_t st) {
    if (!prefill_attention_fits(a.nh, a.nkv, HD) || a.cnt < 1 || a.p0 < 0 || a.p0 + a.cnt > a.max_seq)
        return fail("prefill attention: head_dim 128, query heads a power-of-two multiple (<= 16) of kv heads");
    const int hq = a.out ? a.nh : 0;
    hipLaunchKernelGGL(k_prefill_qk, dim3(a.cnt, hq + a.nkv), dim3(64), 0, st, a.qkv, a.ldq, a.qn, a.kn, a.rope,
                       a.kc, a.vc, a.max_seq, a.p0, a.nh, a.nkv, a.eps, a.qbuf, hq);
    if (!a.out) return CMF_OK;
    const int hpk = a.nh / a.nkv;
    const int n = a.p0 + a.cnt, npad = (n + KT2 - 1) / KT2 * KT2;
    const bool small = n <= FA64_KEYS;
    const int ppb = (small ? 64 : FQ) / hpk;
    const int nqb = (a.cnt + ppb - 1) / ppb;  // query blocks, paired
    const int np = (nqb + 1) / 2;
    const bool xcd = a.nkv == 8 && xl_device_fits() && a.allow_xcd && a.cells && a.perr &&
                     (small ? 8 * nqb : 16 * np) <= PREFILL_XCD_CELLS;
    int4v* op = (int4v*)a.khl;  // nkv x npad x 1 KiB
    hipLaunchKernelGGL(small ? k_prefill_fakv<false> : k_prefill_fakv<true>, dim3(npad / FT, a.nkv), dim3(256), 0, st,
                       a.kc, a.vc, a.max_seq, n, npad, op);
    if (small) {
        typedef void (*KernS)(const float*, const int4v*, int, int, int, int, int, float*, unsigned long long*, int*,
                              unsigned long long);
        KernS k;
        switch (hpk) {
            case 1: k = xcd ? k_prefill_fa64<1, true> : k_prefill_fa64<1, false>; break;
            case 2: k = xcd ? k_prefill_fa64<2, true> : k_prefill_fa64<2, false>; break;
            case 4: k = xcd ? k_prefill_fa64<4, true> : k_prefill_fa64<4, false>; break;
            case 8: k = xcd ? k_prefill_fa64<8, true> : k_prefill_fa64<8, false>; break;
            default: k = xcd ? k_prefill_fa64<16, true> : k_prefill_fa64<16, false>; break;
        }
        static const bool attr = [] {  // (96 KiB: above the default dynamic LDS limit)
            bool ok = true;
            for (KernS f : {k_prefill_fa64<1, true>, k_prefill_fa64<1, false>, k_prefill_fa64<2, true>,
                            k_prefill_fa64<2, false>, k_prefill_fa64<4, true>, k_prefill_fa64<4, false>,
                            k_prefill_fa64<8, true>, k_prefill_fa64<8, false>, k_prefill_fa64<16, true>,
                            k_prefill_fa64<16, false>})
                ok &= hipFuncSetAttribute((const void*)f, hipFuncAttributeMaxDynamicSharedMemorySize, 3 * FT_BYTES) ==
                      hipSuccess;
            return ok;
        }();
        if (!attr) return fail("prefill attention: dynamic LDS attribute");
        hipLaunchKernelGGL(k, xcd ? dim3(8 * np) : dim3(np, a.nkv), dim3(512), 3 * FT_BYTES, st, a.qbuf, op, npad, a.cnt,
                           a.p0, a.nh, nqb, a.out, a.cells, a.perr, a.tag);
        return CMF_OK;
    }
    typedef void (*KernF)(const float*, const int4v*, int, int, int, int, int, float*, unsigned long long*, int*,
                          unsigned long long*, unsigned long long, float4v*, float2v*);
    KernF k;
    switch (hpk) {
        case 1: k = xcd ? k_prefill_fa<1, true> : k_prefill_fa<1, false>; break;
        case 2: k = xcd ? k_prefill_fa<2, true> : k_prefill_fa<2, false>; break;
        case 4: k = xcd ? k_prefill_fa<4, true> : k_prefill_fa<4, false>; break;
        case 8: k = xcd ? k_prefill_fa<8, true> : k_prefill_fa<8, false>; break;
        default: k = xcd ? k_prefill_fa<16, true> : k_prefill_fa<16, false>; break;
    }
    const dim3 grid = xcd ? dim3(16 * np) : dim3(2 * np, a.nkv);
    static const bool attr = [] {  // (128 KiB: above the default dynamic LDS limit)
        bool ok = true;
        for (KernF f : {k_prefill_fa<1, true>, k_prefill_fa<1, false>, k_prefill_fa<2, true>, k_prefill_fa<2, false>,
                        k_prefill_fa<4, true>, k_prefill_fa<4, false>, k_prefill_fa<8, true>, k_prefill_fa<8, false>,
                        k_prefill_fa<16, true>, k_prefill_fa<16, false>})
            ok &= hipFuncSetAttribute((const void*)f, hipFuncAttributeMaxDynamicSharedMemorySize, 4 * FT_BYTES) ==
                  hipSuccess;
        return ok;
    }();
    if (!attr) return fail("prefill attention: dynamic LDS attribute");
    float4v* pt = (float4v*)a.part;
    float2v* pml = (float2v*)(pt + (size_t)np * a.nkv * 2 * (FQ * HD / 4));
    hipLaunchKernelGGL(k, grid, dim3(512), 4 * FT_BYTES, st, a.qbuf, op, npad, a.cnt, a.p0, a.nh, nqb, a.out,
                       a.cells, a.perr, a.mcell, a.tag, pt, pml);
    return CMF_OK;
}

}  // namespace cmf
