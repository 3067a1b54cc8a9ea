// SPDX-License-Identifier: MIT
// FLASH_ATTN_EXT for the absorbed MLA of DeepSeek-style models, fused: dk 576, dv 512, V the first
// 512 dims of K (one cache, read once for both products). Same semantics as mx_fa_wide.hip, which
// keeps every other head dim past 256 and calls whose V is not that view of K.
//
// A block takes 64 query rows of one KV head (row = token * heads per KV head + head, so a block
// spans few tokens and a causal mask skips whole key tiles) and walks 64-key tiles; K's [64][576]
// tile arrives in LDS by DMA, two buffers, one landing while the other is used. Four waves, one a
// SIMD, with 512 registers each (eight waves of 256 spilled, and a spill's reload waits for the DMA in
// flight: 218 us where this takes 110). Per tile:
//   scores  wave (kg, qg) = (w / 2, w % 2) computes S^T of 32 keys x 32 queries: 18 32-deep steps
//           of four 16x16x32 MFMAs, its Q fragments (144 registers) held for the whole kernel;
//   softmax the two key groups exchange their row maxima through LDS (one barrier), every wave
//           follows the running max of all 64 rows, and P goes to LDS as fp16 (a second barrier);
//   output  wave w computes O^T of dims 128 w .. 128 w + 127 x 64 queries (128 accumulators), V^T read
//           from the K tile by ds_read_b64_tr_b16.
// What bounds it: per tile 2176 clocks of MFMA a SIMD and 2480 of LDS traffic a CU (147 KB of K
// fragments, 64 KB of V and 32 KB of P fragments, 74 KB of DMA), but also some 1500 clocks of softmax,
// which one wave a SIMD cannot overlap with its MFMAs: 2.9 us a tile, 12 us of prologue and 7 us for a
// split's partial rows. Three registers a lane spill, outside the loop over the tiles: a reload in it would wait
// for the next tile's DMA, as a mixed tile's mask loads do (with ten spilled, T 512 n_kv 4096 took 160 us with
// soft-cap, now 144; with a mask of holes in every tile 151, now 148). 64 rows a block because the O tile of 128 would leave no registers for Q; the key
// range is split across blocks to fill the chip, partial rows merged by fa_combine. The older form
// (fp16 Q and keys, transposed values, F32 scores through HBM, a softmax pass, two GEMMs) moved 134 MB of
// scores and P out and back. Whole call, 16 heads on one KV head, causal (older -> this, us): T 512 n_kv
// 4096 247 -> 116, n_kv 1024 107 -> 53; T 77 n_kv 3350 110 -> 49; T 16 n_kv 1024 43 -> 34; T 1 n_kv 4096 60 ->
// 41; 128 heads, T 512 n_kv 4096 1785 -> 729.
//
// Numerics as there: Q scaled, divided by its row's max and rounded to fp16, fp32 scores, P rounded to
// fp16 (the row sums are over the rounded P), fp32 accumulation; fully masked rows are zeros.

#include "mx_common.h"
#include "mx_kernels_impl.h"

namespace mx {

namespace {

constexpr int ML_DK = 576, ML_DV = 512, ML_BQ = 64, ML_KT = 64, ML_THREADS = 256;
constexpr int ML_RB = ML_DK * 2;                       // bytes per K row in LDS: 72 16-byte chunks
constexpr int ML_TILE = ML_KT * ML_RB;                 // 73728
constexpr int ML_PER = ML_TILE / (ML_THREADS * 16);    // 18 DMA instructions per wave and tile
constexpr int ML_P = 2 * ML_TILE;                      // P: [64 queries][64 keys] fp16
constexpr int ML_MAX = ML_P + ML_BQ * ML_KT * 2;       // row maxima: [64 queries][2 key groups]
constexpr int ML_SCALE = ML_MAX + ML_BQ * 8;           // Q row scales [64], then the range
constexpr int ML_TOK = ML_SCALE + ML_BQ * 4 + 16;      // mask row of each query row [64]
constexpr int ML_CLS = ML_TOK + ML_BQ * 4;             // the block's class of every key tile
constexpr int ML_MAX_TILES = FA_MLA_MAX_KV / ML_KT;
constexpr int ML_LDS = ML_CLS + ML_MAX_TILES;
static_assert(ML_PER * ML_THREADS * 16 == ML_TILE && ML_LDS <= 160 * 1024, "LDS");
constexpr int ML_QS = ML_DK / 32;                      // 32-deep steps of a score
constexpr int ML_Q1 = 13;                              // the first 13 keep their Q fragments in AGPRs (104 of them)
constexpr float ML_LAZY = 8.0f;   // how far a score may pass the running max, both in units of log 2

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef void __attribute__((address_space(3))) * ml_lptr;

__device__ __forceinline__ f32x4 ml_mfma(const half8 & a, const half8 & b, const f32x4 & c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}
// The same with b in AGPRs. In assembly, because the compiler copies such an operand to VGPRs for each
// use. It does not see that this is an MFMA, so the waits are here, those it puts around the builtin form
// on gfx950 (there is no interlock): two wait states between a vector instruction that writes an operand
// and the MFMA (s_nop 1 before each; under the MFMA before it they cost nothing), eight between the MFMA
// (16x16x32, 4 passes) and a vector or store instruction that reads its result (s_nop 7: ml_settle, between
// the last of these and anything else that touches their accumulators), and none between MFMAs that pass
// one accumulator on.
__device__ __forceinline__ void ml_mfma_a(const half8 & a, const half8 & b, f32x4 & c) {
    asm volatile("s_nop 1\nv_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "a"(b));
}
__device__ __forceinline__ void ml_settle(f32x4 (&s)[2][2]) {
    asm volatile("s_nop 7" : "+v"(s[0][0]), "+v"(s[0][1]), "+v"(s[1][0]), "+v"(s[1][1]));
}
// 16-byte chunk c of row r of the K tile (and of P, whose rows are 128 bytes): the low three bits of
// c by r / 2. Rows are 4.5 (P: 0.5) 256-byte bank windows apart, so the 16 rows of a fragment read
// fall on 16 distinct chunk slots.
__device__ __forceinline__ int ml_chunk(int r, int c) { return c ^ ((r >> 1) & 7); }

// The max over the four lanes of one query (16 lanes apart), by the row-swap exchanges: no LDS round trip.
__device__ __forceinline__ float ml_max_groups(float x) {
    const uint32_t u = __float_as_uint(x);
    const auto a = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    x = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
    const uint32_t w = __float_as_uint(x);
    const auto b = __builtin_amdgcn_permlane32_swap(w, w, false, false);
    return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

// s_waitcnt vmcnt(N) lgkmcnt(0)
template <int N> __device__ __forceinline__ void ml_wait() {
    __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (0 << 8) | ((N >> 4) << 14));
}
__device__ __forceinline__ void ml_barrier_lgkm() {   // LDS work done; global loads may be in flight
    __builtin_amdgcn_s_waitcnt(0xC07F);
    __builtin_amdgcn_s_barrier();
}

// A transposing read: lane i of each 16-lane group gets dim i of the 4 keys its group's lanes point at.
typedef _Float16 half4v __attribute__((ext_vector_type(4)));
typedef short short4v __attribute__((ext_vector_type(4)));
typedef short4v __attribute__((address_space(3))) * ml_s4ptr;
__device__ __forceinline__ half4v ml_tr_read(uint32_t lds) {
    return __builtin_bit_cast(half4v, __builtin_amdgcn_ds_read_tr16_b64_v4i16((ml_s4ptr)(uintptr_t)lds));
}

enum : uint8_t { ML_SKIP = 0, ML_FULL = 1, ML_MIXED = 2 };   // the classes fa_prep_kernel writes

}  // namespace

template <bool SOFTCAP>
__global__ void __launch_bounds__(ML_THREADS) __attribute__((amdgpu_waves_per_eu(1, 1))) fa_mla_kernel(FaArgs a) {
#ifdef __HIP_DEVICE_COMPILE__   // the buffer resource type exists in the device pass only
    extern __shared__ __align__(64) uint8_t smem[];
    const int t = threadIdx.x, lane = t % WAVE, wave = __builtin_amdgcn_readfirstlane(t / WAVE);
    const int lc = lane % 16, lg = lane / 16;
    const int kg = wave / 2, qg = wave % 2;
    const int g = a.H / a.HK, rows = g * a.T;
    const int nqb = (rows + ML_BQ - 1) / ML_BQ;
    int b = xcd_tile(blockIdx.x, gridDim.x);   // the blocks that read the same keys share an XCD's L2
    const int r0 = (b % nqb) * ML_BQ;
    b /= nqb;
    const int split = b % a.nsplit, hk = b / a.nsplit;
    const int nkt = a.kvp / ML_KT;

    // the key tiles some query of the block sees: the class rows of its tokens' 32-query tiles
    const int q_first = r0 / g / 32, q_last = (min(r0 + ML_BQ, rows) - 1) / g / 32;
    int * range = (int *)(smem + ML_SCALE + ML_BQ * 4);
    if (t == 0) { range[0] = nkt; range[1] = 0; }
    __syncthreads();
    {
        int lo = nkt, hi = 0;
        for (int kt = t; kt < nkt; kt += ML_THREADS) {
            int any = 0;
            bool full = true;
            for (int q = q_first; q <= q_last; q++) {
                const int x = a.cls[(int64_t)q * a.cls_stride + kt];
                any |= x;
                full = full && x == ML_FULL;
            }
            smem[ML_CLS + kt] = any == ML_SKIP ? ML_SKIP : full ? ML_FULL : ML_MIXED;
            if (any != ML_SKIP) {
                lo = min(lo, kt);
                hi = max(hi, kt + 1);
            }
        }
        if (lo < nkt) atomicMin(&range[0], lo);
        if (hi > 0) atomicMax(&range[1], hi);
    }

    // Q: wave w scales, normalises and rounds rows 16 w .. 16 w + 15 into the second tile buffer, 16 lanes a
    // row (the row max is then four exchanges inside 16 lanes for four rows at once; a whole wave a
    // row, 96 dependent exchanges in all, made this prologue 24 us)
    {
        uint8_t * qs = smem + ML_TILE;
#pragma unroll 2
        for (int p = 0; p < 4; p++) {
            const int r = 16 * wave + 4 * p + lg, row = r0 + r;
            const bool ok = row < rows;
            const int tok = ok ? row / g : 0, h = hk * g + (ok ? row % g : 0);
            const float * q = a.q + (int64_t)h * a.q_nb2 + (int64_t)tok * a.q_nb1;
            float4v v[9];
            float amax = 0.0f;
#pragma unroll
            for (int j = 0; j < 9; j++) v[j] = *(const float4v *)(q + 4 * (lc + 16 * j));
#pragma unroll
            for (int j = 0; j < 9; j++)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    v[j][e] = ok ? mul_rn(v[j][e], a.scale) : 0.0f;
                    amax = fmaxf(amax, fabsf(v[j][e]));
                }
#pragma unroll
            for (int x = 1; x < 16; x <<= 1) amax = fmaxf(amax, __shfl_xor(amax, x, WAVE));
            const float s = amax > 0.0f ? amax : 1.0f;
            const float inv = 1.0f / s;
#pragma unroll
            for (int j = 0; j < 9; j++) {
                const int c = lc + 16 * j;   // of the row's 144 float4
                u32x2 o;
                o[0] = pack2h(mul_rn(v[j][0], inv), mul_rn(v[j][1], inv));
                o[1] = pack2h(mul_rn(v[j][2], inv), mul_rn(v[j][3], inv));
                *(u32x2 *)(qs + r * ML_RB + (ml_chunk(r, c / 2) << 4) + 8 * (c % 2)) = o;
            }
            if (lc == 0) ((float *)(smem + ML_SCALE))[r] = s;
        }
    }
    ml_barrier_lgkm();
    const int lo = __builtin_amdgcn_readfirstlane(range[0]), hi = __builtin_amdgcn_readfirstlane(range[1]);
    const int per = (max(0, hi - lo) + a.nsplit - 1) / a.nsplit;
    const int tile0 = lo + split * per;
    const int nt = max(0, min(hi, tile0 + per) - tile0);

    // DMA: slot (row, physical chunk) of the tile holds the row's logical chunk; key rows past the
    // last one read the last one (their scores are masked)
    const __amdgpu_buffer_rsrc_t kr = __builtin_amdgcn_make_buffer_rsrc((void *)(a.k + (int64_t)hk * a.k_nb2), 0, 0x7FFFFFFF, 0x00020000);
    const int krow = (int)(2 * a.k_nb1);   // bytes
    // instruction q + 9 fetches the rows 32 further on, in the same chunks (9 * 256 slots are 32 rows, and the
    // swizzle repeats every 16)
    constexpr int HALF = ML_PER / 2;
    static_assert(HALF * ML_THREADS == 32 * 72, "half a tile is 32 rows");
    int koff[HALF];
#pragma unroll
    for (int q = 0; q < HALF; q++) {
        const int slot = q * ML_THREADS + t, r = slot / 72;
        koff[q] = r * krow + 16 * ml_chunk(r, slot % 72);
    }
    auto issue = [&](int i) {
        const int j0 = (tile0 + i) * ML_KT;
        uint8_t * dst = smem + (i & 1) * ML_TILE + wave * 1024;
        if (j0 + ML_KT <= a.KV) {
#pragma unroll
            for (int q = 0; q < ML_PER; q++)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(kr, (ml_lptr)(dst + q * 4096), 16, koff[q % HALF], (j0 + 32 * (q / HALF)) * krow, 0, 0);
            return;
        }
#pragma unroll
        for (int q = 0; q < ML_PER; q++) {
            const int r = (q % HALF * ML_THREADS + t) / 72;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(kr, (ml_lptr)(dst + q * 4096), 16,
                                                     koff[q % HALF] + (min(j0 + 32 * (q / HALF) + r, a.KV - 1) - r) * krow, 0, 0, 0);
        }
    };
    if (nt > 0) issue(0);

    // this wave's Q fragments: queries 32 qg + 16 i + lc, values 32 s + 8 lg ..
    half8 qf[2][ML_QS];
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const int r = 32 * qg + 16 * i + lc;
#pragma unroll
        for (int s = 0; s < ML_QS; s++) qf[i][s] = *(const half8 *)(smem + ML_TILE + r * ML_RB + (ml_chunk(r, 4 * s + lg) << 4));
    }
    // the first ML_Q1 steps' sit beside the output accumulators in AGPRs, which MFMAs read directly
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int s = 0; s < ML_Q1; s++) asm volatile("" : "+a"(qf[i][s]));
    if (t < ML_BQ) ((int *)(smem + ML_TOK))[t] = min(r0 + t, rows - 1) / g;   // the mask rows
    ml_barrier_lgkm();   // the second buffer is free
    if (nt > 1) {
        issue(1);
        ml_wait<ML_PER>();
    } else {
        ml_wait<0>();
    }
    __builtin_amdgcn_s_barrier();

    f32x4 o[8][4];   // [dim tile][query tile]: dims 128 w + 16 d + 4 lg + e, query 16 q + lc
#pragma unroll
    for (int d = 0; d < 8; d++)
#pragma unroll
        for (int q = 0; q < 4; q++) o[d][q] = f32x4{0, 0, 0, 0};
    // running maxima, times log2(e): of query 16 q + lc
    float m_run[4] = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
    float m_own[2] = {-INFINITY, -INFINITY};   // the same of this wave's score queries, 32 qg + 16 q + lc
    float lsum[2] = {0.0f, 0.0f};              // and this lane's share of their row sums
    const float inv_cap = SOFTCAP ? 1.0f / a.softcap : 0.0f;
    const float LOG2E = 1.4426950408889634f;
    // V^T source lanes: lane s of a 16-lane group points at 4 dims (4 (s % 4)) of one of 4 keys; read h
    // of group lg takes keys 8 lg + 4 (s / 8) + 2 h + (s / 4 % 2) of a 32-key step, which puts the 16
    // rows of one instruction on all chunk slots twice (the least for 512 bytes). Element 4 h + j of
    // the fragment is then key 8 lg + 4 (j / 2) + 2 h + j % 2, and P is stored in that order.
    const int vs = lane % 16;
    const int vkey = 8 * lg + 4 * (vs / 8) + (vs / 4) % 2;   // h = 0; its swizzle (key / 2 % 8) is even, h = 1's one more
    const uint32_t smem_lds = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const uint8_t *)smem;
    const uint32_t vbase0 = smem_lds + vkey * ML_RB + 256 * wave + 16 * ((vs % 4) / 2) + 8 * (vs % 2);
    const uint32_t vx = 16 * ((vkey >> 1) & 6);              // dim tile d sits (32 d) ^ vx bytes on
    // fragment reads at 32-deep step st: chunk 4 st + lg of a row, i.e. one of two lane offsets (st even,
    // odd) plus 128 bytes every two steps
    const int fx = (lc >> 1) & 7;
    const int fo0 = (lg ^ fx) << 4, fo1 = ((4 + lg) ^ fx) << 4;
    const int pw = ML_P + (32 * qg + lc) * 128 + 4 * (lg % 2);   // + the chunk of key tile kt
    const int pc0 = ((4 * kg + lg / 2) ^ fx) << 4, pc1 = ((4 * kg + 2 + lg / 2) ^ fx) << 4;

    // The accumulators stay in AGPRs: left alone the compiler keeps them in VGPRs between the rescale's
    // branch and the output MFMAs, where they push out the rest of the loop's values.
    auto pin_o = [&]() {
#pragma unroll
        for (int d = 0; d < 8; d++)
#pragma unroll
            for (int q = 0; q < 4; q++) asm volatile("" : "+a"(o[d][q]));
    };
    // a tile's class is read a tile early, and from LDS: a global load would wait for the K tile in
    // flight (loads retire in order)
    int cls_next = nt > 0 ? smem[ML_CLS + tile0] : 0;
    for (int i = 0; i < nt; i++) {
        const int tile = tile0 + i, j0 = tile * ML_KT;
        const uint8_t * ks = smem + (i & 1) * ML_TILE;
        const int cls = __builtin_amdgcn_readfirstlane(cls_next);
        if (cls != ML_SKIP) {
            // ---- S^T: keys 32 kg + 16 k + 4 lg + e, queries 32 qg + 16 q + lc ----
            f32x4 s[2][2];
#pragma unroll
            for (int k = 0; k < 2; k++)
#pragma unroll
                for (int q = 0; q < 2; q++) s[k][q] = f32x4{0, 0, 0, 0};
            {
                const uint8_t * kp0 = ks + (32 * kg + lc) * ML_RB + fo0, * kp1 = ks + (32 * kg + lc) * ML_RB + fo1;
                // the fragments of two steps are read four steps ahead of their MFMAs: with one wave a
                // SIMD nothing else covers an LDS read
                half8 kf[3][2][2];
                auto read2 = [&](int b) {
#pragma unroll
                    for (int j = 0; j < 2; j++) {
                        const int st = 2 * b + j;
                        const uint8_t * kp = (st % 2 ? kp1 : kp0) + 128 * (st / 2);
                        kf[b % 3][j][0] = *(const half8 *)kp;
                        kf[b % 3][j][1] = *(const half8 *)(kp + 16 * ML_RB);
                    }
                };
                read2(0);
                read2(1);
                ml_settle(s);
#pragma unroll
                for (int b = 0; b < ML_QS / 2; b++) {
                    if (b + 2 < ML_QS / 2) read2(b + 2);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int j = 0; j < 2; j++)
#pragma unroll
                        for (int k = 0; k < 2; k++)
#pragma unroll
                            for (int q = 0; q < 2; q++) {
                                const int st = 2 * b + j;
                                if (st == ML_Q1 && k + q == 0) ml_settle(s);
                                if (st < ML_Q1) ml_mfma_a(kf[b % 3][j][k], qf[q][st], s[k][q]);
                                else s[k][q] = ml_mfma(kf[b % 3][j][k], qf[q][st], s[k][q]);
                            }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            // scores in units of log 2: s * f with f = Q's row scale * log2(e); softcap, mask and the key
            // bound, where the tile has them, work on the scaled score first
            // (the row scales and mask rows come from LDS each time: held, they would spill, and a spill's
            // reload waits for the K tile in flight)
            float qsc[2], f[2];
#pragma unroll
            for (int q = 0; q < 2; q++) {
                qsc[q] = ((const float *)(smem + ML_SCALE))[32 * qg + 16 * q + lc];
                f[q] = qsc[q] * LOG2E;
            }
            const bool tail = j0 + ML_KT > a.KV;
            if (SOFTCAP || tail || (cls == ML_MIXED && a.mask)) {
#pragma unroll
                for (int q = 0; q < 2; q++) {
                    const int tk = ((const int *)(smem + ML_TOK))[32 * qg + 16 * q + lc];
                    const uint16_t * mrow = a.mask + (int64_t)tk * a.mask_nb1;
#pragma unroll
                    for (int k = 0; k < 2; k++) {
                        const int jk = j0 + 32 * kg + 16 * k + 4 * lg;   // first of this lane's 4 keys
                        f32x4 x = s[k][q] * qsc[q];
                        if (SOFTCAP)
#pragma unroll
                            for (int e = 0; e < 4; e++) x[e] = a.softcap * tanhf(x[e] * inv_cap);
                        if (cls == ML_MIXED && a.mask) {
                            if (jk + 3 < a.KV) {
                                const u32x2 mm = *(const u32x2 *)(mrow + jk);
                                x[0] += h2f_bits((uint16_t)(mm[0] & 0xFFFFu));
                                x[1] += h2f_bits((uint16_t)(mm[0] >> 16));
                                x[2] += h2f_bits((uint16_t)(mm[1] & 0xFFFFu));
                                x[3] += h2f_bits((uint16_t)(mm[1] >> 16));
                            } else {
#pragma unroll
                                for (int e = 0; e < 4; e++)
                                    if (jk + e < a.KV) x[e] += h2f_bits(mrow[jk + e]);
                            }
                        }
                        if (tail)
#pragma unroll
                            for (int e = 0; e < 4; e++)
                                if (jk + e >= a.KV) x[e] = -INFINITY;
                        s[k][q] = x;
                    }
                    f[q] = LOG2E;
                }
            }
#pragma unroll
            for (int q = 0; q < 2; q++) {
                float m = fmaxf(fmaxf(s[0][q][0], s[0][q][1]), s[0][q][2]);
                m = fmaxf(fmaxf(m, s[0][q][3]), s[1][q][0]);
                m = fmaxf(fmaxf(m, s[1][q][1]), s[1][q][2]);
                m = ml_max_groups(fmaxf(m, s[1][q][3])) * f[q];
                if (lg == 0) ((float *)(smem + ML_MAX))[(32 * qg + 16 * q + lc) * 2 + kg] = m;
            }
            ml_barrier_lgkm();
            // ---- the running max of every row, moved only when a score passes it by 2^8 (in P) ----
            float mt[4];
            bool up = false;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const float2v x = *(const float2v *)(smem + ML_MAX + (16 * q + lc) * 8);
                mt[q] = fmaxf(x[0], x[1]);
                up |= mt[q] > m_run[q] + ML_LAZY;
            }
            pin_o();
            if (__any(up)) {   // the same in every wave: all see all 64 rows
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const float mn = fmaxf(m_run[q], mt[q]);
                    const float al = m_run[q] == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m_run[q] - mn);
                    m_run[q] = mn;
#pragma unroll
                    for (int d = 0; d < 8; d++) {   // one at a time through VGPRs
                        o[d][q] *= al;
                        asm volatile("" : "+a"(o[d][q]));
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
#pragma unroll
                for (int q = 0; q < 2; q++) {
                    const float2v x = *(const float2v *)(smem + ML_MAX + (32 * qg + 16 * q + lc) * 8);
                    const float mn = fmaxf(m_own[q], fmaxf(x[0], x[1]));
                    lsum[q] *= m_own[q] == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m_own[q] - mn);
                    m_own[q] = mn;
                }
            }
            // ---- P to LDS: this lane's 4 keys are 2 + 2 of the V^T order ----
#pragma unroll
            for (int q = 0; q < 2; q++) {
                const float mb = m_own[q] == -INFINITY ? 0.0f : m_own[q];
#pragma unroll
                for (int k = 0; k < 2; k++) {
                    float p[4];
#pragma unroll
                    for (int e = 0; e < 4; e++) p[e] = __builtin_amdgcn_exp2f(fmaf(s[k][q][e], f[q], -mb));
                    const uint32_t p01 = pack2h(p[0], p[1]), p23 = pack2h(p[2], p[3]);
                    const half2v one2 = {(_Float16)1.0f, (_Float16)1.0f};
                    lsum[q] = __builtin_amdgcn_fdot2(__builtin_bit_cast(half2v, p01), one2, lsum[q], false);
                    lsum[q] = __builtin_amdgcn_fdot2(__builtin_bit_cast(half2v, p23), one2, lsum[q], false);
                    uint8_t * pr = smem + pw + 2048 * q + (k ? pc1 : pc0);
                    *(uint32_t *)pr = p01;
                    *(uint32_t *)(pr + 8) = p23;
                }
            }
            ml_barrier_lgkm();
            pin_o();
            // ---- O^T += V^T . P^T: four groups of 32 keys (g / 2) x 64 dims (g % 2), the fragments of
            // a group read under the MFMAs of the one before ----
            half8 pf[4], vf[2][4];
            auto read_v = [&](int g) {
#pragma unroll
                for (int d = 0; d < 4; d++) {   // h = 1: two rows on, its chunk one over
                    const uint32_t x = ((32u * d) ^ vx) + (uint32_t)((i & 1) * ML_TILE + 32 * (g / 2) * ML_RB + 128 * (g % 2));
                    const half4v lo = ml_tr_read(vbase0 + x), hi = ml_tr_read((vbase0 ^ 16) + x + 2 * ML_RB);
                    vf[g % 2][d] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
                }
            };
            auto read_p = [&](int st) {
#pragma unroll
                for (int q = 0; q < 4; q++) pf[q] = *(const half8 *)(smem + ML_P + (16 * q + lc) * 128 + (st ? fo1 : fo0));
            };
            read_p(0);
            read_v(0);
#pragma unroll
            for (int g = 0; g < 4; g++) {
                if (g < 3) read_v(g + 1);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int d = 0; d < 4; d++)
#pragma unroll
                    for (int q = 0; q < 4; q++) o[4 * (g % 2) + d][q] = ml_mfma(vf[g % 2][d], pf[q], o[4 * (g % 2) + d][q]);
                __builtin_amdgcn_sched_barrier(0);
                if (g == 1) read_p(1);
            }
        }
        pin_o();
        cls_next = smem[ML_CLS + min(tile + 1, nkt - 1)];
        // the next tile has landed for every wave, and every wave is done with this one
        ml_wait<0>();
        __builtin_amdgcn_s_barrier();
        if (i + 2 < nt) issue(i + 2);
    }

    // ---- row sums: over the lane groups, then the two key groups through LDS ----
#pragma unroll
    for (int q = 0; q < 2; q++) {
        float l = lsum[q] + __shfl_xor(lsum[q], 16, WAVE);
        l += __shfl_xor(l, 32, WAVE);
        if (lg == 0) ((float *)(smem + ML_MAX))[(32 * qg + 16 * q + lc) * 2 + kg] = l;
    }
    ml_barrier_lgkm();
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const float2v x = *(const float2v *)(smem + ML_MAX + (16 * q + lc) * 8);
        const float l = x[0] + x[1];
        const int row = r0 + 16 * q + lc;
        if (row >= rows) continue;
        const int tok = row / g, h = hk * g + row % g;
        float * dst;
        float f = 1.0f;
        if (a.nsplit == 1) {
            dst = a.dst + (int64_t)tok * a.dst_nb2 + (int64_t)h * a.dst_nb1;
            f = l > 0.0f ? 1.0f / l : 0.0f;
        } else {   // unnormalised partial; fa_combine merges them
            const int64_t pr = (int64_t)split * a.T * a.H + (int64_t)tok * a.H + h;
            dst = a.part_o + pr * ML_DV;
            if (wave == 0 && lg == 0) {
                a.part_ml[2 * pr] = m_run[q] / LOG2E;
                a.part_ml[2 * pr + 1] = l;
            }
        }
#pragma unroll
        for (int d = 0; d < 8; d++) *(float4v *)(dst + 128 * wave + 16 * d + 4 * lg) = o[d][q] * f;
    }
#endif
}

int fa_mla_blocks(const FaArgs & a) { return a.HK * ((a.H / a.HK * a.T + ML_BQ - 1) / ML_BQ); }

hipError_t launch_fa_mla(const FaArgs & a, bool prep, hipStream_t st) {
    const int nb = fa_mla_blocks(a) * a.nsplit;
    if (nb <= 0) return hipSuccess;
    hipError_t e = hipSuccess;
    if (prep && (e = launch_fa_prep(a, st)) != hipSuccess) return e;
    static bool attr = false;
    if (!attr) {
        for (const void * k : {(const void *)fa_mla_kernel<false>, (const void *)fa_mla_kernel<true>})
            if ((e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, ML_LDS)) != hipSuccess) return e;
        attr = true;
    }
    if (a.softcap != 0.0f) hipLaunchKernelGGL(fa_mla_kernel<true>, dim3(nb), dim3(ML_THREADS), ML_LDS, st, a);
    else hipLaunchKernelGGL(fa_mla_kernel<false>, dim3(nb), dim3(ML_THREADS), ML_LDS, st, a);
    if ((e = hipGetLastError()) != hipSuccess || a.nsplit == 1) return e;
    return launch_fa_combine(a, st);
}

}  // namespace mx
