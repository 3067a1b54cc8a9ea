// SPDX-License-Identifier: MIT
// The prefill GEMM family for gfx950.
//
//   pack_act      F32 activations [M][K] -> fp16 [M][K] divided by a per-row scale (the row's
//                 max |x|), plus the scales. This is the activation contract of the reference
//                 (rk_pack_act_row, ggml-rocket.cpp:1451-1475): C = s * ((A/s) . W).
//   gemm          C[M][N] (F32) = scale[m] * sum_k A16[m][k] * W[n][k], W in any of the HBM
//                 weight formats of mx_weights.h, decoded to fp16 while it is staged into LDS.
//                 fp16 MFMA (v_mfma_f32_32x32x16_f16) with fp32 accumulation, F32 written
//                 straight from the accumulators: no fp16 output surface.
//                 Up to four weights that share A run in one launch over their concatenated N
//                 (the fused QKV / gate-up groups of ggml-rocket.cpp:4956-5160).
//   dequant_f16   a weight panel -> fp16 [rows][K] (the resident-fp16 form, "prepacked-q").
//   pack_weight   a ggml Q8_0 / Q6_K / MXFP4 payload -> its split HBM layout (mx_weights.h).
//
// The GEMM kernels: a register-staged one that decodes any weight format into LDS (gemm_kernel);
// for fp16 weights two that move both operands into LDS by DMA, gemm_f16_1w_kernel for tiled
// weights and gemm_f16_kernel (with its two-width variant gemm_f16_cols_kernel) for row-major
// ones; for Q4_K and Q8_0 one that moves every operand by DMA and decodes from LDS
// (gemm_q4k_kernel); and for M <= 128 one that decodes the weight straight into MFMA operands
// (gemm_skinny_kernel). The launcher picks a kernel and tile configuration per call from the
// output shape.

#include <algorithm>
#include <cmath>

#include "mx_weights.h"
#include "mx_kernels_impl.h"

namespace mx {

// ---------------------------------------------------------------------------------------------
// activation pack: one 256-thread block per row. A row of up to PACK_REG_MAX floats is read
// once into registers (all loads in flight together), reduced, scaled and written; longer rows
// take a second pass over memory.
// ---------------------------------------------------------------------------------------------
constexpr int PACK_THREADS = 256;
constexpr int PACK_VEC = 16;                                 // float4 per thread held in registers
constexpr int PACK_REG_MAX = PACK_THREADS * PACK_VEC * 4;    // 16384 floats

// TL: write A16 in the tiled layout (tiled_index over M rows) instead of rows of lda.
// ZC (optional): an F32 output whose row m (ZN values) the block also clears, for a GEMM that
// adds its K splits into it; one launch fewer than a separate fill.
template <bool TL>
__global__ void __launch_bounds__(PACK_THREADS) pack_act_kernel(const float * __restrict__ X, int64_t ldx,
                                                                int M, int K, uint16_t * __restrict__ A16,
                                                                int64_t lda, float * __restrict__ scales,
                                                                float * __restrict__ ZC, int64_t ldzc, int ZN) {
    __shared__ float red[PACK_THREADS / WAVE];
    const int t = threadIdx.x, lane = t % WAVE, wave = t / WAVE;
    const int m = blockIdx.x;
    if (ZC) {
        float * zrow = ZC + (int64_t)m * ldzc;
        int c0 = 0;
        if ((reinterpret_cast<uintptr_t>(zrow) & 15) == 0) {
            for (int c = 4 * t; c + 3 < ZN; c += 4 * PACK_THREADS) *(float4v *)(zrow + c) = float4v{0, 0, 0, 0};
            c0 = ZN & ~3;
        }
        for (int c = c0 + t; c < ZN; c += PACK_THREADS) zrow[c] = 0.0f;
    }
    const int n4 = K / 4;
    // the destination of the 4 values starting at column 4c
    auto dst = [&](int c) -> uint16_t * {
        return TL ? A16 + tiled_index(m, 4 * c, K) : A16 + (int64_t)m * lda + 4 * c;
    };
    const float * x = X + (int64_t)m * ldx;
    float4v v[PACK_VEC];
    float amax = 0.0f;
#pragma unroll
    for (int i = 0; i < PACK_VEC; i++) {
        const int c = t + i * PACK_THREADS;
        v[i] = c < n4 ? *(const float4v *)(x + 4 * c) : float4v{0, 0, 0, 0};
        amax = fmaxf(amax, fmaxf(fmaxf(fabsf(v[i][0]), fabsf(v[i][1])), fmaxf(fabsf(v[i][2]), fabsf(v[i][3]))));
    }
    for (int c = t + PACK_VEC * PACK_THREADS; c < n4; c += PACK_THREADS) {
        const float4v w = *(const float4v *)(x + 4 * c);
        amax = fmaxf(amax, fmaxf(fmaxf(fabsf(w[0]), fabsf(w[1])), fmaxf(fabsf(w[2]), fabsf(w[3]))));
    }
    amax = wave_max(amax);
    if (lane == 0) red[wave] = amax;
    __syncthreads();
    amax = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    const float s = amax > 0.0f ? amax : 1.0f;
    const float inv = 1.0f / s;
    // x * inv is rounded to f32 and then to fp16, as the CPU pack does: mul_rn keeps the compiler
    // from folding the product into the conversion (v_fma_mix rounds once)
#pragma unroll
    for (int i = 0; i < PACK_VEC; i++) {
        const int c = t + i * PACK_THREADS;
        if (c < n4) {
            u32x2 o;
            o[0] = pack2h(mul_rn(v[i][0], inv), mul_rn(v[i][1], inv));
            o[1] = pack2h(mul_rn(v[i][2], inv), mul_rn(v[i][3], inv));
            *(u32x2 *)dst(c) = o;
        }
    }
    for (int c = t + PACK_VEC * PACK_THREADS; c < n4; c += PACK_THREADS) {
        const float4v w = *(const float4v *)(x + 4 * c);
        u32x2 o;
        o[0] = pack2h(mul_rn(w[0], inv), mul_rn(w[1], inv));
        o[1] = pack2h(mul_rn(w[2], inv), mul_rn(w[3], inv));
        *(u32x2 *)dst(c) = o;
    }
    if (t == 0) scales[m] = s;
}

// Rows of up to PACK_WAVE_K values: one wave a row (pack_row_wave), four rows a block; for
// short rows (an expert's 768- or 2048-wide activations, thousands of them) the block form's
// barrier and its idle threads dominate.
template <bool TL>
__global__ void __launch_bounds__(PACK_THREADS) pack_act_wave_kernel(const float * __restrict__ X, int64_t ldx,
                                                                     int M, int K, uint16_t * __restrict__ A16,
                                                                     int64_t lda, float * __restrict__ scales,
                                                                     float * __restrict__ ZC, int64_t ldzc, int ZN) {
    const int lane = threadIdx.x % WAVE;
    const int m = blockIdx.x * (PACK_THREADS / WAVE) + threadIdx.x / WAVE;
    if (m >= M) return;   // the whole wave
    if (ZC) {
        float * zrow = ZC + (int64_t)m * ldzc;
        int c0 = 0;
        if ((reinterpret_cast<uintptr_t>(zrow) & 15) == 0) {
            for (int c = 4 * lane; c + 3 < ZN; c += 4 * WAVE) *(float4v *)(zrow + c) = float4v{0, 0, 0, 0};
            c0 = ZN & ~3;
        }
        for (int c = c0 + lane; c < ZN; c += WAVE) zrow[c] = 0.0f;
    }
    pack_row_wave<TL>(X + (int64_t)m * ldx, m, K, A16, lda, scales, lane);
}

// The widest row the wave form packs: 2048 values (measured: 8.5% faster for the 4096 rows of 768
// of an expert down projection, within 3% either way for 512 rows of 4096; MI355X_PACK_WAVE_K
// overrides, for tests and tuning, up to 4096; 0 keeps every row on the block form).
static int pack_wave_k() {
    const char * e = getenv("MI355X_PACK_WAVE_K");
    return (e && *e) ? std::min(atoi(e), PACK_WAVE_K) : 2048;
}

// ---------------------------------------------------------------------------------------------
// GEMM
//
// Block = 256 threads (4 waves in a WM x WN grid), output tile BM x BN, K staged BK = 64 at a
// time through a double-buffered, XOR-swizzled LDS tile. Global loads run R slabs ahead in a ring
// of register sets (the loop is unrolled by R so the sets are static registers): slab k+R is
// requested while slab k is multiplied, and slab k+1 is written to LDS only after that, which
// hides HBM latency behind R-1 slabs of MFMA work.
// KSPLIT > 1 splits K between that many blocks that add their parts atomically into a zeroed
// output; KSPLIT = 0 takes the split count from the launcher (args.ksplit), which sizes it to fill
// the chip when the output has few tiles (a skinny M: 32 rows of a 3072-wide output are 24
// tiles). Two addends sum the same in either order; with more, the rounding of the sum depends
// on the order the blocks finish in.
// ---------------------------------------------------------------------------------------------
constexpr int BK = 64;
constexpr int GEMM_THREADS = 256;

template <int BM, int BN, int WM, int WN, int R>
struct GemmCfg {
    static constexpr int TM = BM / WM, TN = BN / WN;        // wave tile
    static constexpr int MI = TM / 32, NJ = TN / 32;        // MFMA blocks per wave
    static constexpr int A_CHUNKS = BM * (BK / 8) / GEMM_THREADS;   // 16-byte chunks per thread
    static constexpr int B_ITEMS = BN * 2 / GEMM_THREADS;           // (row, half) items per thread
    static constexpr int A_BYTES = BM * BK * 2, B_BYTES = BN * BK * 2;
    static constexpr int STAGE = A_BYTES + B_BYTES;
    static constexpr int LDS = 2 * STAGE;
    static_assert(WM * WN == 4, "4 waves");
    static_assert(A_CHUNKS >= 1 && B_ITEMS >= 1, "tile too small");
};

// One pipeline stage in registers: raw loads plus whether each item is real; the masking is
// applied when the stage is written to LDS, so the loads stay in flight until then.
template <int WT, int NA, int NB>
struct Slab {
    u32x4 a[NA];
    bool a_ok[NA];
    WLoad<WT> b[NB];
};

template <int WT, class C>
__device__ __forceinline__ void slab_load(Slab<WT, C::A_CHUNKS, C::B_ITEMS> & s, const GemmArgs & args,
                                          const GemmGroup & G, int m0, int n0, int64_t k0, int t) {
    const int M = args.M, K = args.K;
#pragma unroll
    for (int i = 0; i < C::A_CHUNKS; i++) {
        const int c = t + i * GEMM_THREADS;
        const int r = m0 + c / 8;
        const int64_t k = k0 + 8 * (c % 8);
        s.a_ok[i] = r < M && k < K;
        s.a[i] = *(const u32x4 *)(args.A + (int64_t)(r < M ? r : M - 1) * args.lda + (k < K ? k : 0));
    }
    const uint8_t * W = (const uint8_t *)G.W;
#pragma unroll
    for (int i = 0; i < C::B_ITEMS; i++) {
        const int it = t + i * GEMM_THREADS;
        const int n = n0 + it / 2;
        const bool ok = n < G.N;
        s.b[i].load(W, G.rows_total, K, G.row0 + (ok ? n : G.N - 1), k0, it % 2, ok);
    }
}

template <int WT, class C>
__device__ __forceinline__ void slab_store(const Slab<WT, C::A_CHUNKS, C::B_ITEMS> & s, uint8_t * st, int t) {
#pragma unroll
    for (int i = 0; i < C::A_CHUNKS; i++) {
        const int c = t + i * GEMM_THREADS;
        *(u32x4 *)(st + swz<8>(c / 8, c % 8)) = s.a_ok[i] ? s.a[i] : u32x4{0, 0, 0, 0};
    }
    uint8_t * bs = st + C::A_BYTES;
#pragma unroll
    for (int i = 0; i < C::B_ITEMS; i++) {
        const int it = t + i * GEMM_THREADS;
        const int r = it / 2;
        u32x4 out[4];
        int run0, run1;
        s.b[i].decode(it % 2, out, run0, run1);
        *(u32x4 *)(bs + swz<8>(r, run0 / 8)) = out[0];
        *(u32x4 *)(bs + swz<8>(r, run0 / 8 + 1)) = out[1];
        *(u32x4 *)(bs + swz<8>(r, run1 / 8)) = out[2];
        *(u32x4 *)(bs + swz<8>(r, run1 / 8 + 1)) = out[3];
    }
}

template <class C>
__device__ __forceinline__ void mma_slab(const uint8_t * st, int wm, int wn, int lane,
                                         float16v (&acc)[C::MI][C::NJ]) {
    const uint8_t * As = st;
    const uint8_t * Bs = st + C::A_BYTES;
    const int lr = lane % 32, lg = lane / 32;
#pragma unroll
    for (int ks = 0; ks < BK / 16; ks++) {
        const int c = 2 * ks + lg;
        half8 a[C::MI], b[C::NJ];
#pragma unroll
        for (int i = 0; i < C::MI; i++) a[i] = *(const half8 *)(As + swz<8>(wm * C::TM + i * 32 + lr, c));
#pragma unroll
        for (int j = 0; j < C::NJ; j++) b[j] = *(const half8 *)(Bs + swz<8>(wn * C::TN + j * 32 + lr, c));
#pragma unroll
        for (int i = 0; i < C::MI; i++)
#pragma unroll
            for (int j = 0; j < C::NJ; j++) acc[i][j] = mfma32(a[i], b[j], acc[i][j]);
    }
}

// Where a K-split block writes: with partials (a split past two ways) its split's slab of them,
// row stride ldp, group g's columns from pcol; otherwise the group's own output, which it adds
// into when the split is two ways.
__device__ __forceinline__ void split_target(const GemmArgs & a, int g, int split, float *& Cp, int64_t & ldc) {
    if (!a.part) return;
    int64_t pcol = a.g[0].pcol;
#pragma unroll
    for (int i = 1; i < GEMM_MAX_GROUPS; i++)
        if (i == g) pcol = a.g[i].pcol;
    Cp = a.part + (int64_t)split * a.M * a.ldp + pcol;
    ldc = a.ldp;
}

template <int WT, int BM, int BN, int WM, int WN, int R, int KSPLIT>
__global__ void __launch_bounds__(GEMM_THREADS)
__attribute__((amdgpu_waves_per_eu((BM == 128 && BN == 128) ? 2 : 1, (BM == 128 && BN == 128) ? 2 : 1)))
gemm_kernel(GemmArgs args) {
    // waves_per_eu pins the register budget to the occupancy the LDS allows anyway (2 blocks of
    // a 128x128 tile per CU, 1 of the larger tiles), so the scheduler does not sink the prefetch
    // loads next to their use to save registers.
    using C = GemmCfg<BM, BN, WM, WN, R>;
    extern __shared__ __align__(16) uint8_t smem[];

    const int t = threadIdx.x, lane = t % WAVE, wave = t / WAVE;
    const int wm = wave / WN, wn = wave % WN;

    // block -> (k split, global n tile, m tile); m is the fast index so the blocks that share a
    // weight panel are neighbours (and, after xcd_tile, on one XCD)
    const int nblocks = gridDim.x;
    const int ks = KSPLIT > 0 ? KSPLIT : args.ksplit;   // 0: the launcher's split count
    int tile = xcd_tile(blockIdx.x, nblocks);
    const int split = tile % ks;
    tile /= ks;
    const int mt = tile % args.m_tiles, nt = tile / args.m_tiles;
    int g = 0;
#pragma unroll
    for (int i = 1; i < GEMM_MAX_GROUPS; i++)
        if (i < args.ng && nt >= args.g[i].ntile_begin) g = i;
    GemmGroup G;
    G.W = args.g[0].W; G.rows_total = args.g[0].rows_total; G.row0 = args.g[0].row0; G.N = args.g[0].N;
    G.C = args.g[0].C; G.ldc = args.g[0].ldc; G.ntile_begin = args.g[0].ntile_begin;
#pragma unroll
    for (int i = 1; i < GEMM_MAX_GROUPS; i++)
        if (i == g) {
            G.W = args.g[i].W; G.rows_total = args.g[i].rows_total; G.row0 = args.g[i].row0; G.N = args.g[i].N;
            G.C = args.g[i].C; G.ldc = args.g[i].ldc; G.ntile_begin = args.g[i].ntile_begin;
        }
    split_target(args, g, split, G.C, G.ldc);
    const int n0 = (nt - G.ntile_begin) * BN;
    const int m0 = mt * BM;

    const int nk_all = (args.K + BK - 1) / BK;
    const int per = (nk_all + ks - 1) / ks;
    const int kb = split * per;
    const int nk = max(0, min(nk_all, kb + per) - kb);

    float16v acc[C::MI][C::NJ];
#pragma unroll
    for (int i = 0; i < C::MI; i++)
#pragma unroll
        for (int j = 0; j < C::NJ; j++)
#pragma unroll
            for (int e = 0; e < 16; e++) acc[i][j][e] = 0.0f;

    // Two register stages. Step kk: request slab kk+2 into ring[kk&1] (its previous contents,
    // slab kk, are already in LDS), multiply slab kk from LDS, then write slab kk+1 (requested a
    // step earlier) into the other LDS buffer. Slab indices past the end are clamped to the last
    // slab, so every step issues the same loads and stores with no branch around them (a load
    // behind a branch makes the compiler wait for every outstanding load); the extra slab written
    // on the last step lands in the buffer nobody reads again.
    static_assert(R == 2, "two register stages");
    Slab<WT, C::A_CHUNKS, C::B_ITEMS> ring[2];
    const int last = kb + (nk > 0 ? nk - 1 : 0);
    auto slab_k0 = [&](int kk) -> int64_t { return (int64_t)min(kb + kk, last) * BK; };
    auto step = [&](int kk, Slab<WT, C::A_CHUNKS, C::B_ITEMS> & mine, Slab<WT, C::A_CHUNKS, C::B_ITEMS> & next) {
        slab_load<WT, C>(mine, args, G, m0, n0, slab_k0(kk + 2), t);
        mma_slab<C>(smem + (kk & 1) * C::STAGE, wm, wn, lane, acc);
        slab_store<WT, C>(next, smem + ((kk + 1) & 1) * C::STAGE, t);
        __syncthreads();
    };
    if (nk > 0) {
        slab_load<WT, C>(ring[0], args, G, m0, n0, slab_k0(0), t);
        slab_load<WT, C>(ring[1], args, G, m0, n0, slab_k0(1), t);
        slab_store<WT, C>(ring[0], smem, t);
        __syncthreads();
        int kk = 0;
        for (; kk + 2 <= nk; kk += 2) {
            step(kk, ring[0], ring[1]);
            step(kk + 1, ring[1], ring[0]);
        }
        if (kk < nk) step(kk, ring[0], ring[1]);
    }

    // epilogue: C = scale[m] * acc
    const int lr = lane % 32, lg = lane / 32;
    scale_rows(acc, args.scales, m0 + wm * C::TM, lg, args.M);
#pragma unroll
    for (int i = 0; i < C::MI; i++) {
#pragma unroll
        for (int e = 0; e < 16; e++) {
            const int r = m0 + wm * C::TM + i * 32 + 8 * (e / 4) + 4 * lg + (e % 4);
            if (r >= args.M) continue;
            float * crow = G.C + (int64_t)r * G.ldc;
#pragma unroll
            for (int j = 0; j < C::NJ; j++) {
                const int n = n0 + wn * C::TN + j * 32 + lr;
                if (n < G.N) {
                    if (ks == 1 || args.part) crow[n] = acc[i][j][e];
                    else unsafeAtomicAdd(crow + n, acc[i][j][e]);
                }
            }
        }
    }
}

// ---------------------------------------------------------------------------------------------
// Skinny GEMM (M <= 128): a launch this narrow is bound by latency, not by MFMA rate or HBM, so the
// weight goes from HBM straight into registers and is decoded there into MFMA operands (no LDS round
// trip for the weight). A block is KW ways along K of NW waves over NW*32 weight rows, and a run of K
// groups of CH 64-deep chunks that its ways take in turn (way w groups w, w + KW, ..). One way alone
// leaves one wave a SIMD, whose chain load -> decode -> LDS read -> MFMA nothing hides, and a wave by
// itself issues VALU at half rate; more blocks instead write more slabs of partials. The ways' sums
// meet in LDS, added in way order. Lane (r, g) of a wave loads
// decoder item g of each chunk for weight row r, and the 32 values it decodes (two runs of 16
// consecutive k) are its B operands for the chunk's four 16-deep MFMA steps, so lane (r, g) of
// the A operand reads the same k from activation row r. Per group the activation slice
// [32 MT][64 CH] fp16 sits in LDS (16-byte chunks XOR-swizzled by row), double-buffered per way, and
// the weight of the next group is in flight in a second register set while this one is multiplied.
// Issue order matters: one vmcnt counter covers every load in issue order, so each step issues
// the next group's activation loads before its weight loads (their LDS store then waits for them
// alone, not for the weight), and nothing consumes a loaded value before the step's compute: the
// activation's row / K mask is applied at its LDS store, since a select right after a load would
// make the compiler wait for that load before issuing the next. Past the block's last group the
// loads re-fetch it and are never multiplied (or, where another way still has a group, as zeros), so
// the loop body has no branch between a load and its use. The weights are decoded by the packed-fp16
// decoders (decode_fast: a quarter to a half of the VALU instructions of the exact decode). Blocks
// split K too: past two ways each writes its slab of the partials, summed in split order by
// reduce_splits_kernel; two ways add into a zeroed output.
// Whole calls on cold weights, us, one way of four waves -> this: Q4_K 8192 x 3072 M 8 / 64 / 90 / 128
// 17.0 / 24.1 / 31.5 / 33.3 -> 13.2 / 18.4 / 22.7 / 27.5; 14336 x 4096 M 64 35.2 -> 28.5; 28672 x 4096 M 64
// 53.6 -> 41.5; Q8_0 3072 x 3072 M 32 15.5 -> 14.9. A weight staged by LDS DMA (a kernel that was here for
// Q6_K and Q8_0) was slower: Q6_K 8192 x 3072 M 32 24.9 -> 18.4, Q8_0 M 128 32.2 -> 28.1. One way, two blocks
// a CU, stays at the widths, depths and types skinny_shape names (up to 32 rows).
// ---------------------------------------------------------------------------------------------
constexpr int SK_MAX_M = 128;

template <int MT, int CH, int NW, int KW>
constexpr int skinny_lds() {
    const int ring = KW * 2 * 32 * MT * 8 * CH * 16;
    const int merge = KW > 1 ? KW * NW * MT * 16 * WAVE * 4 : 0;
    return ring > merge ? ring : merge;
}
// waves a SIMD: the block's own, or two blocks' of one K way
constexpr int skinny_waves(int nw, int kw) { return kw == 1 ? 2 : nw * kw / 4; }

template <int WT, int MT, int CH, int NW, int KW>
__global__ void __launch_bounds__(NW * KW * WAVE)
__attribute__((amdgpu_waves_per_eu(skinny_waves(NW, KW), skinny_waves(NW, KW))))
gemm_skinny_kernel(GemmArgs args, int groups_per_block) {
    constexpr int CPR = 8 * CH;               // 16-byte chunks per activation row of the slice
    constexpr int ACH = 32 * MT * CPR;        // 16-byte chunks of the slice
    constexpr int APT = ACH / (NW * WAVE);    // per thread
    constexpr int SLICE = ACH * 16;
    static_assert(ACH % (NW * WAVE) == 0, "slice split");
    extern __shared__ __align__(16) uint8_t sk_smem[];

    // t, wave: within this thread's K way, which has its own pair of activation slices
    const int way = __builtin_amdgcn_readfirstlane(threadIdx.x / (NW * WAVE));
    const int t = threadIdx.x % (NW * WAVE), lane = t % WAVE, wave = t / WAVE;
    uint8_t * const sa = sk_smem + way * (2 * SLICE);
    const int lr = lane % 32, lg = lane / 32;
    const int ks = args.ksplit;
    const int split = blockIdx.x % ks;
    const int nt = blockIdx.x / ks;
    int g = 0;
#pragma unroll
    for (int i = 1; i < GEMM_MAX_GROUPS; i++)
        if (i < args.ng && nt >= args.g[i].ntile_begin) g = i;
    GemmGroup G;
    G.W = args.g[0].W; G.rows_total = args.g[0].rows_total; G.row0 = args.g[0].row0; G.N = args.g[0].N;
    G.C = args.g[0].C; G.ldc = args.g[0].ldc; G.ntile_begin = args.g[0].ntile_begin;
#pragma unroll
    for (int i = 1; i < GEMM_MAX_GROUPS; i++)
        if (i == g) {
            G.W = args.g[i].W; G.rows_total = args.g[i].rows_total; G.row0 = args.g[i].row0; G.N = args.g[i].N;
            G.C = args.g[i].C; G.ldc = args.g[i].ldc; G.ntile_begin = args.g[i].ntile_begin;
        }
    split_target(args, g, split, G.C, G.ldc);
    const int n = (nt - G.ntile_begin) * (32 * NW) + 32 * wave + lr;   // this lane's weight row
    const bool okn = n < G.N;
    const int64_t row = G.row0 + (okn ? n : G.N - 1);
    const int nchunks = (args.K + 63) / 64;
    const int ngroups = (nchunks + CH - 1) / CH;
    const int gb = split * groups_per_block;                             // first group of the block
    const int gn = max(0, min(ngroups, gb + groups_per_block) - gb);    // groups of the block
    const int glast = gb + max(gn, 1) - 1;

    // rows past M and k past K read as zero: the load takes a valid address and the mask is
    // applied when the value is stored to LDS (where the load is waited for anyway), so no
    // wait sits between one load and the next
    auto load_a = [&](u32x4 (&av)[APT], uint32_t & amask, int grp) {
        const int64_t kb = (int64_t)min(grp, glast) * CH * 64;
        amask = 0;
#pragma unroll
        for (int i = 0; i < APT; i++) {
            const int q = t + i * NW * WAVE, r = q / CPR, c = q % CPR;
            const int64_t k = kb + 8 * c;
            const bool ok = r < args.M && k < args.K && grp <= glast;
            av[i] = *(const u32x4 *)(args.A + (ok ? (int64_t)r * args.lda + k : 0));
            amask |= ok ? (1u << i) : 0u;
        }
    };
    auto store_a = [&](const u32x4 (&av)[APT], uint32_t amask, int buf) {
#pragma unroll
        for (int i = 0; i < APT; i++) {
            const int q = t + i * NW * WAVE, r = q / CPR, c = q % CPR;
            const bool ok = (amask >> i) & 1u;
            const u32x4 v = {ok ? av[i][0] : 0u, ok ? av[i][1] : 0u, ok ? av[i][2] : 0u, ok ? av[i][3] : 0u};
            *(u32x4 *)(sa + buf * SLICE + (r * CPR + (c ^ (r & 7))) * 16) = v;
        }
    };
    auto load_w = [&](WLoad<WT> (&w)[CH], int grp) {
        const bool live = okn && grp <= glast && gn > 0;
        const int c0 = min(grp, glast) * CH;
#pragma unroll
        for (int c = 0; c < CH; c++) {
            const int cc = c0 + c;
            w[c].load((const uint8_t *)G.W, G.rows_total, args.K, row, (int64_t)min(cc, nchunks - 1) * 64, lg,
                      live && cc < nchunks);
        }
    };
    float16v acc[MT][1];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int e = 0; e < 16; e++) acc[i][0][e] = 0.0f;
    auto compute = [&](const WLoad<WT> (&w)[CH], int buf) {
#pragma unroll
        for (int c = 0; c < CH; c++) {
            u32x4 b[4];
            int run0, run1;
            w[c].decode_fast(lg, b, run0, run1);
#pragma unroll
            for (int s = 0; s < 4; s++) {
                const int ch = 8 * c + (s < 2 ? run0 + 8 * s : run1 + 8 * (s - 2)) / 8;   // slice chunk
                const half8 bf = __builtin_bit_cast(half8, b[s]);
#pragma unroll
                for (int i = 0; i < MT; i++) {
                    const int r = 32 * i + lr;
                    const half8 af = *(const half8 *)(sa + buf * SLICE + (r * CPR + (ch ^ (r & 7))) * 16);
                    acc[i][0] = mfma32(af, bf, acc[i][0]);
                }
            }
        }
    };

    WLoad<WT> w0[CH], w1[CH];
    u32x4 av[APT];
    uint32_t amask;
    // step j multiplies group gb + KW j + way; a way's group past the block's last one is all zeros
    const int steps = (gn + KW - 1) / KW, g0 = gb + way;
    load_a(av, amask, g0);
    load_w(w0, g0);
    store_a(av, amask, 0);
    __syncthreads();
    int q = 0;
    for (; q + 2 <= steps; q += 2) {
        load_a(av, amask, g0 + KW * (q + 1));
        load_w(w1, g0 + KW * (q + 1));
        compute(w0, 0);
        store_a(av, amask, 1);
        __syncthreads();
        load_a(av, amask, g0 + KW * (q + 2));
        load_w(w0, g0 + KW * (q + 2));
        compute(w1, 1);
        store_a(av, amask, 0);
        __syncthreads();
    }
    if (q < steps) compute(w0, 0);

    scale_rows(acc, args.scales, 0, lg, args.M);
    constexpr int OWN = MT * 16 / KW;   // elements of the tile this way stores
    if constexpr (KW > 1) {
        // the ways' sums, added in way order: way w finishes elements [w OWN, (w + 1) OWN) of the tile
        constexpr int WS = NW * MT * 16 * WAVE;
        float * mg = (float *)sk_smem + wave * (MT * 16 * WAVE) + lane;   // [way][wave][element][lane]
        __syncthreads();   // the last slices have been read
#pragma unroll
        for (int w = 0; w < KW; w++)
            if (w != way)
#pragma unroll
                for (int x = w * OWN; x < (w + 1) * OWN; x++) mg[way * WS + x * WAVE] = acc[x / 16][0][x % 16];
        __syncthreads();
#pragma unroll
        for (int w = 0; w < KW; w++)
            if (w == way)
#pragma unroll
                for (int x = w * OWN; x < (w + 1) * OWN; x++) {
                    float s = w == 0 ? acc[x / 16][0][x % 16] : mg[x * WAVE];
#pragma unroll
                    for (int v = 1; v < KW; v++) s += v == w ? acc[x / 16][0][x % 16] : mg[v * WS + x * WAVE];
                    acc[x / 16][0][x % 16] = s;
                }
    }
    if (!okn || gn == 0) return;
#pragma unroll
    for (int i = 0; i < MT; i++) {
#pragma unroll
        for (int e = 0; e < 16; e++) {
            if ((i * 16 + e) / OWN != way) continue;
            const int r = i * 32 + 8 * (e / 4) + 4 * lg + (e % 4);
            if (r >= args.M) continue;
            float * p = G.C + (int64_t)r * G.ldc + n;
            if (ks == 1 || args.part) *p = acc[i][0][e];
            else unsafeAtomicAdd(p, acc[i][0][e]);
        }
    }
}

// ---------------------------------------------------------------------------------------------
// fp16-weight GEMM with LDS DMA
//
// For fp16 weights nothing has to be decoded between HBM and LDS, so both operands go straight
// into LDS with global_load_lds_dwordx4 (gfx950): no staging registers, no ds_write. K is staged
// DK (32, 64 or 128) values at a time through a ring of NS LDS stages; while one stage is
// multiplied the next NS-1 are landing. A block is WGM x WGN waves, each owning a
// (BM/WGM) x (BN/WGN) tile of 32x32x16 MFMAs with its accumulators in AGPRs. With 8 waves two
// share each SIMD, so one wave's MFMAs cover the other's LDS reads and barrier waits.
//
// A DMA instruction writes 64 lanes x 16 bytes to 1 KB of consecutive LDS; lane l lands at
// base + 16 l. Each lane therefore fetches the global chunk that belongs at its LDS slot under
// the swizzle: a row of DK values holds CH = DK/8 chunks, and slot (row, p) holds logical chunk
// p ^ ((row / (16/CH)) & (CH-1)), so the 16 rows of an MFMA fragment read hit 16 distinct bank
// groups. With DK >= 64 every DMA instruction covers whole 128-byte lines of A and W, which
// halves the cache-line lookups per byte against DK = 32 (the limit of this path when all its
// data hits in L2). Rows past M or N are clamped to the last real row (their results are never
// stored); K must be a multiple of DK, so there is no K tail.
//
// The waits are explicit, and the compiler is kept from adding its own around the DMA:
//   * before every barrier, s_waitcnt on this wave's DMA count (the stage about to be read has
//     landed, the NS-2 behind it may still be in flight) and on lgkmcnt (this wave's LDS reads of
//     the stage about to be overwritten are done);
//   * every iteration issues exactly one stage of DMA (past the last stage it re-fetches the last
//     one into a buffer nobody reads again), so those counts are the same every time and the loop
//     body has no branch;
//   * the compiler waits for all outstanding LDS reads before an MFMA whose fragment is still in
//     flight (it cannot order them against the DMA), so each fragment read is issued after the
//     first MFMA that would otherwise wait for it, and scheduling barriers keep that order.
// KSPLIT = 2 splits K between two blocks that add their halves atomically into a zeroed output
// (two addends: the sum is the same in either order).
// ---------------------------------------------------------------------------------------------
template <int BM, int BN, int WGM, int WGN, int DK, int NS>
struct F16Cfg {
    static constexpr int NW = WGM * WGN, THREADS = WAVE * NW;
    static constexpr int TM = BM / WGM, TN = BN / WGN, MI = TM / 32, NJ = TN / 32;
    static constexpr int CH = DK / 8, RPW = 16 / CH, RB = DK * 2;
    static constexpr int A_BYTES = BM * RB, B_BYTES = BN * RB, STAGE = A_BYTES + B_BYTES;
    static constexpr int LDS = NS * STAGE;
    static constexpr int PA = A_BYTES / (THREADS * 16), PB = B_BYTES / (THREADS * 16);   // DMA per wave
    static constexpr int PER = PA + PB;
    static_assert(MI >= 1 && NJ >= 1 && TM % 32 == 0 && TN % 32 == 0, "wave tile");
    static_assert(PA >= 1 && PB >= 1 && PA * THREADS * 16 == A_BYTES && PB * THREADS * 16 == B_BYTES, "DMA split");
    static_assert(NS >= 2 && (NS - 1) * PER <= 63, "vmcnt range");
    static_assert(LDS <= 160 * 1024, "LDS");
};

typedef const void __attribute__((address_space(1))) * gptr_t;
typedef void __attribute__((address_space(3))) * lptr_t;

__device__ __forceinline__ void dma16(const void * g, void * l) {
    __builtin_amdgcn_global_load_lds((gptr_t)g, (lptr_t)l, 16, 0, 0);
}

// s_waitcnt with vmcnt(N), expcnt(7) (no wait), lgkmcnt(0): gfx9 encoding.
template <int N>
__device__ __forceinline__ void wait_vm_lgkm0() {
    static_assert(N >= 0 && N <= 63, "vmcnt");
    __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (0 << 8) | ((N >> 4) << 14));
}

template <int BM, int BN, int WGM, int WGN, int DK, int NS, int KSPLIT, bool TL>
__global__ void __launch_bounds__(WAVE * WGM * WGN)
__attribute__((amdgpu_waves_per_eu(WGM * WGN / 4, WGM * WGN / 4)))
gemm_f16_kernel(GemmArgs args) {
    using C = F16Cfg<BM, BN, WGM, WGN, DK, NS>;
    extern __shared__ __align__(16) uint8_t smem[];
    const int t = threadIdx.x, lane = t % WAVE, wave = t / WAVE;
    const int wm = wave / WGN, wn = wave % WGN;

    int tile = xcd_tile(blockIdx.x, gridDim.x);
    const int split = tile % KSPLIT;
    tile /= KSPLIT;
    const int mt = tile % args.m_tiles, nt = tile / args.m_tiles;
    int g = 0;
#pragma unroll
    for (int i = 1; i < GEMM_MAX_GROUPS; i++)
        if (i < args.ng && nt >= args.g[i].ntile_begin) g = i;
    const uint16_t * W = (const uint16_t *)args.g[0].W;
    int64_t row0 = args.g[0].row0;
    int N = args.g[0].N, ntb = args.g[0].ntile_begin;
    float * Cp = args.g[0].C;
    int64_t ldc = args.g[0].ldc;
#pragma unroll
    for (int i = 1; i < GEMM_MAX_GROUPS; i++)
        if (i == g) {
            W = (const uint16_t *)args.g[i].W; row0 = args.g[i].row0; N = args.g[i].N;
            ntb = args.g[i].ntile_begin; Cp = args.g[i].C; ldc = args.g[i].ldc;
        }
    const int n0 = (nt - ntb) * BN, m0 = mt * BM;
    const int M = args.M, K = args.K;
    const int nk_all = K / DK;
    const int per = (nk_all + KSPLIT - 1) / KSPLIT;
    const int kb = split * per;
    const int nk = max(0, min(nk_all, kb + per) - kb);

    // this lane's global sources, one row chunk per DMA instruction, advanced by one stage's K
    // per stage: DK values in rows, DK/32 tiles of 512 values in the tiled layout (TL), where the
    // 16 rows x DK of one instruction are whole 64-byte tile rows
    const uint16_t * asrc[C::PA];
    const uint16_t * bsrc[C::PB];
#pragma unroll
    for (int q = 0; q < C::PA; q++) {
        const int slot = (q * C::NW + wave) * WAVE + lane;
        const int r = slot / C::CH, c = (slot % C::CH) ^ ((r / C::RPW) & (C::CH - 1));
        const int64_t row = min(m0 + r, M - 1), k = (int64_t)kb * DK + 8 * c;
        asrc[q] = args.A + (TL ? tiled_index(row, k, K) : row * args.lda + k);
    }
#pragma unroll
    for (int q = 0; q < C::PB; q++) {
        const int slot = (q * C::NW + wave) * WAVE + lane;
        const int r = slot / C::CH, c = (slot % C::CH) ^ ((r / C::RPW) & (C::CH - 1));
        const int64_t row = row0 + min(n0 + r, N - 1), k = (int64_t)kb * DK + 8 * c;
        bsrc[q] = W + (TL ? tiled_index(row, k, K) : row * K + k);
    }
    // the LDS destination of a DMA instruction must be wave-uniform (it goes to M0): take the
    // wave index from an SGPR so the address arithmetic stays scalar
    const int wave_s = __builtin_amdgcn_readfirstlane(wave);
    // stage s into ring buffer s % NS; past the last stage the last one is fetched again into
    // the buffer just freed (nobody reads it again)
    auto issue = [&](int s) {
        uint8_t * st = smem + (s % NS) * C::STAGE;
        s = min(s, nk - 1);
        const int64_t off = (int64_t)s * (TL ? DK * 16 : DK);
#pragma unroll
        for (int q = 0; q < C::PA; q++) dma16(asrc[q] + off, st + (q * C::NW + wave_s) * 1024);
#pragma unroll
        for (int q = 0; q < C::PB; q++) dma16(bsrc[q] + off, st + C::A_BYTES + (q * C::NW + wave_s) * 1024);
    };

    float16v acc[C::MI][C::NJ];
#pragma unroll
    for (int i = 0; i < C::MI; i++)
#pragma unroll
        for (int j = 0; j < C::NJ; j++)
#pragma unroll
            for (int e = 0; e < 16; e++) acc[i][j][e] = 0.0f;

    // fragment rows (w*T + i*32 + lr), logical chunk (2 ks + lg); the row part of the swizzle
    // depends on lr only, because w*T + i*32 is a multiple of 16
    const int lr = lane % 32, lg = lane / 32, x = (lr / C::RPW) & (C::CH - 1);
    const int a_off = (wm * C::TM + lr) * C::RB, b_off = C::A_BYTES + (wn * C::TN + lr) * C::RB;
    struct Frags {
        half8 a[C::MI], b[C::NJ];
    };
    auto read_frags = [&](int s, int ks, Frags & f) {
        const uint8_t * st = smem + (s % NS) * C::STAGE;
        const int co = ((2 * ks + lg) ^ x) * 16;
#pragma unroll
        for (int i = 0; i < C::MI; i++) f.a[i] = *(const half8 *)(st + a_off + i * 32 * C::RB + co);
#pragma unroll
        for (int j = 0; j < C::NJ; j++) f.b[j] = *(const half8 *)(st + b_off + j * 32 * C::RB + co);
    };
    // the MFMAs of one 16-deep K step; `part` 0 = only the first, 1 = all but the first
    auto mma = [&](const Frags & f, int part) {
#pragma unroll
        for (int i = 0; i < C::MI; i++)
#pragma unroll
            for (int j = 0; j < C::NJ; j++)
                if ((part == 0) == (i == 0 && j == 0)) acc[i][j] = mfma32(f.a[i], f.b[j], acc[i][j]);
    };

    // Software pipeline over the 16-deep K steps of each stage, fragments alternating between f0
    // and f1: the next step's fragments are read while this step's MFMAs run. At the last step of
    // a stage: one barrier (the next stage has landed for every wave, and every wave is done
    // reading this one), the next stage's first fragments, and the DMA of the stage NS ahead
    // into the buffer just freed.
    if (nk > 0) {
        Frags f0, f1;
#pragma unroll
        for (int p = 0; p < NS; p++) issue(p);
        wait_vm_lgkm0<(NS - 1) * C::PER>();
        __builtin_amdgcn_s_barrier();
        read_frags(0, 0, f0);
        constexpr int KS = DK / 16;
        for (int s = 0; s < nk; s++) {
#pragma unroll
            for (int ks = 0; ks < KS; ks++) {
                Frags & F = (ks % 2 == 0) ? f0 : f1;
                Frags & G = (ks % 2 == 0) ? f1 : f0;
                mma(F, 0);
                __builtin_amdgcn_sched_barrier(0);
                if (ks + 1 < KS) {
                    read_frags(s, ks + 1, G);
                    __builtin_amdgcn_sched_barrier(0);
                } else {
                    wait_vm_lgkm0<(NS - 2) * C::PER>();
                    __builtin_amdgcn_s_barrier();
                    read_frags(s + 1, 0, G);
                    __builtin_amdgcn_sched_barrier(0);
                    issue(s + NS);
                    __builtin_amdgcn_sched_barrier(0);
                }
                mma(F, 1);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        wait_vm_lgkm0<0>();   // no DMA may still be writing this block's LDS when it exits
    }

    // epilogue: C = scale[m] * acc
    scale_rows(acc, args.scales, m0 + wm * C::TM, lg, M);
#pragma unroll
    for (int i = 0; i < C::MI; i++) {
#pragma unroll
        for (int e = 0; e < 16; e++) {
            const int r = m0 + wm * C::TM + i * 32 + 8 * (e / 4) + 4 * lg + (e % 4);
            if (r >= M) continue;
            float * crow = Cp + (int64_t)r * ldc;
#pragma unroll
            for (int j = 0; j < C::NJ; j++) {
                const int n = n0 + wn * C::TN + j * 32 + lr;
                if (n < N) {
                    if (KSPLIT == 1) crow[n] = acc[i][j][e];
                    else unsafeAtomicAdd(crow + n, acc[i][j][e]);
                }
            }
        }
    }
}

// ---------------------------------------------------------------------------------------------
// The same LDS-DMA pipeline with a block tile whose two wave columns differ in width: BN0 + BN1
// columns (e.g. 128 + 96 = 224), 8 waves in a 4 x 2 grid. A 256 x 224 tile cuts an N of 28672
// (the fused gate/up of an 8B model) into 128 x 2 = 256 blocks, one per CU, where 256 x 256
// leaves 32 CUs idle. Wave w takes column w / 4, so each SIMD (w % 4) holds one wave of each
// width. Each column's four waves fetch that column's B rows, so the DMA count per stage, and
// with it the vmcnt of every wait, is a per-column constant; the body below is instantiated once
// per column width, and both instances meet at the same barriers (one before the loop, one per
// stage).
// Where a column's B rows of one stage are not a whole number of DMA instructions per wave of
// that column (96 rows x 32 K: 6 KB for four waves), all eight waves share the B tile instead:
// instruction i (1 KB, 1024 / RB rows) goes to wave i % 8, and the waves whose last slot has no
// real instruction fetch the last real chunk again into a 1 KB LDS slot nobody reads, so every
// wave issues the same number of DMA instructions a stage and the wait counts stay constants.
// ---------------------------------------------------------------------------------------------
template <int BM_, int BN0, int BN1, int DK, int NS>
struct ColsCfg {
    static constexpr int NW = 8, THREADS = WAVE * NW, WGM = 4;
    static constexpr int BM = BM_, BN = BN0 + BN1, TM = BM / WGM, MI = TM / 32;
    static constexpr int CH = DK / 8, RPW = 16 / CH, RB = DK * 2, NSTAGES = NS;
    static constexpr int A_BYTES = BM * RB, B_BYTES = BN * RB, STAGE = A_BYTES + B_BYTES;
    static constexpr bool PERCOL = (BN0 * RB) % (4 * 1024) == 0 && (BN1 * RB) % (4 * 1024) == 0;
    static constexpr int NBI = B_BYTES / 1024;                       // B DMA instructions a stage
    static constexpr int PBW = (NBI + NW - 1) / NW;                  // per wave when shared
    static constexpr int RING = NS * STAGE;
    static constexpr int LDS = RING + (PERCOL ? 0 : (NW * PBW - NBI) * 1024);
    static constexpr int PA = A_BYTES / (THREADS * 16);
    static constexpr int PER_MAX = PA + (PERCOL ? BN0 * RB / 4096 : PBW);
    static_assert(MI >= 1 && TM % 32 == 0 && BN0 % 32 == 0 && BN1 % 32 == 0 && BN0 % 16 == 0, "wave tile");
    static_assert(PA * THREADS * 16 == A_BYTES, "A DMA split");
    static_assert(B_BYTES % 1024 == 0, "B DMA split");
    static_assert(NS >= 2 && (NS - 1) * PER_MAX <= 63, "vmcnt range");
    static_assert(LDS <= 160 * 1024, "LDS");
};

// The weight group a block's N tile falls in, resolved once per block from the kernel
// arguments (a select chain: indexing args.g with a runtime value would copy the array to
// scratch).
struct ColsTile {
    const uint16_t * W;
    int64_t row0;
    float * C;
    int64_t ldc;
    int N, n0, m0;
};

template <class C, int TNW, int COL0>
__device__ __forceinline__ void cols_body(const uint16_t * __restrict__ Ap, const float * __restrict__ scales,
                                          int64_t lda, int M, int K, ColsTile tb, uint8_t * smem, int wm) {
    constexpr int DK = C::RB / 2, NS = C::NSTAGES, NJ = TNW / 32;
    constexpr int PB = C::PERCOL ? TNW * C::RB / 4096 : C::PBW;   // this wave's B DMA a stage
    constexpr int PER = C::PA + PB;
    const int t = threadIdx.x, lane = t % WAVE, wave = t / WAVE;
    const uint16_t * W = tb.W;
    const int64_t row0 = tb.row0;
    const int N = tb.N;
    float * Cp = tb.C;
    const int64_t ldc = tb.ldc;
    const int n0 = tb.n0, m0 = tb.m0;
    const int nk = K / DK;

    const uint16_t * asrc[C::PA];
    const uint16_t * bsrc[PB];
#pragma unroll
    for (int q = 0; q < C::PA; q++) {
        const int slot = (q * C::NW + wave) * WAVE + lane;
        const int r = slot / C::CH, c = (slot % C::CH) ^ ((r / C::RPW) & (C::CH - 1));
        const int64_t row = min(m0 + r, M - 1), k = 8 * c;
        asrc[q] = Ap + row * lda + k;
    }
#pragma unroll
    for (int q = 0; q < PB; q++) {
        if constexpr (C::PERCOL) {
            // rows COL0 .. COL0 + TNW of the B tile, fetched by this column's four waves; COL0 is a
            // multiple of 16, so the swizzle of a row depends on its offset inside the column only
            const int slot = (q * 4 + wm) * WAVE + lane;
            const int r = slot / C::CH, c = (slot % C::CH) ^ ((r / C::RPW) & (C::CH - 1));
            const int64_t row = row0 + min(n0 + COL0 + r, N - 1), k = 8 * c;
            bsrc[q] = W + row * K + k;
        } else {
            // instruction q * 8 + wave of the whole B tile (rows of both columns in order; the
            // swizzle is the same, since BN0 is a multiple of 16)
            const int slot = min(q * C::NW + wave, C::NBI - 1) * WAVE + lane;
            const int r = slot / C::CH, c = (slot % C::CH) ^ ((r / C::RPW) & (C::CH - 1));
            const int64_t row = row0 + min(n0 + r, N - 1), k = 8 * c;
            bsrc[q] = W + row * K + k;
        }
    }
    const int wave_s = __builtin_amdgcn_readfirstlane(wave), wm_s = __builtin_amdgcn_readfirstlane(wm);
    auto issue = [&](int s) {
        uint8_t * st = smem + (s % NS) * C::STAGE;
        s = min(s, nk - 1);
        const int64_t off = (int64_t)s * DK;
#pragma unroll
        for (int q = 0; q < C::PA; q++) dma16(asrc[q] + off, st + (q * C::NW + wave_s) * 1024);
#pragma unroll
        for (int q = 0; q < PB; q++) {
            if constexpr (C::PERCOL) {
                dma16(bsrc[q] + off, st + C::A_BYTES + COL0 * C::RB + (q * 4 + wm_s) * 1024);
            } else {
                const int gi = q * C::NW + wave_s;
                dma16(bsrc[q] + off, gi < C::NBI ? st + C::A_BYTES + gi * 1024 : smem + C::RING + (gi - C::NBI) * 1024);
            }
        }
    };

    float16v acc[C::MI][NJ];
#pragma unroll
    for (int i = 0; i < C::MI; i++)
#pragma unroll
        for (int j = 0; j < NJ; j++)
#pragma unroll
            for (int e = 0; e < 16; e++) acc[i][j][e] = 0.0f;

    const int lr = lane % 32, lg = lane / 32, x = (lr / C::RPW) & (C::CH - 1);
    const int a_off = (wm * C::TM + lr) * C::RB, b_off = C::A_BYTES + (COL0 + lr) * C::RB;
    struct Frags {
        half8 a[C::MI], b[NJ];
    };
    auto read_frags = [&](int s, int ks, Frags & f) {
        const uint8_t * st = smem + (s % NS) * C::STAGE;
        const int co = ((2 * ks + lg) ^ x) * 16;
#pragma unroll
        for (int i = 0; i < C::MI; i++) f.a[i] = *(const half8 *)(st + a_off + i * 32 * C::RB + co);
#pragma unroll
        for (int j = 0; j < NJ; j++) f.b[j] = *(const half8 *)(st + b_off + j * 32 * C::RB + co);
    };
    auto mma = [&](const Frags & f, int part) {
#pragma unroll
        for (int i = 0; i < C::MI; i++)
#pragma unroll
            for (int j = 0; j < NJ; j++)
                if ((part == 0) == (i == 0 && j == 0)) acc[i][j] = mfma32(f.a[i], f.b[j], acc[i][j]);
    };

    // the pipeline of gemm_f16_kernel, stage for stage (same barriers, same DMA order)
    if (nk > 0) {
        Frags f0, f1;
#pragma unroll
        for (int p = 0; p < NS; p++) issue(p);
        wait_vm_lgkm0<(NS - 1) * PER>();
        __builtin_amdgcn_s_barrier();
        read_frags(0, 0, f0);
        constexpr int KS = DK / 16;
        for (int s = 0; s < nk; s++) {
#pragma unroll
            for (int ks = 0; ks < KS; ks++) {
                Frags & F = (ks % 2 == 0) ? f0 : f1;
                Frags & G = (ks % 2 == 0) ? f1 : f0;
                mma(F, 0);
                __builtin_amdgcn_sched_barrier(0);
                if (ks + 1 < KS) {
                    read_frags(s, ks + 1, G);
                    __builtin_amdgcn_sched_barrier(0);
                } else {
                    wait_vm_lgkm0<(NS - 2) * PER>();
                    __builtin_amdgcn_s_barrier();
                    read_frags(s + 1, 0, G);
                    __builtin_amdgcn_sched_barrier(0);
                    issue(s + NS);
                    __builtin_amdgcn_sched_barrier(0);
                }
                mma(F, 1);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        wait_vm_lgkm0<0>();
    }

    scale_rows(acc, scales, m0 + wm * C::TM, lg, M);
#pragma unroll
    for (int i = 0; i < C::MI; i++) {
#pragma unroll
        for (int e = 0; e < 16; e++) {
            const int r = m0 + wm * C::TM + i * 32 + 8 * (e / 4) + 4 * lg + (e % 4);
            if (r >= M) continue;
            float * crow = Cp + (int64_t)r * ldc;
#pragma unroll
            for (int j = 0; j < NJ; j++) {
                const int n = n0 + COL0 + j * 32 + lr;
                if (n < N) crow[n] = acc[i][j][e];
            }
        }
    }
}

template <int BM, int BN0, int BN1, int DK, int NS>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
gemm_f16_cols_kernel(GemmArgs args) {
    using C = ColsCfg<BM, BN0, BN1, DK, NS>;
    extern __shared__ __align__(16) uint8_t smem[];
    const int wave = threadIdx.x / WAVE;
    const int tile = xcd_tile(blockIdx.x, gridDim.x);
    const int mt = tile % args.m_tiles, nt = tile / args.m_tiles;
    ColsTile tb;
    tb.W = (const uint16_t *)args.g[0].W; tb.row0 = args.g[0].row0; tb.N = args.g[0].N;
    tb.C = args.g[0].C; tb.ldc = args.g[0].ldc;
    int ntb = args.g[0].ntile_begin;
#pragma unroll
    for (int i = 1; i < GEMM_MAX_GROUPS; i++)
        if (i < args.ng && nt >= args.g[i].ntile_begin) {
            tb.W = (const uint16_t *)args.g[i].W; tb.row0 = args.g[i].row0; tb.N = args.g[i].N;
            tb.C = args.g[i].C; tb.ldc = args.g[i].ldc; ntb = args.g[i].ntile_begin;
        }
    tb.n0 = (nt - ntb) * C::BN;
    tb.m0 = mt * C::BM;
    if (wave / 4 == 0) cols_body<C, BN0, 0>(args.A, args.scales, args.lda, args.M, args.K, tb, smem, wave % 4);
    else cols_body<C, BN1, BN0>(args.A, args.scales, args.lda, args.M, args.K, tb, smem, wave % 4);
}

// ---------------------------------------------------------------------------------------------
// Tiled fp16 weights (T_F16T): one wave per SIMD, every memory instruction under an MFMA
//
// What bounds a tile of gemm_f16_kernel above is the CU's LDS and the instruction order, not the
// MFMAs: eight waves of 64 x 128 read 96 bytes of LDS a clock at the full MFMA rate beside the 32
// the DMA writes (128 is the CU's limit), and all of them issue their reads and DMA in one burst
// after each stage's barrier. Here a block is four waves, one per SIMD, so a wave has 512 registers
// and takes up to 128 x 112 of the output (accumulators in AGPRs): a 256 x 224 tile reads 69 bytes
// a clock at the full MFMA rate (39 beside the DMA's 20 at the 0.54 it reaches at 512 x 28672 x
// 4096). With no second wave to cover for it, the wave has to keep its own MFMAs issuing: stage
// s is multiplied from registers while stage s + 1's fragments are read and stage s + NS's DMA is
// issued, one read or one DMA after each MFMA (a 16 x 16 x 32 MFMA takes 16 clocks, a read or a
// DMA 4 to 8 of issue). Two things keep those gaps that short: buffer loads, whose source is a
// fixed lane offset plus one scalar stage offset (global loads took a scalar chain and a 64-bit
// vector add each: 119 us instead of 107 at 512 x 28672 x 4096), and the empty asm statements at the
// stage's end, which hold the accumulators in AGPRs across the loop (left alone, the compiler moves
// them through VGPRs: hundreds of moves a stage).
//
// A stage is 32 values of K for the tile's BM + BN rows; LDS slot (row r, chunk p) of its 4 chunks a
// row holds logical chunk p ^ ((r / 4) & 3), so the 16 rows of a fragment read fall on 16 distinct
// 16-byte slots of 256 bytes. SQ_LDS_BANK_CONFLICT still counts four cycles a read (none for the
// 128-byte rows of gemm_f16_kernel), under the MFMAs: the waves wait on LDS 4-8% of their time. Per
// stage, after its first MFMA (whose operands are the wave's last reads of the
// stage's buffer): wait until stage s + 1 has landed (the (NS - 2) stages behind it may be in
// flight), one barrier, then buffer s % NS is refilled with stage s + NS. Past the last stage the
// last one is fetched again into buffers nobody reads, so the wait counts are constants.
// Rows past M or N read the last real row. The MFMA's first operand is the weight, so a lane holds
// 4 consecutive output columns of one row and stores 16 bytes at once. The two widest tiles spill
// outside the loop over the stages: 8 registers (256 x 224) and 74 (256 x 256) a lane, once per block.
//
// A launch of few tiles splits K args.ksplit ways (each split a slab of args.part, summed in split
// order by reduce_splits_kernel). Measured against gemm_f16_kernel and its two-width variant on
// cold weights, one box, M x N x K (us): 512 x 28672 x 4096 118.2 -> 102.6, 2048 x 6144 x 4096 101.1 ->
// 85.6, 2048 x 3072 x 8192 121.2 -> 93.7, 512 x 4096 x 14336 83.1 -> 69 (split 4), 512 x 4096 x 4096
// 29.9 -> 24.2, 48 x 1536 x 8960 30.8 -> 13.1 (split 8); over 95 shapes 1.2x (M 48-2048).
// ---------------------------------------------------------------------------------------------
typedef float f32x4 __attribute__((ext_vector_type(4)));
// D(16x16, f32) += A(16x32, f16) . B(32x16, f16). Lane l holds A row and B column l % 16, K slots
// 8 (l / 16) + 0..7; D: column l % 16, rows 4 (l / 16) + 0..3.
__device__ __forceinline__ void mfma16(const half8 & a, const half8 & b, f32x4 & c) {
    c = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

template <int BM_, int BN_, int WGM_, int WGN_, int NS_>
struct OneWaveCfg {
    static constexpr int BM = BM_, BN = BN_, NS = NS_, NW = 4, THREADS = 256, WGN = WGN_;
    static constexpr int TM = BM / WGM_, TN = BN / WGN_, MI = TM / 16, NJ = TN / 16;
    static constexpr int RB = 64;                                   // bytes of a row's 32 values
    // DMA instructions per wave and stage, 4 KB of LDS a block each; a BN of 96, 160 or 224 ends
    // half-way through one, whose other half fetches rows nobody reads into the stage's padding
    static constexpr int PA = (BM * RB + 4095) / 4096, PB = (BN * RB + 4095) / 4096, PER = PA + PB;
    static constexpr int A_BYTES = PA * 4096, STAGE = A_BYTES + PB * 4096, LDS = NS * STAGE;
    static_assert(WGM_ * WGN_ == 4 && TM % 16 == 0 && TN % 16 == 0, "wave tile");
    static_assert(LDS <= 160 * 1024 && NS >= 3 && (NS - 1) * PER <= 63, "ring");
};

template <int BM, int BN, int WGM, int WGN, int NS>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1)))
gemm_f16_1w_kernel(GemmArgs args) {
#ifdef __HIP_DEVICE_COMPILE__   // the buffer resource type exists in the device pass only
    using C = OneWaveCfg<BM, BN, WGM, WGN, NS>;
    extern __shared__ __align__(16) uint8_t smem[];
    const int t = threadIdx.x, lane = t % WAVE, wave = __builtin_amdgcn_readfirstlane(t / WAVE);
    const int wm = wave / WGN, wn = wave % WGN;
    const int ks = args.ksplit > 1 ? args.ksplit : 1;
    int tile = xcd_tile(blockIdx.x, gridDim.x);
    const int split = tile % ks;
    tile /= ks;
    const int mt = tile % args.m_tiles, nt = tile / args.m_tiles;
    int g = 0;
    const uint16_t * W = (const uint16_t *)args.g[0].W;
    int64_t row0 = args.g[0].row0;
    int N = args.g[0].N, ntb = args.g[0].ntile_begin;
    float * Cp = args.g[0].C;
    int64_t ldc = args.g[0].ldc;
#pragma unroll
    for (int i = 1; i < GEMM_MAX_GROUPS; i++)
        if (i < args.ng && nt >= args.g[i].ntile_begin) {
            g = i;
            W = (const uint16_t *)args.g[i].W; row0 = args.g[i].row0; N = args.g[i].N;
            ntb = args.g[i].ntile_begin; Cp = args.g[i].C; ldc = args.g[i].ldc;
        }
    split_target(args, g, split, Cp, ldc);
    const int n0 = (nt - ntb) * BN, m0 = mt * BM;
    const int M = args.M, K = args.K, nk_all = K / 32;
    const int per = (nk_all + ks - 1) / ks, kb = split * per;
    const int nk = max(0, min(nk_all, kb + per) - kb);

    // each operand's buffer starts at the tile's first 16-row block; a lane's offset in it, the stage's
    // included, stays below 17 * 32 * K bytes: 256 rows from a row0 inside a block touch 17 of them
    // (the launcher keeps K under ONE_WAVE_MAX_K)
    constexpr int KSTEP = 1024;   // bytes of a row block one stage of K takes
    const int64_t a0 = tiled_index(m0, 0, K), b0 = tiled_index((row0 + n0) & ~(int64_t)15, 0, K);
    const char * abase = (const char *)(args.A + a0) + (int64_t)kb * KSTEP;
    const char * bbase = (const char *)(W + b0) + (int64_t)kb * KSTEP;
    int aoff[C::PA], boff[C::PB];
#pragma unroll
    for (int q = 0; q < C::PA; q++) {
        const int slot = (q * 4 + wave) * WAVE + lane, r = slot / 4, c = (slot % 4) ^ ((r / 4) & 3);
        const int64_t row = min(m0 + r, M - 1);
        aoff[q] = (int)(2 * (tiled_index(row, 8 * c, K) - a0));
    }
#pragma unroll
    for (int q = 0; q < C::PB; q++) {
        const int slot = (q * 4 + wave) * WAVE + lane, r = slot / 4, c = (slot % 4) ^ ((r / 4) & 3);
        const int64_t row = row0 + min(n0 + r, N - 1);
        boff[q] = (int)(2 * (tiled_index(row, 8 * c, K) - b0));
    }
    const __amdgpu_buffer_rsrc_t ar = __builtin_amdgcn_make_buffer_rsrc((void *)abase, 0, 0x7FFFFFFF, 0x00020000);
    const __amdgpu_buffer_rsrc_t br = __builtin_amdgcn_make_buffer_rsrc((void *)bbase, 0, 0x7FFFFFFF, 0x00020000);
    auto issue1 = [&](uint8_t * st, int soff, int q) {
        if (q < C::PA)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(ar, (lptr_t)(st + wave * 1024 + q * 4096), 16, aoff[q], soff, 0, 0);
        else
            __builtin_amdgcn_raw_ptr_buffer_load_lds(br, (lptr_t)(st + wave * 1024 + q * 4096), 16, boff[q - C::PA], soff, 0, 0);
    };
    const int lr = lane % 16, lg = lane / 16;
    const int co = (lg ^ ((lr / 4) & 3)) * 16;
    const int a_off = (wm * C::TM + lr) * 64 + co, b_off = C::A_BYTES + (wn * C::TN + lr) * 64 + co;

    f32x4 acc[C::MI][C::NJ];
#pragma unroll
    for (int i = 0; i < C::MI; i++)
#pragma unroll
        for (int j = 0; j < C::NJ; j++) acc[i][j] = f32x4{0, 0, 0, 0};

    struct Frags {
        half8 a[C::MI], b[C::NJ];
    };
    auto read1 = [&](const uint8_t * st, Frags & f, int r) {
        if (r < C::NJ) f.b[r] = *(const half8 *)(st + b_off + r * 1024);
        else f.a[r - C::NJ] = *(const half8 *)(st + a_off + (r - C::NJ) * 1024);
    };
    constexpr int NR = C::MI + C::NJ, NM = C::MI * C::NJ;
    int buf = 0;                                   // byte offset of the stage being multiplied
    const int last = (nk - 1) * KSTEP;
    int soff = min(NS * KSTEP, last);              // source offset of the stage NS ahead
    auto stage = [&](const Frags & F, Frags & G) {
        const int nbuf = buf == (NS - 1) * C::STAGE ? 0 : buf + C::STAGE;
        const uint8_t * st = smem + nbuf;
        uint8_t * fill = smem + buf;
#pragma unroll
        for (int p = 0; p < NM; p++) {
            const int i = p / C::NJ, j = p % C::NJ;
            mfma16(F.b[j], F.a[i], acc[i][j]);
            __builtin_amdgcn_sched_barrier(0);
            if (p == 0) {   // stage s + 1 has landed, and every wave is done with this stage's buffer
                wait_vm_lgkm0<(NS - 2) * C::PER>();
                __builtin_amdgcn_s_barrier();
                __builtin_amdgcn_sched_barrier(0);
            }
            constexpr int RS = NM >= 3 * NR ? 2 : 1;
            if (p >= 1 && (p - 1) % RS == 0 && (p - 1) / RS < NR) {
                read1(st, G, (p - 1) / RS);
                __builtin_amdgcn_sched_barrier(0);
            }
            constexpr int DS = (NM - 2) / C::PER > 0 ? (NM - 2) / C::PER : 1;
            if (p >= 2 && (p - 2) % DS == 0 && (p - 2) / DS < C::PER) {
                issue1(fill, soff, (p - 2) / DS);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        static_assert((NR - 1) * (NM >= 3 * NR ? 2 : 1) + 1 < NM && C::PER <= NM - 2, "a slot for every read and DMA");
        // the accumulators stay in AGPRs from stage to stage
#pragma unroll
        for (int i = 0; i < C::MI; i++)
#pragma unroll
            for (int j = 0; j < C::NJ; j++) asm volatile("" : "+a"(acc[i][j]));
        buf = nbuf;
        soff = min(soff + KSTEP, last);
    };
    if (nk > 0) {
        Frags f0, f1;
#pragma unroll
        for (int p = 0; p < NS; p++)
#pragma unroll
            for (int q = 0; q < C::PER; q++) issue1(smem + p * C::STAGE, min(p * KSTEP, last), q);
        wait_vm_lgkm0<(NS - 1) * C::PER>();
        __builtin_amdgcn_s_barrier();
#pragma unroll
        for (int r = 0; r < NR; r++) read1(smem, f0, r);
        int s = 0;
        for (; s + 2 <= nk; s += 2) {
            stage(f0, f1);
            stage(f1, f0);
        }
        if (s < nk) stage(f0, f1);
        wait_vm_lgkm0<0>();
    }
    // epilogue: the lane holds output row lr of each 16-row block, columns 4 lg .. 4 lg + 3 of each
    // 16-column one. Every scale is loaded before the first store (loads and stores retire in order).
    float sc[C::MI];
#pragma unroll
    for (int i = 0; i < C::MI; i++) sc[i] = args.scales[min(m0 + wm * C::TM + i * 16 + lr, M - 1)];
    const bool vec = ((reinterpret_cast<uintptr_t>(Cp) | (uintptr_t)(4 * ldc)) & 15) == 0;
#pragma unroll
    for (int i = 0; i < C::MI; i++) {
        const int r = m0 + wm * C::TM + i * 16 + lr;
        if (r >= M) continue;
        float * crow = Cp + (int64_t)r * ldc;
#pragma unroll
        for (int j = 0; j < C::NJ; j++) {
            const int n = n0 + wn * C::TN + j * 16 + 4 * lg;
            const f32x4 v = acc[i][j] * sc[i];
            if (n >= N) continue;
            if (vec) *(f32x4 *)(crow + n) = v;
            else
#pragma unroll
                for (int e = 0; e < 4; e++) crow[n + e] = v[e];
        }
        __builtin_amdgcn_sched_barrier(0);   // one row block's products at a time: few spills (see above)
    }
#endif
}

// ---------------------------------------------------------------------------------------------
// Q4_K GEMM with every operand by LDS DMA (the per-call dequant route for Q4_K weights).
//
// The weight stays in its Q4_K HBM layout (144-byte blocks of 256 values: d, dmin, 12 bytes of
// 6-bit scales and mins, 128 bytes of nibbles). Per 64-deep K stage a 256-row weight tile needs
// 32 bytes of nibbles a row (sub-blocks 2j and 2j+1 of the block, j = stage % 4) and, per block,
// its 16-byte header. Three LDS rings are filled by global_load_lds_dwordx4:
//   A  the row-scaled fp16 activations, two stages;
//   Q  the nibbles, three stages: thread t owns 16 bytes (row t/2, half t%2), landing at t*16;
//   H  the headers, two blocks: lanes 0-31 of wave w fetch rows 32w..32w+31, the rows its
//      threads decode.
// Q and H are private to the wave that fetches them, so only A needs the block's barrier. Each
// thread decodes its 32 values (rounding exactly as ggml's dequantizer) from Q and H into a
// double-buffered fp16 tile B; A and B use the 8-chunk XOR swizzle of the fp16 kernels, so the
// MFMA fragment reads are theirs. HBM and L2 traffic per weight is the Q4_K size, 0.5625 bytes
// (a resident fp16 copy moves 2).
//
// Per stage s (fragments of K step 0 already in registers; loop unrolled by 4, so s % 4 and
// with it every wait count below is a compile-time constant):
//   - the MFMAs of s, the fragments of the next K step read under each step's MFMAs;
//   - at one K step, a wait for the nibbles (and header) of s+1, issued two stages earlier, and
//     their decode into the free B buffer. Waves 4-7 decode two K steps after waves 0-3: the
//     waves that share a SIMD (w and w+4) take turns, one decoding while the other multiplies;
//   - after the first MFMA of the last K step: a wait for the activations of s+1 and this wave's
//     LDS writes, one barrier, the first fragments of s+1, then the DMA of the activations of
//     s+2, the nibbles of s+3 and, when s % 4 == 1, the header of the next block; the rest of the
//     step's MFMAs run under these.
// DMA instructions retire in order, so each wait counts the ones issued after its target (QD =
// the quant DMA instructions a thread issues per stage, 1 for Q4_K):
//   before the decode in stage s:  PA + QD, or PA + QD + 1 when s % 4 == 2 (a header was issued last)
//   at the end of stage s:         QD, or QD + 1 when s % 4 == 2.
// K % 256 == 0; a K split (args.ksplit) divides whole blocks. Past the last stage the last one
// is fetched and decoded again into the free buffers, so every stage issues the same DMA.
//
// The same pipeline takes Q8_0 weights in their split layout (int8 quants [rows][K], then fp16 d
// [rows][K/32]): a thread's 32 values are 32 quant bytes (QD = 2 instructions, the Q ring twice as
// wide) and the "header" of 256 values is the row's 8 block scales, 16 bytes as for Q4_K. The
// decode is Q8_0's packed one (exact: the int8 code under 1024, less the offset, times d rounds
// the exact product once). The wider Q ring leaves room for the 128 x 256 tile only.
// ---------------------------------------------------------------------------------------------
template <int WT, int BM, int WGM, int WGN>
struct Q4kCfg {
    static constexpr int BN = 256, NW = WGM * WGN, THREADS = WAVE * NW;
    static constexpr int TM = BM / WGM, TN = BN / WGN, MI = TM / 32, NJ = TN / 32;
    static constexpr int DK = 64, RB = 128;                         // 8 chunks of 16 bytes a row
    static constexpr int QD = WT == T_Q8_0 ? 2 : 1;                 // quant DMA per thread and stage
    static constexpr int A_BYTES = BM * RB, B_BYTES = BN * RB;
    static constexpr int Q_BYTES = BN * 32 * QD, H_BYTES = BN * 16;
    static constexpr int OFF_B = 2 * A_BYTES, OFF_Q = OFF_B + 2 * B_BYTES, OFF_H = OFF_Q + 3 * Q_BYTES;
    static constexpr int LDS = OFF_H + 2 * H_BYTES;
    static constexpr int PA = A_BYTES / (THREADS * 16);             // activation DMA per wave
    static_assert(WT == T_Q4_K || WT == T_Q8_0, "weight type");
    static_assert(NW == 8 && THREADS == 2 * BN, "one (row, half) item per thread");
    static_assert(MI >= 1 && NJ >= 1 && TM % 32 == 0 && TN % 32 == 0, "wave tile");
    static_assert(PA >= 1 && PA * THREADS * 16 == A_BYTES, "DMA split");
    static_assert(LDS <= 160 * 1024, "LDS");
};

// s_waitcnt with vmcnt(N) only (expcnt and lgkmcnt at their maximum): gfx9 encoding.
template <int N>
__device__ __forceinline__ void wait_vm() {
    static_assert(N >= 0 && N <= 63, "vmcnt");
    __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | ((N >> 4) << 14));
}

template <int WT, int BM, int WGM, int WGN>
__global__ void __launch_bounds__(WAVE * WGM * WGN)
__attribute__((amdgpu_waves_per_eu(2, 2)))
gemm_q4k_kernel(GemmArgs args) {
    using C = Q4kCfg<WT, BM, WGM, WGN>;
    extern __shared__ __align__(16) uint8_t smem[];
    const int t = threadIdx.x, lane = t % WAVE, wave = t / WAVE;
    const int wm = wave / WGN, wn = wave % WGN;

    const int ks = args.ksplit > 1 ? args.ksplit : 1;
    int tile = xcd_tile(blockIdx.x, gridDim.x);
    const int split = tile % ks;
    tile /= ks;
    const int mt = tile % args.m_tiles, nt = tile / args.m_tiles;
    int g = 0;
#pragma unroll
    for (int i = 1; i < GEMM_MAX_GROUPS; i++)
        if (i < args.ng && nt >= args.g[i].ntile_begin) g = i;
    const uint8_t * W = (const uint8_t *)args.g[0].W;
    int64_t row0 = args.g[0].row0, rows_total = args.g[0].rows_total;
    int N = args.g[0].N, ntb = args.g[0].ntile_begin;
    float * Cp = args.g[0].C;
    int64_t ldc = args.g[0].ldc;
#pragma unroll
    for (int i = 1; i < GEMM_MAX_GROUPS; i++)
        if (i == g) {
            W = (const uint8_t *)args.g[i].W; row0 = args.g[i].row0; N = args.g[i].N;
            ntb = args.g[i].ntile_begin; Cp = args.g[i].C; ldc = args.g[i].ldc;
            rows_total = args.g[i].rows_total;
        }
    split_target(args, g, split, Cp, ldc);
    const int n0 = (nt - ntb) * C::BN, m0 = mt * BM;
    const int M = args.M, K = args.K;
    const int nsb = K / 256;                                   // 256-value blocks a row
    const int per = (nsb + ks - 1) / ks;
    const int sb0 = split * per;
    const int nk = 4 * max(0, min(nsb, sb0 + per) - sb0);      // stages of this split

    // activation DMA: one 16-byte chunk of a row per instruction, the chunk that belongs at the
    // lane's LDS slot under the swizzle; rows past M read the last row (never stored)
    const uint16_t * asrc[C::PA];
#pragma unroll
    for (int q = 0; q < C::PA; q++) {
        const int slot = (q * C::NW + wave) * WAVE + lane;
        const int r = slot / 8, c = (slot % 8) ^ ((r / 2) & 7);
        asrc[q] = args.A + (int64_t)min(m0 + r, M - 1) * args.lda + (int64_t)sb0 * 256 + 8 * c;
    }
    // weight DMA: the quants of item t (row t/2, half t%2) and, for lanes 0-31, the header of
    // row 32 * wave + lane; rows past N read the last row (their outputs are never stored).
    // Q4_K: per block qs_blk bytes apart, the header at the block's start, the nibbles of
    // quarter j at 16 + 32 j; Q8_0: the quants at 64 bytes a stage, the 8 scales of a block
    // 16 bytes apart in the scale plane.
    const int64_t qrow = row0 + min(n0 + t / 2, N - 1), hrow = row0 + min(n0 + 32 * wave + lane % 32, N - 1);
    const uint8_t * qsrc;
    const uint8_t * hsrc;
    if constexpr (WT == T_Q4_K) {
        const int64_t rowb = (int64_t)(K / 256) * 144;
        qsrc = W + qrow * rowb + (int64_t)sb0 * 144 + 16 + 16 * (t % 2);
        hsrc = W + hrow * rowb + (int64_t)sb0 * 144;
    } else {
        qsrc = W + qrow * K + (int64_t)sb0 * 256 + 32 * (t % 2);
        hsrc = W + rows_total * K + (hrow * (K / 32) + (int64_t)sb0 * 8) * 2;
    }
    const int wave_s = __builtin_amdgcn_readfirstlane(wave);

    auto issue_a = [&](int s) {
        uint8_t * st = smem + (s & 1) * C::A_BYTES;
        const int64_t off = (int64_t)min(s, nk - 1) * C::DK;
#pragma unroll
        for (int q = 0; q < C::PA; q++) dma16(asrc[q] + off, st + (q * C::NW + wave_s) * 1024);
    };
    // the quant DMA of item t lands at (q * THREADS + t) * 16 of its Q stage, q < QD
    auto issue_q = [&](int s) {
        const int sc = min(s, nk - 1);
        const uint8_t * src = WT == T_Q4_K ? qsrc + (sc / 4) * 144 + 32 * (sc % 4) : qsrc + (int64_t)sc * 64;
#pragma unroll
        for (int q = 0; q < C::QD; q++)
            dma16(src + 16 * q, smem + C::OFF_Q + (s % 3) * C::Q_BYTES + (q * C::NW + wave_s) * 1024);
    };
    auto issue_h = [&](int b) {
        const int bc = min(b, nk / 4 - 1);
        if (lane < 32)
            dma16(hsrc + (WT == T_Q4_K ? bc * 144 : bc * 16), smem + C::OFF_H + (b & 1) * C::H_BYTES + wave_s * 512);
    };
    // decode the item of stage s (J = s % 4) into B buffer s & 1
    auto decode = [&](int s, auto Jc) {
        constexpr int J = decltype(Jc)::value;
        const u32x4 hdr = *(const u32x4 *)(smem + C::OFF_H + ((s / 4) & 1) * C::H_BYTES + (t / 2) * 16);
        const uint8_t * qs = smem + C::OFF_Q + (s % 3) * C::Q_BYTES + t * 16;
        u32x4 out[4];
        int run0, run1;
        if constexpr (WT == T_Q4_K) {
            WLoad<T_Q4_K> w;
            w.hdr = hdr;
            w.qs = *(const u32x4 *)qs;
            w.j = J;
            w.ok = true;
            w.decode(t % 2, out, run0, run1);
        } else {
            // block 2 J + half of the 256 values: its scale is half (t % 2) of word J
            WLoad<T_Q8_0> w;
            w.q[0] = *(const u32x4 *)qs;
            w.q[1] = *(const u32x4 *)(qs + C::THREADS * 16);
            w.d = (uint16_t)(hdr[J] >> (16 * (t % 2)));
            w.ok = true;
            w.decode_fast(t % 2, out, run0, run1);
        }
        uint8_t * bs = smem + C::OFF_B + (s & 1) * C::B_BYTES;
        const int r = t / 2;
        *(u32x4 *)(bs + swz<8>(r, run0 / 8)) = out[0];
        *(u32x4 *)(bs + swz<8>(r, run0 / 8 + 1)) = out[1];
        *(u32x4 *)(bs + swz<8>(r, run1 / 8)) = out[2];
        *(u32x4 *)(bs + swz<8>(r, run1 / 8 + 1)) = out[3];
    };

    float16v acc[C::MI][C::NJ];
#pragma unroll
    for (int i = 0; i < C::MI; i++)
#pragma unroll
        for (int j = 0; j < C::NJ; j++)
#pragma unroll
            for (int e = 0; e < 16; e++) acc[i][j][e] = 0.0f;

    const int lr = lane % 32, lg = lane / 32, x = (lr / 2) & 7;
    const int a_off = (wm * C::TM + lr) * C::RB, b_off = C::OFF_B + (wn * C::TN + lr) * C::RB;
    struct Frags {
        half8 a[C::MI], b[C::NJ];
    };
    auto read_frags = [&](int s, int kstep, Frags & f) {
        const uint8_t * as = smem + (s & 1) * C::A_BYTES;
        const uint8_t * bs = smem + (s & 1) * C::B_BYTES;
        const int co = ((2 * kstep + lg) ^ x) * 16;
#pragma unroll
        for (int i = 0; i < C::MI; i++) f.a[i] = *(const half8 *)(as + a_off + i * 32 * C::RB + co);
#pragma unroll
        for (int j = 0; j < C::NJ; j++) f.b[j] = *(const half8 *)(bs + b_off + j * 32 * C::RB + co);
    };
    // the MFMAs of one 16-deep K step; `part` 0 = only the first, 1 = all but the first
    auto mma = [&](const Frags & f, int part) {
#pragma unroll
        for (int i = 0; i < C::MI; i++)
#pragma unroll
            for (int j = 0; j < C::NJ; j++)
                if ((part == 0) == (i == 0 && j == 0)) acc[i][j] = mfma32(f.a[i], f.b[j], acc[i][j]);
    };
    constexpr int KST = C::DK / 16;
    const int kd = wave_s >= 4 ? 2 : 0;   // the K step at which this wave decodes
    Frags f0, f1;
    // stage s, J = s % 4
    auto stage = [&](int s, auto Jc) {
        constexpr int J = decltype(Jc)::value;
#pragma unroll
        for (int kstep = 0; kstep < KST; kstep++) {
            Frags & F = (kstep % 2 == 0) ? f0 : f1;
            Frags & G = (kstep % 2 == 0) ? f1 : f0;
            mma(F, 0);
            __builtin_amdgcn_sched_barrier(0);
            if (kstep + 1 < KST) {
                read_frags(s, kstep + 1, G);
                __builtin_amdgcn_sched_barrier(0);
            }
            if (kstep == kd) {
                wait_vm<C::PA + C::QD + (J == 2 ? 1 : 0)>();
                decode(s + 1, std::integral_constant<int, (J + 1) % 4>());
                __builtin_amdgcn_sched_barrier(0);
            }
            if (kstep + 1 == KST) {
                wait_vm_lgkm0<C::QD + (J == 2 ? 1 : 0)>();
                __builtin_amdgcn_s_barrier();
                read_frags(s + 1, 0, G);
                __builtin_amdgcn_sched_barrier(0);
                issue_a(s + 2);
                issue_q(s + 3);
                if (J == 1) issue_h(s / 4 + 1);   // the next block: its first decode is two stages on
                __builtin_amdgcn_sched_barrier(0);
            }
            mma(F, 1);
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    if (nk > 0) {
        // prologue: stage 0 decoded, then the DMA in the order the steady state has in flight
        // at the start of stage 0: nibbles of 1, activations of 1, nibbles of 2
        issue_h(0);
        issue_q(0);
        issue_a(0);
        wait_vm<0>();
        decode(0, std::integral_constant<int, 0>());
        __builtin_amdgcn_sched_barrier(0);
        issue_q(1);
        issue_a(1);
        issue_q(2);
        __builtin_amdgcn_sched_barrier(0);
        wait_vm_lgkm0<C::PA + 2 * C::QD>();   // this wave's LDS writes; the DMA stays in flight
        __builtin_amdgcn_s_barrier();
        read_frags(0, 0, f0);
        __builtin_amdgcn_sched_barrier(0);
        for (int s = 0; s < nk; s += 4) {
            stage(s, std::integral_constant<int, 0>());
            stage(s + 1, std::integral_constant<int, 1>());
            stage(s + 2, std::integral_constant<int, 2>());
            stage(s + 3, std::integral_constant<int, 3>());
        }
        wait_vm_lgkm0<0>();   // no DMA may still be writing this block's LDS when it exits
    }

    // epilogue: C = scale[m] * acc
    scale_rows(acc, args.scales, m0 + wm * C::TM, lg, M);
#pragma unroll
    for (int i = 0; i < C::MI; i++) {
#pragma unroll
        for (int e = 0; e < 16; e++) {
            const int r = m0 + wm * C::TM + i * 32 + 8 * (e / 4) + 4 * lg + (e % 4);
            if (r >= M) continue;
            float * crow = Cp + (int64_t)r * ldc;
#pragma unroll
            for (int j = 0; j < C::NJ; j++) {
                const int n = n0 + wn * C::TN + j * 32 + lr;
                if (n < N) {
                    if (ks == 1 || args.part) crow[n] = acc[i][j][e];
                    else unsafeAtomicAdd(crow + n, acc[i][j][e]);
                }
            }
        }
    }
}

// The K-split partials summed in split order, C_g[r][n] = P[0][r][pcol_g + n] + P[1][..] + ...:
// one thread per 4 columns of a partial row (every group's N and pcol are multiples of 16).
__global__ void __launch_bounds__(256) reduce_splits_kernel(GemmArgs a, int ks) {
    const int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t per_row = a.ldp / 4;
    if (q >= (int64_t)a.M * per_row) return;
    const int64_t r = q / per_row, c = 4 * (q % per_row);
    int g = 0;
#pragma unroll
    for (int i = 1; i < GEMM_MAX_GROUPS; i++)
        if (i < a.ng && c >= a.g[i].pcol) g = i;
    float * C = a.g[0].C;
    int64_t ldc = a.g[0].ldc, pcol = a.g[0].pcol;
#pragma unroll
    for (int i = 1; i < GEMM_MAX_GROUPS; i++)
        if (i == g) { C = a.g[i].C; ldc = a.g[i].ldc; pcol = a.g[i].pcol; }
    const int64_t slab = (int64_t)a.M * a.ldp;
    const float * p = a.part + r * a.ldp + c;
    float4v s = *(const float4v *)p;
    // loads in batches of 8 (all in flight at once), added in split order
    for (int k0 = 1; k0 < ks; k0 += 8) {
        float4v v[8];
#pragma unroll
        for (int j = 0; j < 8; j++) v[j] = k0 + j < ks ? *(const float4v *)(p + (k0 + j) * slab) : float4v{0, 0, 0, 0};
#pragma unroll
        for (int j = 0; j < 8; j++)
            if (k0 + j < ks)
#pragma unroll
                for (int e = 0; e < 4; e++) s[e] += v[j][e];
    }
    float * o = C + r * ldc + (c - pcol);
    if ((reinterpret_cast<uintptr_t>(o) & 15) == 0) {
        *(float4v *)o = s;
    } else {
#pragma unroll
        for (int e = 0; e < 4; e++) o[e] = s[e];
    }
}

// Zeroes the outputs a split-K launch adds into (a fill kernel rather than a memset, so the launch
// sequence stays capturable): one block per (row, weight group), 16-byte stores where the row
// start allows them.
__global__ void __launch_bounds__(256) zero_rows_kernel(GemmArgs args) {
    const GemmGroup & G = args.g[blockIdx.y];
    float * row = G.C + (int64_t)blockIdx.x * G.ldc;
    const int N = G.N;
    int c0 = 0;
    if ((reinterpret_cast<uintptr_t>(row) & 15) == 0) {
        for (int c = 4 * threadIdx.x; c + 3 < N; c += 4 * blockDim.x) *(float4v *)(row + c) = float4v{0, 0, 0, 0};
        c0 = N & ~3;
    }
    for (int c = c0 + threadIdx.x; c < N; c += blockDim.x) row[c] = 0.0f;
}

// ---------------------------------------------------------------------------------------------
// dequant to fp16 and the weight re-layout
// ---------------------------------------------------------------------------------------------

// One thread per (row, 32-value half of a 64-wide slab): the same decoders the GEMM uses.
template <int WT>
__global__ void __launch_bounds__(256) dequant_f16_kernel(const uint8_t * __restrict__ W, int64_t rows,
                                                          int64_t K, uint16_t * __restrict__ out) {
    const int64_t per_row = K / 32;   // thread items per row
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= rows * per_row) return;
    const int64_t row = i / per_row, item = i % per_row;
    const int64_t k0 = (item / 2) * 64;
    const int u = (int)(item % 2);
    WLoad<WT> wl;
    wl.load(W, rows, K, row, k0, u, true);
    u32x4 o[4];
    int run0, run1;
    wl.decode(u, o, run0, run1);
    uint16_t * d = out + row * K + k0;
    *(u32x4 *)(d + run0) = o[0];
    *(u32x4 *)(d + run0 + 8) = o[1];
    *(u32x4 *)(d + run1) = o[2];
    *(u32x4 *)(d + run1 + 8) = o[3];
}

// The same into the tiled layout: a wave takes 16 rows x 128 K (four whole tiles), a lane one
// 32-value half of one row's slab, and the decoded values pass through LDS so that each store of
// the wave is one tile, 1 KB of consecutive bytes. Bound by HBM: the quantized bytes in, two bytes a
// weight out. Storing from the decode, 16 bytes a lane of 64 rows' half lines, it took 1.3-2x the
// time of those bytes for the types of 32-value blocks: Q8_0 28672 x 4096 97.9 us, Q4_0 86.
// Chunk c (16 bytes) of a tile's row r sits at LDS chunk c ^ (r / 4 % 4) of the row: no bank conflict
// either way. Rows past the last one decode it again into the layout's padding, which nobody reads.
template <int WT>
__global__ void __launch_bounds__(256) dequant_tiled_kernel(const uint8_t * __restrict__ W, int64_t rows,
                                                            int64_t K, uint16_t * __restrict__ out) {
    __shared__ __align__(16) uint8_t st[4 * 4096];
    const int lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE;
    const int nkc = (int)((K + 511) / 512);   // 512 K a block
    const int b = xcd_tile(blockIdx.x, gridDim.x);   // neighbours in K share a row's lines in one L2
    const int64_t rb = b / nkc;
    const int64_t kw = (int64_t)(b % nkc) * 512 + wave * 128;
    uint8_t * ws = st + wave * 4096;
    const int r = lane % 16, j = lane / 16;
    const int64_t k0 = kw + 64 * (j / 2);
    if (k0 < K) {
        WLoad<WT> wl;
        wl.load(W, rows, K, min(rb * 16 + r, rows - 1), k0, j % 2, true);
        u32x4 o[4];
        int run[2];
        wl.decode(j % 2, o, run[0], run[1]);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int kk = 64 * (j / 2) + run[i / 2] + 8 * (i % 2);   // of the wave's 128
            *(u32x4 *)(ws + (kk / 32) * 1024 + r * 64 + ((((kk % 32) / 8) ^ (r / 4)) << 4)) = o[i];
        }
    }
    __syncthreads();
    const int lr = lane / 4, lc = (lane % 4) ^ (lr / 4);
#pragma unroll
    for (int i = 0; i < 4; i++)
        if (kw + 32 * i < K)
            *(u32x4 *)(out + tiled_index(rb * 16, kw + 32 * i, K) + 8 * lane) = *(const u32x4 *)(ws + i * 1024 + lr * 64 + lc * 16);
}

// F32 or BF16 values -> fp16 (round to nearest even): the resident form of an F32 / BF16 weight,
// as rocket_weight_to_fp16 makes it (ggml-rocket.cpp:3855-3890).
__global__ void convert_f16_kernel(int type, const void * __restrict__ src, int64_t n, uint16_t * __restrict__ dst) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float f;
    if (type == T_F32) f = ((const float *)src)[i];
    else f = __builtin_bit_cast(float, (uint32_t)((const uint16_t *)src)[i] << 16);
    dst[i] = f2h_bits(f);
}

// ggml Q8_0 -> split planes. One thread per block.
__global__ void pack_q8_0_kernel(const uint8_t * __restrict__ src, int64_t rows, int64_t K,
                                 uint8_t * __restrict__ dst) {
    const int64_t nb = K / 32;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= rows * nb) return;
    const int64_t row = i / nb, b = i % nb;
    const uint8_t * s = src + i * 34;
    uint8_t * qs = dst + row * K + b * 32;
    for (int l = 0; l < 32; l++) qs[l] = s[2 + l];
    uint8_t * d = dst + rows * K + (row * nb + b) * 2;
    d[0] = s[0];
    d[1] = s[1];
}

// ggml MXFP4 -> split planes. One thread per 17-byte block.
__global__ void pack_mxfp4_kernel(const uint8_t * __restrict__ src, int64_t rows, int64_t K,
                                  uint8_t * __restrict__ dst) {
    const int64_t nb = K / 32;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= rows * nb) return;
    const int64_t row = i / nb, b = i % nb;
    const uint8_t * s = src + i * 17;
    uint8_t * qs = dst + row * (K / 2) + b * 16;
    for (int l = 0; l < 16; l++) qs[l] = s[1 + l];
    dst[rows * (K / 2) + row * nb + b] = s[0];
}

// ggml Q4_0 -> split planes. One thread per block.
__global__ void pack_q4_0_kernel(const uint8_t * __restrict__ src, int64_t rows, int64_t K,
                                 uint8_t * __restrict__ dst) {
    const int64_t nb = K / 32;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= rows * nb) return;
    const int64_t row = i / nb, b = i % nb;
    const uint8_t * s = src + i * 18;
    uint8_t * qs = dst + row * (K / 2) + b * 16;
    for (int l = 0; l < 16; l++) qs[l] = s[2 + l];
    uint8_t * d = dst + rows * (K / 2) + (row * nb + b) * 2;
    d[0] = s[0];
    d[1] = s[1];
}

// ggml Q6_K -> split planes. One thread per block.
__global__ void pack_q6_k_kernel(const uint8_t * __restrict__ src, int64_t rows, int64_t K,
                                 uint8_t * __restrict__ dst) {
    const int64_t nb = K / 256;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= rows * nb) return;
    const int64_t row = i / nb, b = i % nb;
    const uint8_t * s = src + i * 210;
    uint8_t * ql = dst + row * (K / 2) + b * 128;
    uint8_t * qh = dst + rows * (K / 2) + row * (K / 4) + b * 64;
    uint8_t * sc = dst + rows * (K / 2) + rows * (K / 4) + row * (K / 16) + b * 16;
    uint8_t * d = dst + rows * (K / 2) + rows * (K / 4) + rows * (K / 16) + (row * nb + b) * 2;
    for (int l = 0; l < 128; l++) ql[l] = s[l];
    for (int l = 0; l < 64; l++) qh[l] = s[128 + l];
    for (int l = 0; l < 16; l++) sc[l] = s[192 + l];
    d[0] = s[208];
    d[1] = s[209];
}

// ---------------------------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------------------------

hipError_t launch_pack_act(const float * X, int64_t ldx, int M, int K, uint16_t * A16, int64_t lda,
                           float * scales, hipStream_t st, float * zc, int64_t ldzc, int zn) {
    if (M <= 0) return hipSuccess;
    constexpr int RPB = PACK_THREADS / WAVE;   // rows a block of the wave form
    if (K <= pack_wave_k())
        hipLaunchKernelGGL(pack_act_wave_kernel<false>, dim3((M + RPB - 1) / RPB), dim3(PACK_THREADS), 0, st, X, ldx,
                           M, K, A16, lda, scales, zc, ldzc, zn);
    else
        hipLaunchKernelGGL(pack_act_kernel<false>, dim3(M), dim3(PACK_THREADS), 0, st, X, ldx, M, K, A16, lda, scales,
                           zc, ldzc, zn);
    return hipGetLastError();
}

hipError_t launch_pack_act_tiled(const float * X, int64_t ldx, int M, int K, uint16_t * A16, float * scales,
                                 hipStream_t st, float * zc, int64_t ldzc, int zn) {
    if (M <= 0) return hipSuccess;
    constexpr int RPB = PACK_THREADS / WAVE;
    if (K <= pack_wave_k())
        hipLaunchKernelGGL(pack_act_wave_kernel<true>, dim3((M + RPB - 1) / RPB), dim3(PACK_THREADS), 0, st, X, ldx,
                           M, K, A16, (int64_t)K, scales, zc, ldzc, zn);
    else
        hipLaunchKernelGGL(pack_act_kernel<true>, dim3(M), dim3(PACK_THREADS), 0, st, X, ldx, M, K, A16, (int64_t)K,
                           scales, zc, ldzc, zn);
    return hipGetLastError();
}

// Tile configurations. The launcher picks one per call (choose_cfg); MI355X_GEMM_CFG=<id>
// forces one (for tuning and for the tests, which run every configuration).
//   0-3  register-staged kernel with the weight decoded into LDS: every weight type.
//   4-15 LDS-DMA kernel: row-major fp16 weights; 15 has wave columns of two widths
//        (gemm_f16_cols_kernel), 21 and 22 are that tile with 32-deep stages, three or four of
//        them in flight where 15 has one of 64 (the 256 x 224 tile's DMA waits are what bounds
//        it); 23 and 24 are 8 and 14 with eight 32-deep stages. Of these only 8, 9, 10 and 23
//        also take tiled weights, where 25-35 want a K split that has no workspace (choose_tiled).
//   25-35 one wave per SIMD (gemm_f16_1w_kernel): tiled fp16 weights, any K split.
//   16-19 Q4_K with every operand by DMA (gemm_q4k_kernel), K % 256 == 0; 18 and 19 split K
//        (q4k_split). 20 is the skinny kernel's id (use_skinny), not a tile configuration.
// choose_cfg prices a launch from two rates: a block's own pace, rounds * (ov_us + MFMA work
// of a block / tf_cu) (pipeline fill and epilogue, then its per-CU MFMA rate), and the
// aggregate rate at which the L2s feed the CUs for that tile shape, L2->CU bytes of all blocks
// / bw (bigger tiles fetch less per FLOP but keep fewer bytes in flight per CU). The two
// overlap, so the estimate is their 4-norm (pace^4 + feed^4)^(1/4), which follows the measured
// transition between the regimes better than the max; a split-K launch adds zc microseconds per
// MB of output (the zero fill and the second addend's atomics), or for 25-35 the reduction's
// launch and its slabs (ONEW_RED_US + ONEW_RED_US_MB per MB of partials). The four were fitted per
// configuration to measurements on tiled weights, each launch on a weight panel no earlier launch
// left in the caches: 4-24 at M = 128-2048, N = 1024-28672, K = 2880-14336, mean error 2-9% per
// configuration, and over 50 shapes the chosen configurations cost 0.6% more than the best
// measured ones; 25-32 at M = 48-2048, N = 1024-28672, K = 2048-14336 with splits of 1-8, mean error
// 4-10%; 35 has 25's rate with its other two scaled by the tile. 33 and 34, the small tiles, are set to the
// choices themselves, over 540 random shapes (M 16-2048, N 1024-28672, K 1024-14336, every tile and split):
// these cost 1.1% more than the best, 37 of them over 5% (fitted like 25-32, both were priced too low: 2.1%,
// 72 over 5%; 256 x 4096 x 4096 28.5 -> 22.9, 160 x 6144 x 4096 29.3 -> 24.3, 64 x 14336 x 4096 34.6 -> 28.0).
enum CfgKind { REG = 0, DMA = 1, Q4KDMA = 2, NONE = 3, ONEW = 4 };
struct CfgDesc {
    int kind;        // REG: gemm_kernel, DMA: gemm_f16_kernel / _cols, Q4KDMA: gemm_q4k_kernel,
                     // ONEW: gemm_f16_1w_kernel
    int bm, bn, ksplit;
    int dk;          // K per LDS stage (0 for the register-staged kernel)
    double tf_cu;    // TFLOP/s per CU
    double ov_us;    // fixed microseconds per block
    double bw;       // aggregate L2 -> CU TB/s
    double zc;       // split-K: microseconds per MB of output
};
static constexpr CfgDesc kCfgs[] = {
    {REG, 128, 128, 1, 0, 0.0, 0.0, 0.0, 0.0},        // 0: 4 waves of 64x64
    {REG, 128, 128, 2, 0, 0.0, 0.0, 0.0, 0.0},        // 1: same, K split (launcher-sized, >= 2)
    {REG, 256, 128, 1, 0, 0.0, 0.0, 0.0, 0.0},        // 2: 4 waves of 128x64
    {REG, 128, 256, 1, 0, 0.0, 0.0, 0.0, 0.0},        // 3: 4 waves of 64x128
    {DMA, 256, 256, 1, 64, 6.30, 6.0, 8.05, 0.00},   // 4: 8 waves of 64x128, 2 stages of 64
    {DMA, 128, 128, 1, 64, 4.03, 0.0, 13.00, 0.00},  // 5: 8 waves of 32x64, 4 stages of 64
    {DMA, 64, 128, 1, 128, 2.75, 5.0, 16.32, 0.00},  // 6: 4 waves of 32x64, 3 stages of 128
    {DMA, 128, 64, 1, 128, 2.92, 5.9, 16.88, 0.00},  // 7: 4 waves of 64x32, 3 stages of 128
    {DMA, 128, 128, 2, 64, 3.52, 0.0, 25.17, 1.76},  // 8: as 5, K split in two
    {DMA, 64, 128, 2, 128, 2.50, 6.3, 40.00, 0.69},  // 9: as 6, K split in two
    {DMA, 128, 128, 1, 32, 4.43, 0.0, 13.05, 0.00},  // 10: 8 waves of 32x64, 4 stages of 32 (any K)
    {DMA, 128, 128, 1, 32, 4.35, 0.0, 13.10, 0.00},  // 11: 8 waves of 32x64, 8 stages of 32
    {DMA, 256, 128, 1, 64, 5.62, 8.6, 10.70, 0.00},  // 12: 8 waves of 64x64, 3 stages of 64
    {DMA, 128, 256, 1, 64, 5.33, 6.9, 10.85, 0.00},  // 13: 8 waves of 64x64, 3 stages of 64
    {DMA, 64, 128, 1, 64, 2.60, 2.3, 17.23, 0.00},   // 14: 4 waves of 32x64, 6 stages of 64
    {DMA, 256, 224, 1, 64, 5.70, 0.0, 8.88, 0.00},   // 15: 8 waves of 64x128 and 64x96, 2 stages of 64
    {Q4KDMA, 256, 256, 1, 64, 0.0, 0.0, 0.0, 0.0}, // 16: Q4_K by DMA, 8 waves of 64x128
    {Q4KDMA, 128, 256, 1, 64, 0.0, 0.0, 0.0, 0.0}, // 17: Q4_K by DMA, 8 waves of 64x64
    {Q4KDMA, 256, 256, 2, 64, 0.0, 0.0, 0.0, 0.0}, // 18: as 16, K split (launcher-sized, >= 2)
    {Q4KDMA, 128, 256, 2, 64, 0.0, 0.0, 0.0, 0.0}, // 19: as 17, K split (launcher-sized, >= 2)
    {NONE, 0, 0, 1, 0, 0.0, 0.0, 0.0, 0.0},        // 20: the skinny kernel (not a tile configuration)
    {DMA, 256, 224, 1, 32, 7.07, 10.7, 9.00, 0.00},   // 21: as 15, 4 stages of 32
    {DMA, 256, 224, 1, 32, 6.78, 10.1, 8.73, 0.00},   // 22: as 15, 5 stages of 32
    {DMA, 128, 128, 2, 32, 3.59, 0.0, 17.89, 1.65},   // 23: as 8, 8 stages of 32
    {DMA, 64, 128, 1, 32, 2.70, 1.4, 17.12, 0.00},    // 24: as 14, 8 stages of 32
    {ONEW, 256, 224, 1, 32, 7.98, 8.86, 10.36, 0.00},  // 25: tiled weights, 4 waves of 128x112, 5 stages of 32
    {ONEW, 256, 192, 1, 32, 7.79, 7.09, 11.10, 0.00},  // 26: 128x96, 5 stages
    {ONEW, 256, 160, 1, 32, 7.38, 6.43, 11.92, 0.00},  // 27: 128x80, 5 stages
    {ONEW, 256, 128, 1, 32, 6.65, 5.42, 13.21, 0.00},  // 28: 128x64, 6 stages
    {ONEW, 128, 224, 1, 32, 6.44, 6.08, 12.43, 0.00},  // 29: 64x112, 6 stages
    {ONEW, 128, 192, 1, 32, 6.22, 5.35, 13.47, 0.00},  // 30: 64x96, 7 stages
    {ONEW, 128, 128, 1, 32, 5.70, 4.78, 14.32, 0.00},  // 31: 64x64, 9 stages
    {ONEW, 128, 96, 1, 32, 4.66, 3.69, 14.63, 0.00},   // 32: 64x48, 9 stages
    {ONEW, 128, 64, 1, 32, 3.32, 1.68, 22.03, 0.00},   // 33: 64x32, 9 stages
    {ONEW, 64, 128, 1, 32, 3.37, 4.33, 19.99, 0.00},   // 34: 32x64, 9 stages
    {ONEW, 256, 256, 1, 32, 7.98, 10.5, 9.50, 0.00},   // 35: 128x128, 5 stages
};
constexpr int FIRST_DMA_CFG = 4;
constexpr int N_CFGS = sizeof(kCfgs) / sizeof(kCfgs[0]);

template <int WT, int BM, int BN, int WM, int WN, int R, int KS>
static hipError_t launch_one(const GemmArgs & a, int nblocks, hipStream_t st) {
    using C = GemmCfg<BM, BN, WM, WN, R>;
    auto kern = gemm_kernel<WT, BM, BN, WM, WN, R, KS>;
    static bool attr = false;
    if (!attr) {
        hipError_t e = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS);
        if (e != hipSuccess) return e;
        attr = true;
    }
    hipLaunchKernelGGL(kern, dim3(nblocks), dim3(GEMM_THREADS), C::LDS, st, a);
    return hipGetLastError();
}

template <int BM, int BN, int WGM, int WGN, int DK, int NS, int KS, bool TL>
static hipError_t launch_f16(const GemmArgs & a, int nblocks, hipStream_t st) {
    using C = F16Cfg<BM, BN, WGM, WGN, DK, NS>;
    auto kern = gemm_f16_kernel<BM, BN, WGM, WGN, DK, NS, KS, TL>;
    static bool attr = false;
    if (!attr) {
        hipError_t e = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS);
        if (e != hipSuccess) return e;
        attr = true;
    }
    hipLaunchKernelGGL(kern, dim3(nblocks), dim3(C::THREADS), C::LDS, st, a);
    return hipGetLastError();
}

template <int BM, int BN0, int BN1, int DK, int NS>
static hipError_t launch_cols(const GemmArgs & a, int nblocks, hipStream_t st) {
    using C = ColsCfg<BM, BN0, BN1, DK, NS>;
    auto kern = gemm_f16_cols_kernel<BM, BN0, BN1, DK, NS>;
    static bool attr = false;
    if (!attr) {
        hipError_t e = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS);
        if (e != hipSuccess) return e;
        attr = true;
    }
    hipLaunchKernelGGL(kern, dim3(nblocks), dim3(C::THREADS), C::LDS, st, a);
    return hipGetLastError();
}

template <int BM, int BN, int WGM, int WGN, int NS>
static hipError_t launch_1w(const GemmArgs & a, int nblocks, hipStream_t st) {
    using C = OneWaveCfg<BM, BN, WGM, WGN, NS>;
    auto kern = gemm_f16_1w_kernel<BM, BN, WGM, WGN, NS>;
    static bool attr = false;
    if (!attr) {
        hipError_t e = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS);
        if (e != hipSuccess) return e;
        attr = true;
    }
    hipLaunchKernelGGL(kern, dim3(nblocks), dim3(C::THREADS), C::LDS, st, a);
    return hipGetLastError();
}

template <int WT, int BM, int WGM, int WGN>
static hipError_t launch_q4k(const GemmArgs & a, int nblocks, hipStream_t st) {
    using C = Q4kCfg<WT, BM, WGM, WGN>;
    auto kern = gemm_q4k_kernel<WT, BM, WGM, WGN>;
    static bool attr = false;
    if (!attr) {
        hipError_t e = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS);
        if (e != hipSuccess) return e;
        attr = true;
    }
    hipLaunchKernelGGL(kern, dim3(nblocks), dim3(C::THREADS), C::LDS, st, a);
    return hipGetLastError();
}

// row-major fp16 weights
static hipError_t launch_row_cfg(int cfg, const GemmArgs & a, int nblocks, hipStream_t st) {
    switch (cfg) {
        case 15: return launch_cols<256, 128, 96, 64, 2>(a, nblocks, st);
        case 21: return launch_cols<256, 128, 96, 32, 4>(a, nblocks, st);
        case 22: return launch_cols<256, 128, 96, 32, 5>(a, nblocks, st);
        case 23: return launch_f16<128, 128, 4, 2, 32, 8, 2, false>(a, nblocks, st);
        case 24: return launch_f16<64, 128, 2, 2, 32, 8, 1, false>(a, nblocks, st);
        case 4: return launch_f16<256, 256, 4, 2, 64, 2, 1, false>(a, nblocks, st);
        case 5: return launch_f16<128, 128, 4, 2, 64, 4, 1, false>(a, nblocks, st);
        case 6: return launch_f16<64, 128, 2, 2, 128, 3, 1, false>(a, nblocks, st);
        case 7: return launch_f16<128, 64, 2, 2, 128, 3, 1, false>(a, nblocks, st);
        case 8: return launch_f16<128, 128, 4, 2, 64, 4, 2, false>(a, nblocks, st);
        case 9: return launch_f16<64, 128, 2, 2, 128, 3, 2, false>(a, nblocks, st);
        case 10: return launch_f16<128, 128, 4, 2, 32, 4, 1, false>(a, nblocks, st);
        case 11: return launch_f16<128, 128, 4, 2, 32, 8, 1, false>(a, nblocks, st);
        case 12: return launch_f16<256, 128, 4, 2, 64, 3, 1, false>(a, nblocks, st);
        case 13: return launch_f16<128, 256, 2, 4, 64, 3, 1, false>(a, nblocks, st);
        case 14: return launch_f16<64, 128, 2, 2, 64, 6, 1, false>(a, nblocks, st);
        default: return hipErrorInvalidValue;
    }
}

// tiled fp16 weights
static hipError_t launch_tiled_cfg(int cfg, const GemmArgs & a, int nblocks, hipStream_t st) {
    switch (cfg) {
        case 8: return launch_f16<128, 128, 4, 2, 64, 4, 2, true>(a, nblocks, st);
        case 9: return launch_f16<64, 128, 2, 2, 128, 3, 2, true>(a, nblocks, st);
        case 10: return launch_f16<128, 128, 4, 2, 32, 4, 1, true>(a, nblocks, st);
        case 23: return launch_f16<128, 128, 4, 2, 32, 8, 2, true>(a, nblocks, st);
        case 25: return launch_1w<256, 224, 2, 2, 5>(a, nblocks, st);
        case 26: return launch_1w<256, 192, 2, 2, 5>(a, nblocks, st);
        case 27: return launch_1w<256, 160, 2, 2, 5>(a, nblocks, st);
        case 28: return launch_1w<256, 128, 2, 2, 6>(a, nblocks, st);
        case 29: return launch_1w<128, 224, 2, 2, 6>(a, nblocks, st);
        case 30: return launch_1w<128, 192, 2, 2, 7>(a, nblocks, st);
        case 31: return launch_1w<128, 128, 2, 2, 9>(a, nblocks, st);
        case 32: return launch_1w<128, 96, 2, 2, 9>(a, nblocks, st);
        case 33: return launch_1w<128, 64, 2, 2, 9>(a, nblocks, st);
        case 34: return launch_1w<64, 128, 2, 2, 9>(a, nblocks, st);
        case 35: return launch_1w<256, 256, 2, 2, 5>(a, nblocks, st);
        default: return hipErrorInvalidValue;
    }
}

template <int WT>
static hipError_t launch_cfg(int cfg, const GemmArgs & a, int nblocks, hipStream_t st) {
    if (kCfgs[cfg].kind == Q4KDMA) {
        if constexpr (WT == T_Q4_K) {
            switch (cfg) {
                case 16: case 18: return launch_q4k<T_Q4_K, 256, 4, 2>(a, nblocks, st);
                case 17: case 19: return launch_q4k<T_Q4_K, 128, 2, 4>(a, nblocks, st);
                default: return hipErrorInvalidValue;
            }
        } else if constexpr (WT == T_Q8_0) {
            switch (cfg) {
                case 17: case 19: return launch_q4k<T_Q8_0, 128, 2, 4>(a, nblocks, st);
                default: return hipErrorInvalidValue;
            }
        } else {
            return hipErrorInvalidValue;
        }
    }
    if constexpr (WT == T_F16T) return launch_tiled_cfg(cfg, a, nblocks, st);
    else if (kCfgs[cfg].kind == DMA) return WT == T_F16 ? launch_row_cfg(cfg, a, nblocks, st) : hipErrorInvalidValue;
    else switch (cfg) {
        case 0: return launch_one<WT, 128, 128, 2, 2, 2, 1>(a, nblocks, st);
        case 1: return launch_one<WT, 128, 128, 2, 2, 2, 0>(a, nblocks, st);   // split a.ksplit ways
        case 2: return launch_one<WT, 256, 128, 2, 2, 2, 1>(a, nblocks, st);
        case 3: return launch_one<WT, 128, 256, 2, 2, 2, 1>(a, nblocks, st);
        default: return hipErrorInvalidValue;
    }
}

static int cu_count() {
    static int n = 0;
    if (n == 0) {
        int dev = 0;
        hipDeviceProp_t p;
        n = (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&p, dev) == hipSuccess) ? p.multiProcessorCount : 256;
    }
    return n;
}

static int tiles_of(const GemmArgs & a, int bm, int bn) {
    int nt = 0;
    for (int i = 0; i < a.ng; i++) nt += (a.g[i].N + bn - 1) / bn;
    return nt * ((a.M + bm - 1) / bm);
}

static int64_t total_cols(const GemmArgs & a) {
    int64_t n = 0;
    for (int i = 0; i < a.ng; i++) n += a.g[i].N;
    return n;
}

// The K split of the register-staged split configuration (1). Fitted to the fastest split
// measured for Q4_K and Q8_0 at M 32-512, N 3072-14336, K 3072-8192 (1% over the best in
// total): ~6.65 K^0.75 / sqrt(M N). A wider output has more elements to add atomically per
// split, a deeper K more work to share. At least 2 ways, at most 16 and at least 4 K slabs per
// split. MI355X_GEMM_KSPLIT=<n> forces n (for tuning).
static double reg_split_est(const GemmArgs & a) {
    return 6.65 * std::pow((double)a.K, 0.75) / std::sqrt((double)a.M * (double)total_cols(a));
}
static int reg_split(const GemmArgs & a, int cap) {
    const int nk = (a.K + BK - 1) / BK;
    if (const char * e = getenv("MI355X_GEMM_KSPLIT")) {
        const int v = atoi(e);
        if (v >= 2 && v <= nk) return std::min(v, cap);
    }
    int ks = (int)std::lround(reg_split_est(a));
    const int most = std::min(nk / 4 < 16 ? nk / 4 : 16, cap);
    if (ks > most) ks = most;
    return ks < 2 ? 2 : ks;
}

// The K split of the Q4_K DMA split configurations (18, 19): about one block per CU, in whole
// Q4_K blocks of K, at least 2 ways and at least 2 blocks (8 stages) a split.
// MI355X_GEMM_KSPLIT=<n> forces n (for tuning).
static int q4k_split(const GemmArgs & a, int bm, int bn, int cap) {
    const int nsb = a.K / 256;
    const int most = std::min(std::max(2, nsb / 2), cap);
    int ks = 0;
    if (const char * e = getenv("MI355X_GEMM_KSPLIT")) ks = atoi(e);
    if (ks < 2) ks = (int)std::lround((double)cu_count() / tiles_of(a, bm, bn));
    ks = std::min(std::max(ks, 2), most);
    // equal splits of whole blocks: the count that leaves no split empty
    const int per = (nsb + ks - 1) / ks;
    return (nsb + per - 1) / per;
}

// gemm_f16_1w_kernel addresses a tile's rows by 32-bit byte offsets (up to 17 row blocks of 32 K bytes)
constexpr int ONE_WAVE_MAX_K = 1 << 21;
static_assert(17LL * 32 * ONE_WAVE_MAX_K < 0x7FFFFFFF, "32-bit offsets");

static bool cfg_fits(int c, int wt, int K) {
    const CfgDesc & d = kCfgs[c];
    if (d.kind == NONE) return false;
    if (d.kind == REG) return wt != T_F16T;
    if (d.kind == Q4KDMA) return (wt == T_Q4_K || (wt == T_Q8_0 && d.bm == 128)) && K % 256 == 0;
    if (d.kind == ONEW) return wt == T_F16T && K % d.dk == 0 && K <= ONE_WAVE_MAX_K;
    if (wt == T_F16T && c != 8 && c != 9 && c != 10 && c != 23) return false;
    if ((wt != T_F16 && wt != T_F16T) || K % d.dk) return false;
    return d.ksplit == 1 || K / d.dk >= 2;
}

// A configuration's estimated microseconds with a K split (the CfgDesc model), and for the one-wave
// kernel the reduction of its split: a launch, and its slabs written and read back.
constexpr double ONEW_RED_US = 4.65, ONEW_RED_US_MB = 0.335;
// `tiles`: the launch's output tiles, out_mb: its output; an estimate known to pass `limit` (from
// its larger term) is returned as the limit, without the roots.
static double cfg_estimate(const CfgDesc & d, int K, int tiles, double out_mb, int ks, int cus, double limit) {
    const int blocks = tiles * ks;
    const int rounds = (blocks + cus - 1) / cus;
    const double kb = (double)K / ks;
    const double pace = rounds * (d.ov_us + 2.0 * d.bm * d.bn * kb / (d.tf_cu * 1e6));
    const double feed = (double)blocks * (d.bm + d.bn) * kb * 2.0 / (d.bw * 1e6);
    const double split = ks == 1 ? 0.0 : d.kind == ONEW ? ONEW_RED_US + ONEW_RED_US_MB * ks * out_mb : d.zc * out_mb;
    if (std::max(pace, feed) + split >= limit) return limit;
    const double p2 = pace * pace, f2 = feed * feed;
    return std::sqrt(std::sqrt(p2 * p2 + f2 * f2)) + split;
}

// The least estimate among the tiled-weight configurations of one kind, the one-wave kernel's with every
// split of at most `slabs` that leaves a split at least 512 values of K (16 stages; shorter ones are
// mostly pipeline fill), the eight-wave kernel's with their own. Keeps the given best unless beaten.
static void least_tiled(const GemmArgs & a, int kind, int slabs, double & best, int & cfg, int & ks) {
    const int cus = cu_count();
    const double out_mb = (double)a.M * (double)total_cols(a) * 4.0 / 1e6;
    for (int c = FIRST_DMA_CFG; c < N_CFGS; c++) {
        const CfgDesc & d = kCfgs[c];
        if (d.kind != kind || !cfg_fits(c, T_F16T, a.K)) continue;
        const int tiles = tiles_of(a, d.bm, d.bn);
        for (int s : {1, 2, 3, 4, 6, 8}) {
            if (kind == DMA ? s != d.ksplit : s > 1 && (s > slabs || a.K / s < 512)) continue;
            const double us = cfg_estimate(d, a.K, tiles, out_mb, s, cus, best);
            if (us < best - 1e-9) { best = us; cfg = c; ks = s; }
        }
    }
}

// Tiled fp16 weights: the one-wave kernel with its best K split where the workspace holds that split's
// slabs, whatever room is left beside them: the bytes gemm_split_bytes asks for and any more give the same
// launch. With fewer, its best split that fits, against the two-way atomic splits of the eight-wave kernel
// where not even two slabs do (a deep K over few tiles is faster split: 512 x 4096 x 14336 83 us against
// 91; a launch that wanted no split keeps the one-wave tile: 28 x 2560 x 1536 10.0 us against 11.8). K past
// ONE_WAVE_MAX_K: the eight-wave kernel alone.
static void choose_tiled(const GemmArgs & a, int slabs, int & cfg, int & ks) {
    const bool onew = a.K <= ONE_WAVE_MAX_K;
    double best = 1e30;
    cfg = 10;
    ks = 1;
    if (onew) {
        least_tiled(a, ONEW, 64, best, cfg, ks);
        if (ks <= std::max(slabs, 1)) return;
        best = 1e30;
        least_tiled(a, ONEW, slabs, best, cfg, ks);
    }
    if (!onew || slabs < 2) least_tiled(a, DMA, slabs, best, cfg, ks);
}

// Row-major fp16 weights: the DMA configuration with the least estimated time (the CfgDesc model;
// every DMA block has a CU to itself, so a launch runs in ceil(blocks / CUs) rounds).
// Q4_K weights (K % 256 == 0): the all-DMA kernel where it fills the chip (below).
// Other weights: split K when the output is skinny for its depth (reg_split), otherwise the
// unsplit register-staged tile with the best grid fill times its relative per-CU efficiency
// (bigger wave tiles read LDS less per MFMA).
static int choose_cfg(int wt, const GemmArgs & a) {
    if (const char * e = getenv("MI355X_GEMM_CFG")) {
        if (*e) {
            const int c = atoi(e);
            if (c >= 0 && c < N_CFGS && cfg_fits(c, wt, a.K)) return c;
        }
    }
    const int cus = cu_count();
    if (wt == T_F16) {
        int best = -1;
        double best_us = 1e30;
        const double out_mb = (double)a.M * (double)total_cols(a) * 4.0 / 1e6;
        for (int c = FIRST_DMA_CFG; c < N_CFGS; c++) {
            if (kCfgs[c].kind != DMA || !cfg_fits(c, wt, a.K)) continue;
            const CfgDesc & d = kCfgs[c];
            // the model was fitted on tiled weights; on row-major ones a 32-deep stage reads half
            // cache lines per row (qkv at M 512: 496 against 613 TFLOP/s for 64-deep stages), so
            // it is left to the K % 64 != 0 shapes that nothing else takes
            if (d.dk == 32 && a.K % 64 == 0) continue;
            const double us = cfg_estimate(d, a.K, tiles_of(a, d.bm, d.bn), out_mb, d.ksplit, cus, best_us);
            if (us < best_us - 1e-9) { best = c; best_us = us; }
        }
        if (best >= 0) return best;
    }
    // Q4_K with whole blocks: the all-DMA kernel where its tiles fill the chip in one round or
    // more (a 256 x 256 block runs a 64-deep stage in about 2.2 us, a 128 x 256 one in 1.3 us),
    // and its K split where K is deep for the output width. Measured on Q4_K at M 256-2048 for
    // the four projections of an 8B model (qkv 6144 x 4096, o 4096 x 4096, gate/up 28672 x 4096,
    // down 4096 x 14336), these picks are the fastest configuration or within 4% of it, and
    // 1.2-1.4x faster than the register-staged kernel where they apply.
    if (wt == T_Q4_K && a.K % 256 == 0) {
        const int fill = (cus * 7 + 9) / 10;
        if ((int64_t)a.K >= 2 * total_cols(a)) return a.M <= 1024 ? 19 : 18;
        if (tiles_of(a, 256, 256) >= fill) return 16;
        if (tiles_of(a, 128, 256) >= fill) return 17;
    }
    // Q8_0 with whole blocks: the all-DMA kernel on its 128 x 256 tiles, K split where K is deep
    // for the output width or the tiles fill less than half the chip. Measured at M 512 and 2048
    // for N x K in {3072, 8192} x {3072, 8192} and the 8B shapes 14336 x 4096 / 4096 x 14336, the
    // pick is the faster of the two, and 1.1-1.6x faster than the register-staged kernel.
    if (wt == T_Q8_0 && a.K % 256 == 0) {
        const int fill = (cus * 7 + 9) / 10;
        if (((int64_t)a.K >= 2 * total_cols(a) && a.M <= 1024) || tiles_of(a, 128, 256) < fill / 2) return 19;
        return 17;
    }
    // a skinny output: split K (see reg_split); otherwise the unsplit tile with the best fill
    if (reg_split_est(a) >= 1.5 && (a.K / BK) >= 8) return 1;
    const double tile_eff[FIRST_DMA_CFG] = {1.0, 0.97, 1.25, 1.25};
    int best = 0;
    double best_score = -1.0;
    for (int c = 0; c < FIRST_DMA_CFG; c++) {
        if (kCfgs[c].ksplit > 1) continue;
        const int tiles = tiles_of(a, kCfgs[c].bm, kCfgs[c].bn);
        const int blocks = tiles * kCfgs[c].ksplit;
        const int waves = (blocks + cus - 1) / cus;
        const double fill = (double)blocks / ((double)waves * cus);
        const double score = fill * tile_eff[c];
        if (score > best_score + 1e-9) { best_score = score; best = c; }
    }
    return best;
}

__global__ void zero_rows_kernel(GemmArgs args);

// The skinny kernel (configuration 20 for MI355X_GEMM_CFG): every weight format but the tiled
// fp16 one, M <= SK_MAX_M.
constexpr int SKINNY_CFG = 20;
static_assert(kCfgs[SKINNY_CFG].kind == NONE, "the skinny kernel's id");

// Row-major fp16 weights also have the DMA kernels: past M = 32 those win unless K is deep for
// the output width (measured at M 32-128; at M 128, K 14336 x N 4096: 50 us skinny, 60 us DMA;
// N 14336 x K 4096: 51 us skinny, 44 us DMA).
static bool use_skinny(int wt, const GemmArgs & a) {
    if (wt == T_F16T || a.M > SK_MAX_M) return false;
    if (const char * e = getenv("MI355X_GEMM_CFG"))
        if (*e) return atoi(e) == SKINNY_CFG;
    if (wt == T_F16 && a.M > 32 && (int64_t)a.K < 2 * total_cols(a)) return false;
    return true;
}

// A skinny launch's block: nw waves of 32 weight rows, kw ways along K, chunk depth ch; gpb groups
// a block, ks blocks along K (at most `cap`).
struct SkinnyShape { int ch, nw, kw, gpb, ks; };
static int skinny_ntiles(const GemmArgs & a, int nw) {
    int nt = 0;
    for (int i = 0; i < a.ng; i++) nt += (a.g[i].N + 32 * nw - 1) / (32 * nw);
    return nt;
}
// the blocks of one round of the chip: one a CU
static int skinny_blocks() {
    if (const char * e = getenv("MI355X_SKINNY_BLOCKS")) {   // tuning override
        const int v = atoi(e);
        if (v > 0) return v;
    }
    return cu_count();
}
static SkinnyShape skinny_split(const GemmArgs & a, int cap, int ch, int nw, int kw, int blocks) {
    const int nchunks = (a.K + 63) / 64, ngroups = (nchunks + ch - 1) / ch;
    const int steps = (ngroups + kw - 1) / kw;
    const int ks = std::min(std::max(1, blocks / skinny_ntiles(a, nw)), cap);
    const int gpb = (steps + ks - 1) / ks * kw;
    return {ch, nw, kw, gpb, (ngroups + gpb - 1) / gpb};
}
// The block by width, K, M and type, measured over N 1024-28672, K 1024-14336, M 1-128 and seven weight
// types (us, Q4_K unless named; B blocks make one round of the chip, one a CU):
//   64-wide blocks with four K ways while they make one round, the K split then the largest whose
//     blocks stay within it: half the slabs of 128-wide blocks with two ways (8192 x 3072 M 64 18.6
//     against 22.8), although each reads the activations for fewer columns; rounding that split up took
//     a second round (14336 x 4096 M 8 15-30% slower).
//   past one round 128-wide blocks with two ways, which need no K split and read the activations
//     half as often (28672 x 4096 M 64 / 128: 41.5 / 56.3 against 51.1 / 76.9; four ways of one chunk
//     43.7, spilling past 64 rows). Up to 32 rows and from K 4096 on, one way and two blocks a CU where three
//     K splits of such blocks fit in that, 129-170 tiles (17920 x 4096 M 1: Q8_0 43.5 -> 35.5, Q6_K 55.6 -> 43.5,
//     MXFP4 32.3 -> 28.5, Q5_K 42.0 -> 34.4), and for Q8_0, unsplit, past that too (28672 x 4096 M 1 / 32 47.6 /
//     49.1 -> 45.3 / 45.8; other types 0-10% slower).
//   the same 128-wide blocks of two ways, split three ways, where 64-wide ones make less than 2/3 of a
//     round and the three splits fit in one, 129-170 tiles of 64 (9536 x 6400, 149 tiles, M 2 / 100: Q8_0 31.6 /
//     44.0 against 35.5 / 50.9, Q4_K 24.4 / 44.3 against 29.0 / 54.5); from 160 tiles on only past 64 rows, for
//     Q6_K, Q5_K and F16, or from K 8192 on (10240 x 4096 M 32 20.4 the 64-wide way, 21.9 this; M 100 39.9, 35.0; Q6_K
//     M 64 37.2, 31.8), and never under K 2560, where the slabs cost more than the idle CUs (9216 x 1792 M 112 MXFP4
//     28.8 against 21.9).
//   128-wide blocks too where their K split fills a round better by a sixteenth or more: of one way for
//     Q8_0 and F16 up to 32 rows, from K 8192 on or where four ways split in three (4608 x 14336 M 1 Q8_0 0.86 of
//     the time, 4608 x 5376 0.94; the lighter types 0-10% slower there); of two ways past 32 rows, from K 8192 on
//     (6144 x 8192 M 100 42.0 -> 38.1), and for MXFP4 past 64 rows even where both fill it (4096 x 14336 M 100
//     41.1 -> 37.9).
//   chunk depth 1 past 64 rows (the slices of four ways fill LDS); up to 64 rows depth 2 (14336 x 4096
//     M 64 28.5 against 32.0), except where its coarser steps leave a block more of K than depth 1
//     would (3072 x 3072 M 8: 4 against 3 depth-1 steps, 13.9 against 12.9). A block of one depth-2 step
//     stays while that spares it the slabs (1024 x 1024, two splits: 8.2 against 10.5; but 1536 x 1536 M 16,
//     three or six: 11.5 against 10.9). In 128-wide blocks depth 1 by the same rule for Q6_K, Q5_K and MXFP4
//     where they split K (9984 x 4096 M 1 / 64, 22 against 24 chunks: Q6_K 31.2 / 36.2 -> 27.1 / 32.0, MXFP4 M 100
//     36.0 -> 32.5; Q4_K M 64 0.4 slower), and for Q6_K up to 64 rows where they don't (28672 x 4096 M 64 60.7 ->
//     59.0).
//   one way of depth 4, up to 16 rows and K 2048, where its blocks make one step of 4 chunks and the four
//     ways' one of 8: no merge, and nothing to overlap (2464 x 1792 M 6 11.4 -> 11.0; Q6_K and Q5_K 3% slower).
static SkinnyShape skinny_shape(int wt, const GemmArgs & a, int cap) {
    const int B = skinny_blocks(), n2 = skinny_ntiles(a, 2), n4 = skinny_ntiles(a, 4);
    auto split = [&](int ch, int nw, int kw) { return skinny_split(a, cap, ch, nw, kw, B); };
    auto chunks = [](const SkinnyShape & s) { return s.gpb * s.ch; };
    const bool few = a.M <= 32;
    if (n2 > B) {
        if (few && a.K >= 4096 && cap >= 3 && 3 * n4 <= 2 * B) return skinny_split(a, cap, 2, 4, 1, 2 * B);
        if (few && wt == T_Q8_0) return split(2, 4, 1);
        return split(wt == T_Q6_K && a.M <= 64 ? 1 : 2, 4, 2);
    }
    if (2 * n2 > B && 3 * n4 <= B && a.K >= 2560 &&
        (8 * n2 < 5 * B || (cap >= 3 && (a.M > 64 || wt == T_Q6_K || wt == T_Q5_K || wt == T_F16 || a.K >= 8192)))) {
        const SkinnyShape s1 = split(1, 4, 2), s2 = split(2, 4, 2);
        const bool fine = wt == T_Q6_K || wt == T_Q5_K || wt == T_MXFP4;
        return fine && chunks(s1) < chunks(s2) ? s1 : s2;
    }
    const int k2 = B / n2, k4 = B / n4;   // the K splits
    const bool fuller = 16 * (k4 * n4 - k2 * n2) >= B && cap >= k4;
    if (few) {
        if ((wt == T_Q8_0 || wt == T_F16) && fuller && (a.K >= 8192 || (k2 == 3 && a.K >= 1792))) return split(2, 4, 1);
    } else if (a.K >= 8192 && k2 >= 2) {
        if (fuller && (a.M > 64 || k2 >= 3)) return split(1, 4, 2);
        if (wt == T_MXFP4 && a.M > 64 && k2 <= 6 && cap >= k4) return split(1, 4, 2);
    }
    const SkinnyShape s1 = split(1, 2, 4);
    if (a.M > 64) return s1;
    const SkinnyShape s2 = split(2, 2, 4);
    if (chunks(s1) < chunks(s2) && (s2.gpb > s2.kw || s2.ks > 2)) return s1;
    if (a.M <= 16 && a.K <= 2048 && s2.gpb == s2.kw && s2.ks > 2 && wt != T_Q6_K && wt != T_Q5_K) {
        const SkinnyShape s4 = split(4, 4, 1);
        if (s4.gpb == 1) return s4;
    }
    return s2;
}

template <int WT, int MT, int CH, int NW, int KW>
static hipError_t launch_skinny1(const GemmArgs & a, int nblocks, int gpb, hipStream_t st) {
    auto kern = gemm_skinny_kernel<WT, MT, CH, NW, KW>;
    constexpr int lds = skinny_lds<MT, CH, NW, KW>();
    static bool attr = false;
    if (!attr) {
        const hipError_t e = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        if (e != hipSuccess) return e;
        attr = true;
    }
    hipLaunchKernelGGL(kern, dim3(nblocks), dim3(NW * KW * WAVE), lds, st, a, gpb);
    return hipGetLastError();
}

template <int WT>
static hipError_t launch_skinny(const GemmArgs & a, int nblocks, const SkinnyShape & s, hipStream_t st) {
    auto go = [&](auto m) {
        constexpr int MT = decltype(m)::value;
        if constexpr (MT == 1)
            if (s.kw == 1) return s.ch == 4 ? launch_skinny1<WT, MT, 4, 4, 1>(a, nblocks, s.gpb, st)
                                            : launch_skinny1<WT, MT, 2, 4, 1>(a, nblocks, s.gpb, st);
        if (s.nw == 2) {
            if constexpr (MT <= 2)
                if (s.ch == 2) return launch_skinny1<WT, MT, 2, 2, 4>(a, nblocks, s.gpb, st);
            return launch_skinny1<WT, MT, 1, 2, 4>(a, nblocks, s.gpb, st);
        }
        if (s.ch == 1) return launch_skinny1<WT, MT, 1, 4, 2>(a, nblocks, s.gpb, st);
        return launch_skinny1<WT, MT, 2, 4, 2>(a, nblocks, s.gpb, st);
    };
    switch ((a.M + 31) / 32) {
        case 1: return go(std::integral_constant<int, 1>());
        case 2: return go(std::integral_constant<int, 2>());
        case 3: return go(std::integral_constant<int, 3>());
        default: return go(std::integral_constant<int, 4>());
    }
}

// A launch's configuration and K split. A split past two ways takes a slab of the caller's
// workspace per way; the one-wave kernel's always does.
struct GemmPlan {
    bool skinny;
    int cfg;      // kCfgs index (unused for the skinny kernel)
    int ks;       // K split
    SkinnyShape sk;   // skinny kernel: its block and K groups per block
    bool slabs;   // each split writes its slab of the partials (else two ways, added into the output)
};

// partial slabs [M][sum of N] the workspace holds, at most 64
static int split_slabs(const GemmArgs & a, size_t part_bytes) {
    const size_t slab = (size_t)a.M * (size_t)total_cols(a) * sizeof(float);
    return (int)std::min<size_t>(slab ? part_bytes / slab : 0, 64);
}

static GemmPlan plan_gemm(int wt, const GemmArgs & a, int slabs) {
    GemmPlan p{};
    const int cap = std::max(slabs, 2);   // two ways need no slab: they add into the output
    if (wt == T_F16T) {
        const char * e = getenv("MI355X_GEMM_CFG");
        const int forced = (e && *e) ? atoi(e) : -1;
        if (forced >= 0 && forced < N_CFGS && cfg_fits(forced, wt, a.K)) {
            p.cfg = forced;
            p.ks = kCfgs[forced].ksplit;
            if (const char * k = getenv("MI355X_GEMM_KSPLIT"))
                if (kCfgs[forced].kind == ONEW) p.ks = std::min(std::max(atoi(k), 1), std::max(slabs, 1));
        } else {
            choose_tiled(a, slabs, p.cfg, p.ks);
        }
        p.slabs = kCfgs[p.cfg].kind == ONEW && p.ks > 1;
        return p;
    }
    if (use_skinny(wt, a)) {
        p.skinny = true;
        p.cfg = SKINNY_CFG;
        p.sk = skinny_shape(wt, a, cap);
        p.ks = p.sk.ks;
        p.slabs = p.ks > 2;
        return p;
    }
    p.cfg = choose_cfg(wt, a);
    const CfgDesc & d = kCfgs[p.cfg];
    p.ks = p.cfg == 1 ? reg_split(a, cap)
         : (d.kind == Q4KDMA && d.ksplit > 1) ? q4k_split(a, d.bm, d.bn, cap) : d.ksplit;
    p.slabs = p.ks > 2;
    return p;
}

bool gemm_one_round(int wt, const GemmArgs & a) {
    const GemmPlan p = plan_gemm(wt, a, 64);
    return !p.skinny && (int64_t)tiles_of(a, kCfgs[p.cfg].bm, kCfgs[p.cfg].bn) * p.ks <= cu_count();
}

size_t gemm_split_bytes(int wt, const GemmArgs & a) {
    const GemmPlan p = plan_gemm(wt, a, 64);
    return p.slabs ? (size_t)p.ks * (size_t)a.M * (size_t)total_cols(a) * sizeof(float) : 0;
}

bool gemm_accumulates(int wt, const GemmArgs & a, size_t part_bytes) {
    const GemmPlan p = plan_gemm(wt, a, split_slabs(a, part_bytes));
    return p.ks == 2 && !p.slabs;
}

hipError_t launch_gemm(int wt, const GemmArgs & a_in, int /*unused*/, hipStream_t st, bool c_zeroed, float * part,
                       size_t part_bytes) {
    GemmArgs a = a_in;
    const GemmPlan p = plan_gemm(wt, a, part ? split_slabs(a, part_bytes) : 0);
    const int bn = p.skinny ? 32 * p.sk.nw : kCfgs[p.cfg].bn;
    int nt = 0;
    int64_t pcol = 0;
    for (int i = 0; i < a.ng; i++) {
        a.g[i].ntile_begin = nt;
        nt += (a.g[i].N + bn - 1) / bn;
        a.g[i].pcol = pcol;
        pcol += a.g[i].N;
    }
    a.m_tiles = p.skinny ? 1 : (a.M + kCfgs[p.cfg].bm - 1) / kCfgs[p.cfg].bm;
    a.ksplit = p.ks;
    a.part = p.slabs ? part : nullptr;
    a.ldp = pcol;
    const int nblocks = nt * a.m_tiles * a.ksplit;
    if (nblocks <= 0) return hipSuccess;
    if (p.ks == 2 && !p.slabs && !c_zeroed) {
        hipLaunchKernelGGL(zero_rows_kernel, dim3(a.M, a.ng), dim3(256), 0, st, a);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    hipError_t e = hipErrorInvalidValue;
    if (p.skinny) {
        switch (wt) {
            case T_F16: e = launch_skinny<T_F16>(a, nblocks, p.sk, st); break;
            case T_Q8_0: e = launch_skinny<T_Q8_0>(a, nblocks, p.sk, st); break;
            case T_Q4_0: e = launch_skinny<T_Q4_0>(a, nblocks, p.sk, st); break;
            case T_Q4_K: e = launch_skinny<T_Q4_K>(a, nblocks, p.sk, st); break;
            case T_Q5_K: e = launch_skinny<T_Q5_K>(a, nblocks, p.sk, st); break;
            case T_Q6_K: e = launch_skinny<T_Q6_K>(a, nblocks, p.sk, st); break;
            case T_MXFP4: e = launch_skinny<T_MXFP4>(a, nblocks, p.sk, st); break;
            default: break;
        }
    } else {
        switch (wt) {
            case T_F16: e = launch_cfg<T_F16>(p.cfg, a, nblocks, st); break;
            case T_F16T: e = launch_cfg<T_F16T>(p.cfg, a, nblocks, st); break;
            case T_Q8_0: e = launch_cfg<T_Q8_0>(p.cfg, a, nblocks, st); break;
            case T_Q4_0: e = launch_cfg<T_Q4_0>(p.cfg, a, nblocks, st); break;
            case T_Q4_K: e = launch_cfg<T_Q4_K>(p.cfg, a, nblocks, st); break;
            case T_Q5_K: e = launch_cfg<T_Q5_K>(p.cfg, a, nblocks, st); break;
            case T_Q6_K: e = launch_cfg<T_Q6_K>(p.cfg, a, nblocks, st); break;
            case T_MXFP4: e = launch_cfg<T_MXFP4>(p.cfg, a, nblocks, st); break;
            default: break;
        }
    }
    if (e != hipSuccess || !a.part) return e;
    const int64_t threads = (int64_t)a.M * (a.ldp / 4);
    hipLaunchKernelGGL(reduce_splits_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, st, a, a.ksplit);
    return hipGetLastError();
}

template <bool TL>
static hipError_t launch_dequant(int wt, const void * W, int64_t rows, int64_t K, uint16_t * out, hipStream_t st) {
    if (rows <= 0 || K <= 0) return hipSuccess;
    const dim3 grid((unsigned)(TL ? (rows + 15) / 16 * ((K + 511) / 512) : (rows * (K / 32) + 255) / 256));
    const uint8_t * w = (const uint8_t *)W;
    auto go = [&](auto t) {
        constexpr int WT = decltype(t)::value;
        if constexpr (TL) hipLaunchKernelGGL(dequant_tiled_kernel<WT>, grid, dim3(256), 0, st, w, rows, K, out);
        else hipLaunchKernelGGL(dequant_f16_kernel<WT>, grid, dim3(256), 0, st, w, rows, K, out);
        return hipGetLastError();
    };
    switch (wt) {
        case T_F16: return go(std::integral_constant<int, T_F16>());
        case T_Q8_0: return go(std::integral_constant<int, T_Q8_0>());
        case T_Q4_0: return go(std::integral_constant<int, T_Q4_0>());
        case T_Q4_K: return go(std::integral_constant<int, T_Q4_K>());
        case T_Q5_K: return go(std::integral_constant<int, T_Q5_K>());
        case T_Q6_K: return go(std::integral_constant<int, T_Q6_K>());
        case T_MXFP4: return go(std::integral_constant<int, T_MXFP4>());
        default: return hipErrorInvalidValue;
    }
}

hipError_t launch_dequant_f16(int wt, const void * W, int64_t rows, int64_t K, uint16_t * out, hipStream_t st) {
    return launch_dequant<false>(wt, W, rows, K, out, st);
}

hipError_t launch_f16_tiled(int wt, const void * W, int64_t rows, int64_t K, uint16_t * out, hipStream_t st) {
    return launch_dequant<true>(wt, W, rows, K, out, st);
}

hipError_t launch_convert_f16(int type, const void * src, int64_t n, uint16_t * dst, hipStream_t st) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(convert_f16_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, type, src, n, dst);
    return hipGetLastError();
}

hipError_t launch_pack_weight(int wt, const void * src, int64_t rows, int64_t K, void * dst, hipStream_t st) {
    const uint8_t * s = (const uint8_t *)src;
    uint8_t * d = (uint8_t *)dst;
    switch (wt) {
        case T_F16:
        case T_Q4_K:
        case T_Q5_K: {
            const int64_t bytes = packed_weight_bytes(wt, rows, K);
            if (s != d) return hipMemcpyAsync(d, s, (size_t)bytes, hipMemcpyDeviceToDevice, st);
            return hipSuccess;
        }
        case T_Q8_0: {
            const int64_t n = rows * (K / 32);
            if (n <= 0) return hipSuccess;
            hipLaunchKernelGGL(pack_q8_0_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, s, rows, K, d);
            return hipGetLastError();
        }
        case T_Q6_K: {
            const int64_t n = rows * (K / 256);
            if (n <= 0) return hipSuccess;
            hipLaunchKernelGGL(pack_q6_k_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, s, rows, K, d);
            return hipGetLastError();
        }
        case T_Q4_0: {
            const int64_t n = rows * (K / 32);
            if (n <= 0) return hipSuccess;
            hipLaunchKernelGGL(pack_q4_0_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, s, rows, K, d);
            return hipGetLastError();
        }
        case T_MXFP4: {
            const int64_t n = rows * (K / 32);
            if (n <= 0) return hipSuccess;
            hipLaunchKernelGGL(pack_mxfp4_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, s, rows, K, d);
            return hipGetLastError();
        }
        default: return hipErrorInvalidValue;
    }
}

}  // namespace mx
