// mh_prefill.hip — expert-major prefill of one MoE layer with CDNA4 scaled
// MFMA: forward_batch()'s route + expert-major block (engine/midge.c:591-611)
// with expert_apply (engine/midge.c:437-467) as one grouped GEMM per routed
// expert over the tokens routed to it.
//
//   lists      assignments (token t, slot i) grouped by expert: counts,
//              offsets, token of each list position, slot of each position,
//              and the passes (an expert's tokens in runs of up to 128)
//   quantize   xb (per token) -> kTerms planes of fp6 e2m3 with an e8m0
//              scale per 32-element block: x = sum_t q_t * 2^e_t, each term
//              the rounding residual of the previous one (each shrinks the
//              block's largest residual by >= 2^-4). fp4 x fp6 runs the
//              instruction at twice the rate of fp4 x fp8 (measured 8.1
//              against 4.3 PFLOP/s), and an e2m3 term reduces a block's
//              residual as much as an e4m3 one.
//   gate/up    per (pass, 128 row pairs): A = the fp4 gate and up rows
//              verbatim (e2m1 nibbles) with e8m0 scales taken exactly from
//              the f16 powers of two; B = the pass's quantized tokens;
//              V_MFMA_SCALE_F32_16X16X128_F8F6F4 accumulates all terms in
//              f32; epilogue bias + clamped SwiGLU -> h, which never leaves
//              the block: its 128 rows are a K step of the down product, and
//              the block writes them quantized
//   down       per (pass, 128 rows) over h; epilogue + bias -> y of the
//              assignment's slot; the existing prefill combine then adds
//              w * y to each token in ascending expert order.
//
// Operand layout of the 16x16x128 instruction with fp4 A and fp6 B: lane l
// holds A row l % 16 and B column l % 16; with g = l / 16, A's 16 bytes (32
// e2m1 values) and B's 24 bytes (32 e2m3 values, 6 bits each from the lowest
// bit up) are columns 32 g .. 32 g + 31 of the step, in order, and each
// lane's scale covers its own 32 columns. So for K step s (columns 128 s ..
// 128 s + 127) A lane (m, g) takes 16-byte chunk 4 s + g of row m (one MXFP4
// block and its scale) and B lane (n, g) block 4 s + g of token n with its
// scale: activations are quantized in natural 32-column blocks, like the
// weights. Output lane l: column l % 16, rows 4 (l / 16) + i for
// accumulator i.
#include <stdlib.h>

#include <algorithm>
#include <type_traits>

#include "mh_dma.cuh"
#include "mh_fp6.cuh"
#include "mh_internal.h"

namespace mh {

namespace {

constexpr int kWaves = 8;      // waves per GEMM block (two per SIMD)
constexpr int kTile = 16;      // rows and tokens of a matrix instruction
constexpr int kPassTiles = 8;  // token tiles of a pass
constexpr int kRows = kTile * kWaves;   // weight rows (of each matrix) per block
constexpr int kRG = 4;         // row tiles (of each matrix) per wave: half the block's

typedef int v8i __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------- lists

// An expert's T tokens run in passes of up to kPassTiles token tiles, as
// even as tiles allow (260 tokens as 6 + 6 + 5 tiles, not 8 + 8 + 1).
__host__ __device__ inline int pass_tiles(int T) { return (T + kTile - 1) / kTile; }
__host__ __device__ inline int pass_count(int T) { return (pass_tiles(T) + kPassTiles - 1) / kPassTiles; }
// the most passes that N assignments over E experts can make
__host__ inline int64_t pass_max(int64_t N, int64_t E) {
    return std::min<int64_t>(E, N) + N / (kTile * kPassTiles);
}

// The lists in one block (E <= kPlistMaxE): ranks by LDS atomics, an
// exclusive scan of the counts and of the passes, then the scatter.
// Positions within an expert's list follow the atomics' order; every output
// is per assignment, so the order does not change any result.
constexpr int kPlistMaxE = 4096;
constexpr int kPB = 8;
__global__ void __launch_bounds__(1024)
k_plist_one(const int32_t *sel, int N, int E, int k, int *rank, int *offs, int *list_tok, int *slot_of, int *poff,
            int *pexp) {
    __shared__ int cnt[kPlistMaxE];
    __shared__ unsigned long long wsum[16];
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    for (int i = t; i < E; i += 1024) cnt[i] = 0;
    __syncthreads();
    // (kPB assignments per thread at a time: their loads are in flight
    // together, and a list of one batch keeps its ranks in registers)
    int es[kPB], rk[kPB];
    for (int a0 = t; a0 < N; a0 += 1024 * kPB) {
#pragma unroll
        for (int u = 0; u < kPB; ++u) es[u] = a0 + 1024 * u < N ? sel[a0 + 1024 * u] : -1;
#pragma unroll
        for (int u = 0; u < kPB; ++u) {
            rk[u] = es[u] >= 0 && es[u] < E ? atomicAdd(&cnt[es[u]], 1) : -1;
            if (N > 1024 * kPB && a0 + 1024 * u < N) rank[a0 + 1024 * u] = rk[u];
        }
    }
    __syncthreads();
    // thread t owns counters [t * ch, t * ch + ch): local sums (tokens in the
    // low half, passes in the high one), block scan
    const int ch = (E + 1023) / 1024;
    unsigned long long own = 0;
    for (int i = 0; i < ch; ++i) {
        const int e = t * ch + i;
        if (e < E) own += (unsigned)cnt[e] | ((unsigned long long)pass_count(cnt[e]) << 32);
    }
    unsigned long long v = own;
    for (int o = 1; o < 64; o <<= 1) {
        const unsigned long long u = __shfl_up(v, o, 64);
        if (lane >= o) v += u;
    }
    if (lane == 63) wsum[wv] = v;
    __syncthreads();
    unsigned long long run = v - own, total = 0;
    for (int i = 0; i < 16; ++i) {
        if (i < wv) run += wsum[i];
        total += wsum[i];
    }
    for (int i = 0; i < ch; ++i) {
        const int e = t * ch + i;
        if (e < E) {
            const int c = cnt[e], np = pass_count(c), p0 = (int)(run >> 32);
            cnt[e] = (int)run;
            offs[e] = (int)run;
            poff[e] = p0;
            for (int p = 0; p < np; ++p) pexp[p0 + p] = e;
            run += (unsigned)c | ((unsigned long long)np << 32);
        }
    }
    if (t == 0) {
        offs[E] = (int)total;
        poff[E] = (int)(total >> 32);
    }
    __syncthreads();
    for (int a0 = t; a0 < N; a0 += 1024 * kPB) {
        if (N > 1024 * kPB) {
#pragma unroll
            for (int u = 0; u < kPB; ++u) {
                es[u] = a0 + 1024 * u < N ? sel[a0 + 1024 * u] : -1;
                rk[u] = a0 + 1024 * u < N ? rank[a0 + 1024 * u] : -1;
            }
        }
#pragma unroll
        for (int u = 0; u < kPB; ++u) {
            if (rk[u] < 0) continue;
            const int p = cnt[es[u]] + rk[u];
            list_tok[p] = (a0 + 1024 * u) / k;
            slot_of[p] = a0 + 1024 * u;
        }
    }
}

// ---------------------------------------------------------------- quantize

// Rows of K f32 -> records (thread = (row, block); blocks past K are zeros).
__global__ void __launch_bounds__(256)
k_quant_terms(const float *__restrict__ in, int rows, int K, uint8_t *__restrict__ q) {
    const int nst = k_steps(K), nb = 4 * nst;
    const int64_t id = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= (int64_t)rows * nb) return;
    const int r = (int)(id / nb), b = (int)(id - (int64_t)r * nb);
    float v[32];
    if (32 * b < K) {
        const float *p0 = in + (int64_t)r * K + 32 * b;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float4 a = ((const float4 *)p0)[j];
            v[4 * j + 0] = a.x; v[4 * j + 1] = a.y; v[4 * j + 2] = a.z; v[4 * j + 3] = a.w;
        }
    } else {
#pragma unroll
        for (int j = 0; j < 32; ++j) v[j] = 0.f;
    }
    quant_block(v, q + ((int64_t)r * nst + (b >> 2)) * kRec, b & 3);
}

// ---------------------------------------------------------------- GEMM

struct GemmArgs {
    const uint8_t *experts;
    uint64_t stride;
    uint64_t off[9];
    int E, H, F;
    float alpha, limit;
    int act_plain;
    const int *offs;       // [E + 1]
    const int *poff;       // [E + 1] passes before expert e
    const int *pexp;       // expert of each pass
    const int *list_tok;   // [N]
    const int *slot_of;    // [N]
    const uint8_t *bq;     // records of the B rows
    uint8_t *hq;           // records of h, list order (gate/up output)
    float *ye;             // [n * k][H] (down output, slot order)
    unsigned *err;         // set if a weight scale is not a power of two
};

// f16 power of two -> e8m0 (exact); flags anything else.
__device__ __forceinline__ int e8m0_of_f16(uint32_t h, unsigned &bad) {
    const uint32_t f = __float_as_uint(mh_f16((uint16_t)h));
    bad |= f & 0x807FFFFFu;           // sign or mantissa bits: not a positive power of two
    return (int)((f >> 23) & 0xFFu);  // a zero scale (an e8m0 below f16's range) becomes 2^-127
}

// LDS of a block. A step's weights are a ring of three, its tokens two.
//   B    [2][token tile][kRec x 16 tokens]: the tile's low pieces per term as
//        [token][4], its high pieces per term as [token][2], its scale words
//        as [token][4], and 256 unused bytes. Pieces are swizzled within a
//        token (low: block g at g ^ (token / 2) % 4, high: half h at
//        h ^ (token / 4) % 2) so that a read's lanes fall in distinct banks.
//   A    [3][matrix][row tile][row][4] 16-byte chunks, swizzled like B's low
//        pieces
//   AS   [3][row tile][matrix][row][4] f16 scales
constexpr int kLdsBT = kRec * kTile, kLdsB = kPassTiles * kLdsBT;
constexpr int kLdsAT = kTile * 64, kLdsST = 256;
constexpr int gemm_a(int nm) { return nm * kWaves * kLdsAT; }
constexpr int kLdsS = kWaves * kLdsST;
constexpr int gemm_lds(int nm) { return 2 * kLdsB + 3 * gemm_a(nm) + 3 * kLdsS; }
static_assert(gemm_lds(2) <= 160 * 1024, "LDS per workgroup on gfx950");
// gate/up's h, after the steps: floats per block of 32 rows and per token
// (the readers' 8 lanes, 2 tokens x 4 blocks, fall in distinct banks)
constexpr int kHBlk = 36, kHTok = 4 * kHBlk;
static_assert(kPassTiles * kTile * kHTok * 4 <= gemm_lds(2) && kPassTiles * kTile * 4 == 64 * kWaves && kRows == 128,
              "a block's h: one thread per token and 32 rows, one K step of the down product");
static_assert(kWaves == kPassTiles, "wave w loads row tile w and token tile w");

// This wave's loads but the last LEFT, and its LDS reads, are done; then all waves.
template <int LEFT>
__device__ __forceinline__ void step_wait() {
    dma_wait<LEFT>();
    dma_barrier();
}

// MODE 0: gate/up (K = H, rows = F, B rows = tokens through list_tok);
// MODE 1: down (K = F, rows = H, B rows = list positions).
// Block = (pass, 128 rows of each matrix). Wave (rg, tg) = (wave % 2, wave /
// 2) multiplies row tiles 4 rg .. 4 rg + 3 (of each matrix) with token tiles
// tg and tg + 4: the waves of a SIMD hold token tiles tg and tg + 2. Per K
// step of 128 columns wave w loads row tile w two steps ahead and token tile
// w one step ahead, straight into LDS; one barrier a step.
template <int MODE>
__global__ void __launch_bounds__(64 * kWaves, 2) k_moe_gemm(GemmArgs A) {
    constexpr int NM = MODE == 0 ? 2 : 1;   // weight matrices: gate and up, or down
    extern __shared__ __attribute__((aligned(16))) uint8_t glds[];
    const uint32_t lds0 = lds_offset(glds);
    const int K = MODE == 0 ? A.H : A.F;
    const int R = MODE == 0 ? A.F : A.H;
    const int groups = (R + kRows - 1) / kRows;
    // XCD-aware order: the dispatcher deals blocks to the 8 XCDs round robin
    // (block b to XCD b % 8), so equal consecutive shares of the (expert, row
    // group, pass) list per XCD keep an expert's tokens, and the weights its
    // passes share, in one L2
    const int total = A.poff[A.E] * groups, share = (total + 7) / 8;
    const int lin = (int)(blockIdx.x % 8) * share + (int)(blockIdx.x / 8);
    if ((int)(blockIdx.x / 8) >= share || lin >= total) return;   // block-uniform
    const int e = A.pexp[lin / groups];
    const int base = A.offs[e], T = A.offs[e + 1] - base;
    const int np = A.poff[e + 1] - A.poff[e];
    const int in_e = lin - A.poff[e] * groups, rgrp = in_e / np, pass = in_e - rgrp * np;
    const int tiles = pass_tiles(T);
    const int p0 = pass * tiles / np * kTile, p1 = min((pass + 1) * tiles / np * kTile, T);
    const int nt = (p1 - p0 + kTile - 1) / kTile;

    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = threadIdx.x & 63;
    const int m = l & 15, g = l >> 4;
    const uint8_t *ex = A.experts + (uint64_t)e * A.stride;
    const int nsc = K / 32, S = k_steps(K);

    // ---- this lane's sources
    const int swz = (l & 3) ^ ((l >> 3) & 3);   // block of the step that this lane's low piece or chunk holds
    const uint8_t *asrc[NM];
    {
        const size_t row = (size_t)min(rgrp * kRows + wave * kTile + (l >> 2), R - 1);
#pragma unroll
        for (int mt = 0; mt < NM; ++mt) asrc[mt] = ex + A.off[MODE == 0 ? 3 * mt : 6] + row * (size_t)(K / 2);
    }
    const uint8_t *ssrc;
    {
        const size_t row = (size_t)min(rgrp * kRows + wave * kTile + ((l & 31) >> 1), R - 1);
        ssrc = ex + (MODE == 0 ? (l < 32 ? A.off[1] : A.off[4]) : A.off[7]) + row * (size_t)(2 * nsc);
    }
    const uint8_t *bsrc[3];   // low pieces, high pieces of terms 0-1, the rest
    {
        const int tok = kTile * wave;
        auto rec = [&](int n) {
            const int p = min(p0 + tok + n, p1 - 1);
            return A.bq + (size_t)(MODE == 0 ? A.list_tok[base + p] : base + p) * ((size_t)S * kRec);
        };
        const int n1 = (l & 31) >> 1, h1 = (l & 1) ^ ((n1 >> 2) & 1);
        bsrc[0] = rec(l >> 2) + 16 * swz;
        bsrc[1] = rec(n1) + kRecHi + 32 * (l >> 5) + 16 * h1;
        bsrc[2] = l < 32 ? rec(n1) + kRecHi + 64 + 16 * h1 : rec(l & 15) + kRecSc + 16 * ((l >> 4) & 1);
    }
    static_assert(kTerms == 3, "a token tile's pieces: 5 loads of 64");
    const uint32_t ldsA = lds0 + 2 * kLdsB, ldsS = ldsA + 3 * gemm_a(NM);
    auto issue_a = [&](int st, int buf) __attribute__((always_inline)) {
        const uint32_t c = 16u * (uint32_t)min(4 * st + swz, nsc - 1);   // past K: a repeat (the tokens are zero there)
#pragma unroll
        for (int mt = 0; mt < NM; ++mt)
            dma16(ldsA + (uint32_t)buf * gemm_a(NM) + (uint32_t)(mt * kWaves + wave) * kLdsAT, asrc[mt] + c);
        dma4(ldsS + (uint32_t)buf * kLdsS + (uint32_t)wave * kLdsST, ssrc + 4u * (uint32_t)min(2 * st + (l & 1), nsc / 2 - 1));
    };
    constexpr int kALoads = NM + 1;
    const bool loads_b = wave < nt;
    auto issue_b = [&](int st, int buf) __attribute__((always_inline)) {
        if (!loads_b) return;   // wave-uniform
        const uint32_t d = lds0 + (uint32_t)buf * kLdsB + (uint32_t)wave * kLdsBT;
        const uint32_t o = (uint32_t)st * kRec;
#pragma unroll
        for (int t = 0; t < kTerms; ++t) dma16(d + 1024u * t, bsrc[0] + (o + 64u * t));
        dma16(d + 1024u * kTerms, bsrc[1] + o);
        dma16(d + 1024u * (kTerms + 1), bsrc[2] + o);
    };

    const int rg = wave & 1, tg = wave >> 1;
    const int lo_off = 64 * m + 16 * (g ^ ((m >> 1) & 3));            // this lane's chunk or low piece
    const int hi_off = 32 * m + 16 * ((g >> 1) ^ ((m >> 2) & 1)) + 8 * (g & 1);
    unsigned bad = 0;

    auto run = [&](auto ntc) __attribute__((always_inline)) {
        constexpr int TN = decltype(ntc)::value;   // this wave's token tiles
        v4f acc[NM][kRG][TN > 0 ? TN : 1];
#pragma unroll
        for (int mt = 0; mt < NM; ++mt)
#pragma unroll
            for (int r = 0; r < kRG; ++r)
#pragma unroll
                for (int j = 0; j < TN; ++j) acc[mt][r][j] = v4f{0.f, 0.f, 0.f, 0.f};
        issue_b(0, 0);
        issue_a(0, 0);
        if (S > 1) issue_a(1, 1);
        int ab = 0;   // st % 3
        for (int st = 0; st < S; ++st) {
            // step st's loads are done, and every wave is past step st - 1,
            // whose buffers the next loads overwrite
            if (st + 1 < S) step_wait<kALoads>();
            else step_wait<0>();
            if (st + 1 < S) issue_b(st + 1, (st + 1) & 1);
            const int ab2 = ab == 0 ? 2 : ab - 1;   // (st + 2) % 3
            if (st + 2 < S) issue_a(st + 2, ab2);
            if constexpr (TN > 0) {
                const uint8_t *la = glds + 2 * kLdsB + ab * gemm_a(NM) + kRG * rg * kLdsAT + lo_off;
                const uint8_t *ls = glds + 2 * kLdsB + 3 * gemm_a(NM) + ab * kLdsS + kRG * rg * kLdsST + 8 * m + 2 * g;
                const uint8_t *lb = glds + (st & 1) * kLdsB + tg * kLdsBT;
                v8i qb[TN][kTerms];
                int sb[TN];
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    const uint8_t *t0 = lb + 4 * j * kLdsBT;
                    sb[j] = *(const int *)(t0 + kTile * kRecSc + 16 * m + 4 * g);
#pragma unroll
                    for (int t = 0; t < kTerms; ++t) {
                        const mh_u4 lo = *(const mh_u4 *)(t0 + 1024 * t + lo_off);
                        const uint2 hi = *(const uint2 *)(t0 + 1024 * kTerms + 512 * t + hi_off);
                        qb[j][t] = v8i{(int)lo.x, (int)lo.y, (int)lo.z, (int)lo.w, (int)hi.x, (int)hi.y, 0, 0};
                    }
                }
#pragma unroll
                for (int r = 0; r < kRG; ++r) {
#pragma unroll
                    for (int mt = 0; mt < NM; ++mt) {
                        const mh_u4 a = *(const mh_u4 *)(la + (mt * kWaves + r) * kLdsAT);
                        const int sa = e8m0_of_f16(*(const uint16_t *)(ls + r * kLdsST + 128 * mt), bad);
                        const v8i qa = v8i{(int)a.x, (int)a.y, (int)a.z, (int)a.w, 0, 0, 0, 0};
#pragma unroll
                        for (int j = 0; j < TN; ++j) {
                            v4f c = acc[mt][r][j];
                            c = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(qa, qb[j][0], c, 4, 2, 0, sa, 0, sb[j]);
                            c = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(qa, qb[j][1], c, 4, 2, 0, sa, 1, sb[j]);
                            c = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(qa, qb[j][2], c, 4, 2, 0, sa, 2, sb[j]);
                            acc[mt][r][j] = c;
                        }
                    }
                }
            }
            ab = ab == 2 ? 0 : ab + 1;
        }
        // lane (m, g) holds rows 4 g .. 4 g + 3 of each row tile for token m
        // of its token tiles
        const int row0 = rgrp * kRows + kRG * rg * kTile + 4 * g;
        float4 bias[NM][kRG];
#pragma unroll
        for (int r = 0; r < kRG; ++r) {
            const size_t ro = (size_t)min(row0 + kTile * r, R - 4) * 4;
            bias[0][r] = *(const float4 *)(ex + A.off[MODE == 0 ? 2 : 8] + ro);
            if constexpr (MODE == 0) bias[NM - 1][r] = *(const float4 *)(ex + A.off[5] + ro);
        }
        if constexpr (MODE == 0) {
            // h through LDS, [token][block of 32 rows][32 + 4], then thread
            // (token, block) quantizes; rows past F are zeros
            step_wait<0>();   // every wave is past the last step
            float *lh = (float *)glds;
#pragma unroll
            for (int j = 0; j < TN; ++j) {
#pragma unroll
                for (int r = 0; r < kRG; ++r) {
                    const int rr = (kRG * rg + r) * kTile + 4 * g;
                    const float gb[4] = {bias[0][r].x, bias[0][r].y, bias[0][r].z, bias[0][r].w};
                    const float ub[4] = {bias[NM - 1][r].x, bias[NM - 1][r].y, bias[NM - 1][r].z, bias[NM - 1][r].w};
                    float o[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        float gg = acc[0][r][j][i] + gb[i];
                        float uu = acc[NM - 1][r][j][i] + ub[i];
                        if (A.act_plain) {
                            o[i] = gg / (1.0f + expf(-gg)) * uu;
                        } else {
                            if (gg > A.limit) gg = A.limit;
                            if (uu > A.limit) uu = A.limit;
                            if (uu < -A.limit) uu = -A.limit;
                            o[i] = gg / (1.0f + expf(-A.alpha * gg)) * (uu + 1.0f);
                        }
                        if (row0 + kTile * r >= R) o[i] = 0.f;   // wave-uniform: R is a multiple of the tile
                    }
                    *(float4 *)(lh + (kTile * (tg + 4 * j) + m) * kHTok + (rr >> 5) * kHBlk + (rr & 31)) =
                        float4{o[0], o[1], o[2], o[3]};
                }
            }
        } else {
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const int p = p0 + kTile * (tg + 4 * j) + m;
                if (p >= p1) continue;
                float *out = A.ye + (size_t)A.slot_of[base + p] * A.H + row0;
#pragma unroll
                for (int r = 0; r < kRG; ++r) {
                    const v4f c = acc[0][r][j];
                    const float4 b = bias[0][r];
                    if (row0 + kTile * r < R)   // wave-uniform
                        *(float4 *)(out + kTile * r) = float4{c[0] + b.x, c[1] + b.y, c[2] + b.z, c[3] + b.w};
                }
            }
        }
    };
    const int tn = nt > tg ? (nt > tg + 4 ? 2 : 1) : 0;   // wave-uniform
    switch (tn) {
    case 0: run(std::integral_constant<int, 0>{}); break;
    case 1: run(std::integral_constant<int, 1>{}); break;
    default: run(std::integral_constant<int, 2>{}); break;
    }
    if constexpr (MODE == 0) {
        __syncthreads();
        const int tok = threadIdx.x >> 2, blk = threadIdx.x & 3;
        if (p0 + tok < p1) {
            const float *src = (const float *)glds + tok * kHTok + blk * kHBlk;
            float v[32];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const float4 a = *(const float4 *)(src + 4 * j);
                v[4 * j + 0] = a.x; v[4 * j + 1] = a.y; v[4 * j + 2] = a.z; v[4 * j + 3] = a.w;
            }
            quant_block(v, A.hq + ((size_t)(base + p0 + tok) * groups + rgrp) * kRec, blk);
        }
    }
    if (bad) atomicOr(A.err, 1u);
}

}  // namespace

// Assignments grouped by expert (offsets[E + 1], token and slot of each list
// position) and their passes in the S_LIST scratch; E <= 4096.
int launch_expert_lists(const int32_t *sel, int N, int E, int k, ExpertLists *out, hipStream_t s) {
    if (E > kPlistMaxE) return fail(MH_E_UNSUPPORTED, "expert lists: %d experts > %d", E, kPlistMaxE);
    void *pl;
    MH_TRY(scratch(S_LIST, sizeof(int) * (2 * ((size_t)E + 1) + 3 * (size_t)N + (size_t)pass_max(N, E)), &pl));
    int *offs = (int *)pl, *rank = offs + E + 1;
    out->offs = offs;
    out->list_tok = rank + N;
    out->slot_of = rank + 2 * (size_t)N;
    out->poff = rank + 3 * (size_t)N;
    out->pexp = out->poff + E + 1;
    MH_LAUNCH("plist", k_plist_one, dim3(1), dim3(1024), 0, s, sel, N, E, k, rank, offs, out->list_tok, out->slot_of,
              out->poff, out->pexp);
    return hip_check(hipGetLastError(), "expert lists launch");
}

// The widest layers that the scaled-MFMA path takes (wider ones keep the
// per-assignment GEMVs' f32 arithmetic).
constexpr int64_t kMfmaMaxH = 3328, kMfmaMaxF = 4608;

// True when the scaled-MFMA path handles this layer (MXFP4 experts in 16-byte
// chunks, shapes that tile by 64 along K and 32 along rows).
bool prefill_mfma_ok(const DevLayer &L) {
    if (sw(SW_NO_MFMA)) return false;
    return L.expert_dt == MH_DT_MXFP4 && L.hidden % 64 == 0 && L.ffn % 64 == 0 && L.top_k >= 1 &&
           L.n_experts <= kPlistMaxE && L.hidden <= kMfmaMaxH && L.ffn <= kMfmaMaxF && (uintptr_t)L.experts % 16 == 0;
}

// The records of n tokens' x, then of their h (S_Q scratch).
int prefill_records(const DevLayer &L, int n, uint8_t **x, uint8_t **h) {
    const size_t qx = (size_t)kRec * n * k_steps((int)L.hidden);
    void *p;
    MH_TRY(scratch(S_Q, qx + (size_t)kRec * n * L.top_k * k_steps((int)L.ffn), &p));
    *x = (uint8_t *)p;
    *h = *x + qx;
    return MH_OK;
}

// Expert-major MoE of n tokens: x[t] += sum over t's slots, in ascending
// expert order, of w * expert(xb[t]); ye is [n * k][H] scratch read by the
// prefill combine (launched by the caller), written for routed slots only.
// xb null: the router has written the records of x (prefill_records).
int run_expert_major_mfma(const DevLayer &L, int n, const float *xb, const int32_t *sel, float *ye,
                          hipStream_t s) {
    const int k = L.top_k, E = L.n_experts, N = n * k;
    const int H = (int)L.hidden, F = (int)L.ffn;
    if (!prefill_mfma_ok(L)) return fail(MH_E_UNSUPPORTED, "prefill: layer shape not handled by the MFMA path");
    static uint64_t lds_epoch = 0;   // the initialisation the LDS attribute was set under
    if (lds_epoch != init_epoch()) {
        MH_HIP(hipFuncSetAttribute((const void *)k_moe_gemm<0>, hipFuncAttributeMaxDynamicSharedMemorySize, gemm_lds(2)));
        MH_HIP(hipFuncSetAttribute((const void *)k_moe_gemm<1>, hipFuncAttributeMaxDynamicSharedMemorySize, gemm_lds(1)));
        lds_epoch = init_epoch();
    }
    unsigned *scale_err_dev = nullptr;
    MH_TRY(async_flag(F_PREFILL_SCALE, "prefill: an MXFP4 scale is not a positive power of two (e8m0 cannot hold it)",
                      &scale_err_dev));
    ExpertLists lists;
    MH_TRY(launch_expert_lists(sel, N, E, k, &lists, s));
    uint8_t *qx, *qh;
    MH_TRY(prefill_records(L, n, &qx, &qh));

    // ye rows of unroutable slots are not written: the combine skips them

    GemmArgs A;
    A.experts = L.experts;
    A.stride = L.expert_stride;
    for (int i = 0; i < 9; i++) A.off[i] = L.off[i];
    A.E = E;
    A.H = H;
    A.F = F;
    A.alpha = L.alpha;
    A.limit = L.limit;
    A.act_plain = L.act_plain;
    A.offs = lists.offs;
    A.poff = lists.poff;
    A.pexp = lists.pexp;
    A.list_tok = lists.list_tok;
    A.slot_of = lists.slot_of;
    A.bq = qx;
    A.hq = qh;
    A.ye = ye;
    A.err = scale_err_dev;

    // a block for every pass that the assignments can make (those without one return)
    auto grid = [&](int R) {
        const int64_t nb = pass_max(N, E) * ((R + kRows - 1) / kRows);
        return dim3((unsigned)((nb + 7) / 8 * 8));
    };
    if (xb) {
        const int64_t thr = (int64_t)n * 4 * k_steps(H);
        MH_LAUNCH("quant_x", k_quant_terms, dim3((unsigned)((thr + 255) / 256)), dim3(256), 0, s, xb, n, H, qx);
    }
    // gate/up over the quantized tokens, then down over the quantized h
    MH_LAUNCH("moe_gu_mfma", k_moe_gemm<0>, grid(F), dim3(64 * kWaves), gemm_lds(2), s, A);
    A.bq = qh;
    MH_LAUNCH("moe_down_mfma", k_moe_gemm<1>, grid(H), dim3(64 * kWaves), gemm_lds(1), s, A);
    return hip_check(hipGetLastError(), "prefill MFMA launches");
}

}  // namespace mh
