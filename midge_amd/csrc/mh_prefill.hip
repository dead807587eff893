// mh_prefill.hip — expert-major prefill of one MoE layer with CDNA4 scaled
// MFMA: forward_batch()'s route + expert-major block (engine/midge.c:591-611)
// with expert_apply (engine/midge.c:437-467) as one grouped GEMM per routed
// expert over the tokens routed to it.
//
//   lists      assignments (token t, slot i) grouped by expert: counts,
//              offsets, token of each list position, slot of each position,
//              and the passes (an expert's tokens in runs of up to 64)
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
//              V_MFMA_SCALE_F32_32X32X64_F8F6F4 accumulates all terms in
//              f32; epilogue bias + clamped SwiGLU -> h, which never leaves
//              the block: its 128 rows are a K step of the down product, and
//              the block writes them quantized
//   down       per (pass, 128 rows) over h; epilogue + bias -> y of the
//              assignment's slot; the existing prefill combine then adds
//              w * y to each token in ascending expert order.
//
// Operand layout of the 32x32x64 instruction with fp4 A and fp6 B
// (measured on gfx950 with one-hot operands): lane l holds A row l % 32 and
// B column l % 32; with g = l / 32, A's 16 bytes (32 e2m1 values) and B's 24
// bytes (32 e2m3 values, 6 bits each from the lowest bit up) are columns
// 32 g .. 32 g + 31 of the instruction, in order, and each lane's scale covers
// its own 32 columns. So for half h of K step s (columns 128 s + 64 h ..) A
// lane (m, g) takes 16-byte chunk 4 s + 2 h + g of row m (one MXFP4 block and
// its scale) and B lane (n, g) the same block of token n with its scale:
// activations are quantized in natural 32-column blocks, like the weights.
// Output lane l: column l % 32, rows 8 (i / 4) + 4 g + i % 4 for accumulator
// i. (The 16x16x128 instruction takes tiles of 16 tokens but runs these
// operands at half the rate: 4.5 against 9.2 PFLOP/s back to back.)
#include <stdlib.h>

#include <algorithm>
#include <type_traits>

#include "mh_dma.cuh"
#include "mh_fp6.cuh"
#include "mh_internal.h"
#include "mh_mfma16.cuh"

namespace mh {

namespace {

constexpr int kWaves = 4;      // waves per GEMM block (two blocks per CU)
constexpr int kTile = 32;      // rows and tokens of a matrix instruction
constexpr int kPassTiles = 2;  // token tiles of a pass
constexpr int kLoad = 16;      // rows or tokens of a load instruction
constexpr int kRows = 128;     // weight rows (of each matrix) per block
constexpr int kRG = 2;         // row tiles (of each matrix) per wave: half the block's

typedef int v8i __attribute__((ext_vector_type(8)));

// ---------------------------------------------------------------- lists

// An expert's T tokens run in passes of up to kPassTiles token tiles, as
// even as tiles allow.
__host__ __device__ inline int pass_tiles(int T) { return (T + kTile - 1) / kTile; }
__host__ __device__ inline int pass_count(int T) { return (pass_tiles(T) + kPassTiles - 1) / kPassTiles; }
// the most passes that N assignments over E experts can make
__host__ inline int64_t pass_max(int64_t N, int64_t E) {
    return std::min<int64_t>(E, N) + N / (kTile * kPassTiles);
}

// A pass's expert, and what its block needs to find the pass among the
// expert's: the start and length of the expert's list, the passes before it.
struct Pass {
    int e, off, T, before;
};

// The lists in one block (E <= kPlistMaxE): ranks by LDS atomics, an
// exclusive scan of the counts and of the passes, then the scatter.
// Positions within an expert's list follow the atomics' order; every output
// is per assignment, so the order does not change any result.
constexpr int kPlistMaxE = 4096;
constexpr int kPB = 8;
__global__ void __launch_bounds__(1024)
k_plist_one(const int32_t *sel, int N, int E, int k, int *rank, int *list_tok, int *slot_of, Pass *passes, int *npass) {
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
            for (int p = 0; p < np; ++p) passes[p0 + p] = Pass{e, (int)run, c, p0};
            run += (unsigned)c | ((unsigned long long)np << 32);
        }
    }
    if (t == 0) *npass = (int)(total >> 32);
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
    const Pass *passes;
    const int *npass;
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

// LDS of a block: two steps of weights and tokens, four steps of scales.
//   B    [2][token] records as in memory: 19 16-byte pieces, an odd number, so
//        that a read's lanes (one piece of 16 tokens) fall in distinct banks
//   A    [2][matrix][16 rows][row][4] 16-byte chunks, chunk c of a row at
//        c ^ (row / 4) % 4 for the same reason
//   AS   [matrix][row][16] f16 scales
//   I    [32 rows][matrix][row] biases (two of each where there is one matrix)
constexpr int kLdsBT = kRec * kLoad, kLdsB = kPassTiles * 2 * kLdsBT;
constexpr int kLdsAT = kLoad * 64;
constexpr int gemm_a(int nm) { return nm * (kRows / kLoad) * kLdsAT; }
constexpr int gemm_s(int nm) { return nm * kRows * 32; }
constexpr int gemm_lds(int nm) { return 2 * (kLdsB + gemm_a(nm)) + gemm_s(nm) + kWaves * 256; }
static_assert(2 * gemm_lds(2) <= 160 * 1024 && 2 * gemm_lds(1) <= 160 * 1024, "two blocks per CU");
static_assert(kWaves * kLoad == kPassTiles * kTile && kWaves * 32 == kRows, "wave w loads 32 rows and 16 tokens");
static_assert(kRows == 128, "a block's rows of h are one K step of the down product");

// MODE 0: gate/up (K = H, rows = F, B rows = tokens through list_tok);
// MODE 1: down (K = F, rows = H, B rows = list positions).
// Block = (pass, 128 rows of each matrix), two blocks per CU, so that one
// block's start, end and waits run under the other's products. Wave (rg, tg)
// = (wave % 2, wave / 2) multiplies row tiles 2 rg, 2 rg + 1 (of each matrix)
// with token tile tg. Per K step of 128 columns wave w loads rows 32 w ..
// 32 w + 31 and 16 tokens straight into LDS. A step has two barriers: after
// the first the step is in LDS and the waves read their operands, after the
// second all of it is in registers and its buffers take the step after the
// next, so that two buffers keep up to two steps in flight under the
// products (weights alone, with one step in flight, took 118 of 194 us).
// (gpt-oss-20b layer at 512 and 2000 tokens, gate/up + down us: operands
// through registers, one wave per SIMD 190 + 140 at 512; 8 waves per block,
// one block per CU, 16x16x128 tiles and a step's scales per load 151 + 117 and
// 375 + 293; this 156-170 + 91-96 and 362-383 + 212-222. Without products
// 134 + 80 and 290 + 186, without loads 105 + 61 and 273 + 150: the load path
// and the steps' LDS reads and barriers bound it, the matrix instructions
// alone are 93 us of the 2000-token gate/up. Slower: one persistent block
// per CU with the steps running across units (157 + 90 and 427 + 263), the
// same with half the waves a phase behind (167 + 112 and 412 + 288).)
// WORDS: weights in 4-byte loads, for tables off a 16-byte boundary (2000 tokens
// of a 32-expert 2880-wide layer 625 us; 614 in 16-byte loads).
template <int MODE, bool WORDS>
__global__ void __launch_bounds__(64 * kWaves, 2) k_moe_gemm(GemmArgs A) {
    constexpr int NM = MODE == 0 ? 2 : 1;   // weight matrices: gate and up, or down
    extern __shared__ __attribute__((aligned(16))) uint8_t glds[];
    const uint32_t lds0 = lds_offset(glds);
    const int K = MODE == 0 ? A.H : A.F;
    const int R = MODE == 0 ? A.F : A.H;
    const int groups = MODE == 0 ? k_steps(R) : (R + kRows - 1) / kRows;   // (h in whole K steps of down)
    const int nsc = K / 32, S = k_steps(K);
    // XCD-aware order: the dispatcher deals blocks to the 8 XCDs round robin
    // (block b to XCD b % 8), so equal consecutive shares of the (expert, row
    // group, pass) list per XCD keep an expert's tokens, and the weights its
    // passes share, in one L2
    const int total = *A.npass * groups, share = (total + 7) / 8;
    const int lin = (int)(blockIdx.x % 8) * share + (int)(blockIdx.x / 8);
    if ((int)(blockIdx.x / 8) >= share || lin >= total) return;   // block-uniform
    const Pass ps = A.passes[lin / groups];
    const int np = pass_count(ps.T), tiles = pass_tiles(ps.T);
    const int in_e = lin - ps.before * groups, rgrp = in_e / np, pass = in_e - rgrp * np;
    const int p0 = pass * tiles / np * kTile;
    const int base = ps.off + p0, cnt = min((pass + 1) * tiles / np * kTile, ps.T) - p0;   // the pass's list positions

    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = threadIdx.x & 63;
    const int m = l & 31, g = l >> 5, m16 = m & 15;
    const int rg = wave & 1, tg = wave >> 1;
    const uint8_t *ex = A.experts + (uint64_t)ps.e * A.stride;

    // ---- loads: 32-bit lane offsets from scalar bases
    const uint32_t ldsA = lds0 + 2 * kLdsB, ldsS = ldsA + 2 * gemm_a(NM), ldsI = ldsS + gemm_s(NM);
    const int swz = (l & 3) ^ ((l >> 4) & 3);   // block of the step that this lane's low piece or chunk holds
    const int row0 = rgrp * kRows + wave * 32;
    uint32_t aoff[NM][2], soff[NM];
#pragma unroll
    for (int mt = 0; mt < NM; ++mt) {
#pragma unroll
        for (int q = 0; q < 2; ++q)   // (R is a multiple of 32: a wave's rows are all there or none)
            aoff[mt][q] = (uint32_t)A.off[MODE == 0 ? 3 * mt : 6] +
                          (uint32_t)(min(row0, R - 32) + kLoad * q + (WORDS ? l >> 4 : l >> 2)) * (uint32_t)(K / 2) +
                          (WORDS ? 4u * (l & 3) : 16u * swz);
        soff[mt] = (uint32_t)A.off[MODE == 0 ? 1 + 3 * mt : 7] + 4u * (l & 7);
    }
    constexpr int kALoads = (WORDS ? 8 : 2) * NM, kBLoads = 5;
    auto issue_a = [&](int st, int buf) __attribute__((always_inline)) {
        // (past K: what follows the row, in the expert's blob; the tokens are zero there)
#pragma unroll
        for (int mt = 0; mt < NM; ++mt)
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const uint32_t d = ldsA + (uint32_t)(buf * gemm_a(NM) + (mt * (kRows / kLoad) + 2 * wave + q) * kLdsAT);
                if constexpr (WORDS) {
#pragma unroll
                    for (uint32_t j = 0; j < 4; ++j)   // 4 rows' 64 bytes
                        dma4(d + 256u * j, ex + 64 * st, aoff[mt][q] + 2u * j * (uint32_t)K + 16u * (((l >> 2) & 3) ^ j));
                } else {
                    dma16(d, ex + 64 * st, aoff[mt][q]);
                }
            }
    };
    // the scales of 4 steps (32 bytes of a row; 8 rows per load instruction:
    // one step's 8 bytes at a time took as many cache requests as the weights)
    auto issue_s = [&](int st) __attribute__((always_inline)) {
        int lr = l >> 3;
        asm volatile("" : "+v"(lr));   // opaque: else eight rows' offsets stay in registers
#pragma unroll
        for (int mt = 0; mt < NM; ++mt)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                dma4(ldsS + (uint32_t)((mt * kRows + wave * 32 + 8 * q) * 32), ex + 8 * st,
                     soff[mt] + (uint32_t)min(row0 + 8 * q + lr, R - 1) * (uint32_t)(2 * nsc));
    };
    const bool loads_b = wave * kLoad < cnt;
    uint32_t boff[kBLoads];   // pieces l, l + 64, .. of the wave's 16 records
    const uint8_t *bbase = MODE == 0 ? A.bq : A.bq + (size_t)base * ((size_t)S * kRec);
    constexpr int kPieces = kRec / 16;
    static_assert(kLoad * kPieces == 64 * kBLoads - 16, "16 tokens' records: 4 loads of 64 pieces and one of 48");
    auto issue_b = [&](int st, int buf) __attribute__((always_inline)) {
        if (!loads_b) return;   // wave-uniform
        const uint32_t d = lds0 + (uint32_t)(buf * kLdsB + wave * kLdsBT);
        const uint8_t *b = bbase + kRec * st;
#pragma unroll
        for (int j = 0; j < kBLoads; ++j)
            if (j + 1 < kBLoads || l < 48) dma16(d + 1024u * j, b, boff[j]);
    };

    // ---- math: lane (m, g) of the operands and of the outputs' token m
    int a_off[2];   // this lane's chunk of half h
#pragma unroll
    for (int h = 0; h < 2; ++h) a_off[h] = 64 * m16 + 16 * ((2 * h + g) ^ ((m16 >> 2) & 3));
    unsigned bad = 0;
    v16f acc[NM][kRG];
#pragma unroll
    for (int mt = 0; mt < NM; ++mt)
#pragma unroll
        for (int r = 0; r < kRG; ++r) acc[mt][r] = v16f{};
    struct Operands {   // a step's: weights, the tokens' low and high pieces and scales
        mh_u4 a[2][NM][kRG], b[2][kTerms];
        uint2 h[2][kTerms];
        int sb[2];
    };
    const uint8_t *la0 = glds + 2 * kLdsB + (2 * kRG * rg + (m >> 4)) * kLdsAT;
    const uint8_t *lb0 = glds + (kTile * tg + m) * kRec;
    auto read = [&](int buf, Operands &o) __attribute__((always_inline)) {
        const uint8_t *la = la0 + buf * gemm_a(NM), *lb = lb0 + buf * kLdsB;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            o.sb[h] = *(const int *)(lb + kRecSc + 8 * h + 4 * g);
#pragma unroll
            for (int t = 0; t < kTerms; ++t) {
                o.b[h][t] = *(const mh_u4 *)(lb + 64 * t + 32 * h + 16 * g);
                o.h[h][t] = *(const uint2 *)(lb + kRecHi + 32 * t + 16 * h + 8 * g);
            }
#pragma unroll
            for (int r = 0; r < kRG; ++r)
#pragma unroll
                for (int mt = 0; mt < NM; ++mt)
                    o.a[h][mt][r] = *(const mh_u4 *)(la + (mt * (kRows / kLoad) + 2 * r) * kLdsAT + a_off[h]);
        }
    };
    // The e8m0 scales of this lane's rows for 4 steps: byte 2 (s % 2) + h of
    // word s / 2 is block 4 s + 2 h + g's (2^0 past K); two steps later word 1
    // moves to word 0.
    uint32_t sw4[NM][kRG][2];
    auto scales = [&](int st) __attribute__((always_inline)) {
        const uint8_t *ls = glds + 2 * (kLdsB + gemm_a(NM)) + (kRG * rg * kTile + m) * 32;
#pragma unroll
        for (int r = 0; r < kRG; ++r)
#pragma unroll
            for (int mt = 0; mt < NM; ++mt) {
                const uint8_t *p = ls + (mt * kRows + r * kTile) * 32;
                const mh_u4 v[2] = {*(const mh_u4 *)p, *(const mh_u4 *)(p + 16)};
#pragma unroll
                for (int w = 0; w < 2; ++w) {
                    uint32_t x = 0u;
#pragma unroll
                    for (int i = 0; i < 4; ++i) {   // blocks 8 w + 2 i + g
                        const uint32_t d = dword_of(v[w], i);
                        const bool in = 4 * st + 8 * w + 2 * i < nsc;   // uniform
                        unsigned b1 = 0u;
                        const uint32_t e = (uint32_t)e8m0_of_f16(g ? d >> 16 : d & 0xFFFFu, b1);
                        bad |= in ? b1 : 0u;
                        x |= (in ? e : 127u) << (8 * i);
                    }
                    sw4[mt][r][w] = x;
                }
                __builtin_amdgcn_sched_barrier(0);   // (one row tile's at a time: registers)
            }
    };
    auto math = [&](auto bufc, const Operands &o) __attribute__((always_inline)) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            v8i qa[NM][kRG], qb[kTerms];
#pragma unroll
            for (int r = 0; r < kRG; ++r)
#pragma unroll
                for (int mt = 0; mt < NM; ++mt) {
                    const mh_u4 a = o.a[h][mt][r];
                    qa[mt][r] = v8i{(int)a.x, (int)a.y, (int)a.z, (int)a.w, 0, 0, 0, 0};
                }
#pragma unroll
            for (int t = 0; t < kTerms; ++t)
                qb[t] = v8i{(int)o.b[h][t].x, (int)o.b[h][t].y, (int)o.b[h][t].z, (int)o.b[h][t].w,
                            (int)o.h[h][t].x, (int)o.h[h][t].y, 0, 0};
            // (term by term: consecutive instructions add into different tiles)
            auto term = [&](auto hc, auto tc) __attribute__((always_inline)) {
                constexpr int t = decltype(tc)::value, byte = 2 * decltype(bufc)::value + decltype(hc)::value;
#pragma unroll
                for (int r = 0; r < kRG; ++r)
#pragma unroll
                    for (int mt = 0; mt < NM; ++mt)
                        acc[mt][r] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(
                            qa[mt][r], qb[t], acc[mt][r], 4, 2, byte, (int)sw4[mt][r][0], t, o.sb[h]);
            };
            auto terms = [&](auto hc) __attribute__((always_inline)) {
                term(hc, std::integral_constant<int, 0>{});
                term(hc, std::integral_constant<int, 1>{});
                term(hc, std::integral_constant<int, 2>{});
            };
            if (h == 0) terms(std::integral_constant<int, 0>{});
            else terms(std::integral_constant<int, 1>{});
        }
    };
    const bool mine = kTile * tg < cnt;   // this wave has tokens
    issue_s(0);
    issue_a(0, 0);
    {   // the biases of this wave's rows; tokens from the list
        const int bm = NM == 2 ? g : 0;
        dma4(ldsI + 256u * wave, ex + A.off[MODE == 0 ? 2 + 3 * bm : 8] + (size_t)min(row0 + m, R - 1) * 4);
        auto row = [&](int n) {
            const int p = min(wave * kLoad + n, cnt - 1);
            return (uint32_t)(MODE == 0 ? A.list_tok[base + p] : p) * (uint32_t)(S * kRec);
        };
#pragma unroll
        for (int j = 0; j < kBLoads; ++j) {
            const int i = min(64 * j + l, kLoad * kPieces - 1), n = i / kPieces;
            boff[j] = row(n) + 16u * (i - n * kPieces);
        }
    }
    issue_b(0, 0);
    issue_a(1, 1);   // (S >= 2)
    issue_b(1, 1);
    const int p = kTile * tg + m;   // this lane's token
    int slot = 0;
    if constexpr (MODE == 1) slot = A.slot_of[base + min(p, cnt - 1)];
    auto step = [&](auto bufc, int st) __attribute__((always_inline)) {
        constexpr int buf = decltype(bufc)::value;
        __builtin_amdgcn_sched_barrier(0);   // (products moved into the next step would hold two steps' operands)
        // step st is in LDS (the next one's loads stay in flight)
        if (st + 1 == S) dma_wait<0>();
        else if (loads_b) dma_wait<kALoads + kBLoads>();
        else dma_wait<kALoads>();
        dma_barrier();
        Operands ops;
        if (mine) {
            if (buf == 0) {
                if (st % 4 == 0) {
                    scales(st);
                } else {
#pragma unroll
                    for (int mt = 0; mt < NM; ++mt)
#pragma unroll
                        for (int r = 0; r < kRG; ++r) sw4[mt][r][0] = sw4[mt][r][1];
                }
            }
            read(buf, ops);
        }
        // every wave holds the step in registers: its buffers take step st + 2
        dma_barrier();
        if (buf == 0 && st % 4 == 0 && st + 4 < S) issue_s(st + 4);
        if (st + 2 < S) {
            issue_a(st + 2, buf);
            issue_b(st + 2, buf);
        }
        if (mine) math(bufc, ops);
    };
    for (int st = 0; st < S; st += 2) {
        step(std::integral_constant<int, 0>{}, st);
        if (st + 1 < S) step(std::integral_constant<int, 1>{}, st + 1);
    }
    __builtin_amdgcn_sched_barrier(0);
    if (bad) atomicOr(A.err, 1u);
    if (!mine) return;
    // Outputs: the lane holds rows 8 (i / 4) + 4 g + i % 4 of each row tile
    // for its token.
    auto bias = [&](int mt, int r, int q) {   // rows 8 q + 4 g .. of row tile r
        const int rt = kRG * rg + r;
        return *(const float4 *)(glds + 2 * (kLdsB + gemm_a(NM)) + gemm_s(NM) + 256 * rt + 128 * mt +
                                 32 * q + 16 * g);
    };
    const int rt0 = rgrp * kRows + kRG * rg * kTile;   // the wave's first row
    if constexpr (MODE == 0) {
        // A row tile is a 32-block of h, half of it in each of a token's two
        // lanes: lane g gets both halves of tile g and quantizes it. Rows past
        // F are zeros.
        const bool plain = A.act_plain != 0;   // g / (1 + e^-g) u: no limits, alpha 1, nothing added to u
        const float limit = plain ? INFINITY : A.limit, alpha = plain ? 1.0f : A.alpha, one = plain ? 0.0f : 1.0f;
        float hv[kRG][16];
#pragma unroll
        for (int r = 0; r < kRG; ++r)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float4 b0 = bias(0, r, q), b1 = bias(1, r, q);
                const float gb[4] = {b0.x, b0.y, b0.z, b0.w}, ub[4] = {b1.x, b1.y, b1.z, b1.w};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    float gg = acc[0][r][4 * q + e] + gb[e];
                    float uu = acc[NM - 1][r][4 * q + e] + ub[e];
                    if (gg > limit) gg = limit;
                    if (uu > limit) uu = limit;
                    if (uu < -limit) uu = -limit;
                    const float o = gg / (1.0f + expf(-alpha * gg)) * (uu + one);
                    hv[r][4 * q + e] = rt0 + kTile * r < R ? o : 0.f;
                }
                __builtin_amdgcn_sched_barrier(0);   // (four at a time: registers)
            }
        static_assert(kRG == 2, "one row tile per lane of a token");
        typedef unsigned v2u __attribute__((ext_vector_type(2)));
        float v[32];
#pragma unroll
        for (int e = 0; e < 16; ++e) {   // tile 0's upper half of the lanes with tile 1's lower one
            const v2u x = __builtin_amdgcn_permlane32_swap(__float_as_uint(hv[0][e]), __float_as_uint(hv[1][e]), false, false);
            v[8 * (e >> 2) + (e & 3)] = __uint_as_float(x.x);
            v[8 * (e >> 2) + 4 + (e & 3)] = __uint_as_float(x.y);
        }
        if (p < cnt) quant_block(v, A.hq + ((size_t)(base + p) * groups + rgrp) * kRec, kRG * rg + g);
    } else {
        if (p >= cnt) return;
        float *out = A.ye + (size_t)slot * A.H + rt0 + 4 * g;
#pragma unroll
        for (int r = 0; r < kRG; ++r) {
            if (rt0 + kTile * r >= R) break;   // wave-uniform: R is a multiple of the tile
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float4 b = bias(0, r, q);
                *(float4 *)(out + kTile * r + 8 * q) = float4{acc[0][r][4 * q] + b.x, acc[0][r][4 * q + 1] + b.y,
                                                              acc[0][r][4 * q + 2] + b.z, acc[0][r][4 * q + 3] + b.w};
            }
        }
    }
}

}  // namespace

// Assignments grouped by expert (token and slot of each list position) and
// their passes in the S_LIST scratch; E <= 4096.
int launch_expert_lists(const int32_t *sel, int N, int E, int k, ExpertLists *out, hipStream_t s) {
    if (E > kPlistMaxE) return fail(MH_E_UNSUPPORTED, "expert lists: %d experts > %d", E, kPlistMaxE);
    void *pl;
    const size_t np = (size_t)pass_max(N, E);
    MH_TRY(scratch(S_LIST, sizeof(Pass) * np + sizeof(int) * (1 + 3 * (size_t)N), &pl));
    Pass *passes = (Pass *)pl;
    int *npass = (int *)(passes + np), *rank = npass + 1;
    out->passes = passes;
    out->npass = npass;
    out->list_tok = rank + N;
    out->slot_of = rank + 2 * (size_t)N;
    MH_LAUNCH("plist", k_plist_one, dim3(1), dim3(1024), 0, s, sel, N, E, k, rank, out->list_tok, out->slot_of, passes,
              npass);
    return hip_check(hipGetLastError(), "expert lists launch");
}

// The widest layers that the scaled-MFMA path takes. The kernel itself has no
// need of a bound; layers past it have always had the per-assignment GEMVs' f32
// arithmetic, and keep it (the fp6 terms hold an activation to 2^-12 of its
// block's largest).
constexpr int64_t kMfmaMaxH = 3328, kMfmaMaxF = 4608;

// True when the scaled-MFMA path handles this layer (MXFP4 experts on a 4-byte
// boundary, shapes that tile by 64 along K and 32 along rows).
bool prefill_mfma_ok(const DevLayer &L) {
    if (sw(SW_NO_MFMA)) return false;
    return L.expert_dt == MH_DT_MXFP4 && L.hidden % 64 == 0 && L.ffn % 64 == 0 && L.top_k >= 1 &&
           L.n_experts <= kPlistMaxE && L.hidden <= kMfmaMaxH && L.ffn <= kMfmaMaxF && (uintptr_t)L.experts % 4 == 0;
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
        for (const void *f : {(const void *)k_moe_gemm<0, false>, (const void *)k_moe_gemm<0, true>})
            MH_HIP(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, gemm_lds(2)));
        for (const void *f : {(const void *)k_moe_gemm<1, false>, (const void *)k_moe_gemm<1, true>})
            MH_HIP(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, gemm_lds(1)));
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
    A.passes = (const Pass *)lists.passes;
    A.npass = lists.npass;
    A.list_tok = lists.list_tok;
    A.slot_of = lists.slot_of;
    A.bq = qx;
    A.hq = qh;
    A.ye = ye;
    A.err = scale_err_dev;

    // a block for every pass that the assignments can make (those without one return)
    auto grid = [&](int groups) { return dim3((unsigned)((pass_max(N, E) * groups + 7) / 8 * 8)); };
    if (xb) {
        const int64_t thr = (int64_t)n * 4 * k_steps(H);
        MH_LAUNCH("quant_x", k_quant_terms, dim3((unsigned)((thr + 255) / 256)), dim3(256), 0, s, xb, n, H, qx);
    }
    // gate/up over the quantized tokens, then down over the quantized h
    const bool words = (uintptr_t)L.experts % 16 != 0;
    auto gu = words ? k_moe_gemm<0, true> : k_moe_gemm<0, false>;
    auto down = words ? k_moe_gemm<1, true> : k_moe_gemm<1, false>;
    MH_LAUNCH("moe_gu_mfma", gu, grid(k_steps(F)), dim3(64 * kWaves), gemm_lds(2), s, A);
    A.bq = qh;
    MH_LAUNCH("moe_down_mfma", down, grid((H + kRows - 1) / kRows), dim3(64 * kWaves), gemm_lds(1), s, A);
    return hip_check(hipGetLastError(), "prefill MFMA launches");
}

}  // namespace mh
