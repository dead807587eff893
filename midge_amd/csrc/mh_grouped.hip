// mh_grouped.hip — the routed experts of a layer for a few tokens per expert
// (decode steps of several sequences, prompt chunks too short for the scaled
// matrix instruction's tiles) with each routed expert's weights read once for
// all the tokens routed to it: moe()'s per-slot expert work
// (engine/midge.c:514-541: gate and up matvecs + biases, the clamped SwiGLU,
// the down matvec + bias) regrouped by expert, as the reference's
// expert-major prefill groups tokens (engine/midge.c:591-611), on the f16
// matrix cores.
//
//   groups  the assignments of one expert in groups of up to kGroupTok; the
//           router's last block (or k_groups) writes the table of groups
//           (mh_internal.h, GroupTab).
//   units   8 tiles of 8 weight rows, one tile per wave: a gate/up tile is 4
//           pairs (gate rows p0 .. p0 + 3 and up rows p0 .. p0 + 3), a down
//           tile 8 rows. All groups' units are one list, and block b of the
//           grid (two blocks per CU) takes an equal consecutive share of it,
//           group by group. (A grid of 32-tile blocks per group filled
//           the chip 2.25 times at 16 tokens of gpt-oss-120b, the last time
//           to a quarter: gate/up 99 -> 85 us, down 59 -> 48 us. 40 tokens
//           of such a layer, ~92 experts, take 141 + 75 us, 6 TB/s of
//           weights; as per-assignment GEMVs they took 347 + 168 us.)
//   A       a K step is 256 elements: one load instruction reads the tile's
//           8 rows x 128 contiguous bytes (whole cache lines), lane (m, g)
//           the 16-byte MXFP4 chunk 8 s + 2 g + (m >> 3) of row m & 7, kPD
//           steps ahead in a ring of registers that runs on across tiles;
//           e2m1 times the chunk's f16 scale converts to f16 exactly for
//           scales that are zero or powers of two in [2^-23, 2^13].
//           Matrix-core rows m and m + 8 then hold the even and the odd
//           chunks of the same weight row.
//   scales  a tile's f16 scales (8 rows x K / 32) are one or two contiguous
//           runs of whole 16-byte pieces: two loads per lane bring them, and
//           the tile's 8 biases as two more pieces, into the wave's LDS
//           (double-buffered: the next tile's arrive while this one's steps
//           run), and each step reads its lane's scale there. One 16-bit
//           load per lane and step cost as much address work as the step's
//           weight load (92 vs 84 us per gate/up launch at 16 tokens of
//           gpt-oss-120b).
//   other   where nobody has looked at the layer's scales (a prefill takes a
//   scales  layer as it comes; a stack's plan scans them once), the wave
//           checks each tile's: one that f16 cannot carry sends the tile
//           through the vector ALUs (products and sums in f32, any f16
//           scale, like the GEMVs).
//   B       the group's inputs (xb of each assignment's token, or h of each
//           assignment) as two f16 terms, in columns 2j and 2j + 1 for the
//           even chunks and 8 + 2j, 9 + 2j for the odd ones (two LDS regions
//           placed so that a step's reads fall in distinct banks):
//           v' = v 2^-s, hi = RN(v'), lo = RN(v' - hi), with 2^s the power of
//           two that brings the column's max |v'| into [2^14, 2^15) (|v' - hi
//           - lo| <= 2^-22 |v'| + 2^-25); staged once per group and block
//           while the first weight loads fly. A column that holds an
//           infinity keeps only its infinities and NaNs (every row's sum is
//           then theirs).
//   cost    the e2m1 -> f16 conversion (one instruction per two codes) on
//           the vector ALU bounds the kernel with the weight stream: at 16
//           tokens of gpt-oss-120b a gate/up launch converts ~40 experts'
//           weights in ~53 us with its loads served from cache, against ~65
//           us of HBM time.
//   output  C[r][n] + C[r + 8][n + 8] (even plus odd chunks) for n = 2j and
//           2j + 1 added and scaled by 2^s; gate/up: + biases, activation ->
//           h[a][p]; down: + bias -> ye[a][r]. The products and sums run in
//           another order than the reference's row dots, like every
//           matrix-core path here.
#include <algorithm>

#include "mh_gemv.cuh"
#include "mh_mfma16.cuh"

namespace mh {

namespace {

constexpr int kGW = 8;                     // waves per block
constexpr int kGThreads = 64 * kGW;
constexpr int kGT = kGroupTok;             // assignments per group
constexpr int kGCols = 2 * kGT;            // B columns (hi, lo per assignment)
constexpr int kGMaxK = 3072;               // hidden and ffn
constexpr int kGE = kGMaxK / kGThreads;    // staged B elements per thread and column
constexpr int kPD = 4;                     // K steps in flight per wave (a tile's steps: a multiple)
constexpr int kGLdsMax = 80 * 1024;        // LDS per block (two blocks per CU)

struct GrpArgs {
    const uint8_t *experts;   // the layer's expert table
    uint32_t layer_bytes;     // E x stride (< 4 GiB)
    uint32_t stride;
    uint32_t off[9];          // wt_expert_layout offsets (engine/mten.h:136-150)
    int H, F, N, k;           // hidden, ffn, assignments (n k), slots per token
    float alpha, limit;
    int act_plain;
    GroupTab tab;
    const float *in;          // gate/up: xb [n][H]; down: h [N][F]
    float *out;               // gate/up: h [N][F]; down: ye [N][H]
};

// K steps of 256 per tile (rounded up to a multiple of kPD: the steps past
// K read zeros in B), and the f16 per B column of a region: the even (or
// odd) chunks of those steps, + 8, so that a column starts 4 banks after the
// previous one; the odd region starts 32 banks after the even one.
__host__ __device__ inline int grp_nq(int K) { return ((K / 32 + 7) / 8 + kPD - 1) / kPD * kPD; }
__host__ __device__ inline int grp_kh(int K) { return grp_nq(K) * 128 + 8; }
// 16-byte pieces of a tile's scales and biases
__host__ __device__ inline int grp_pc(int K) { return K / 32 + 2; }

// LDS of a block (bytes, 16-aligned parts): B (two regions of kGCols
// columns), the group's output scales, the waves' column maxima, and per
// wave two tiles' pieces.
struct GrpLds {
    size_t b, gs, mx, sc, total;
};
__host__ __device__ inline GrpLds grp_lds(int K) {
    GrpLds L;
    L.b = 0;
    L.gs = L.b + (size_t)2 * kGCols * grp_kh(K) * 2;
    L.mx = L.gs + (size_t)kGT * 4;
    L.sc = (L.mx + (size_t)kGW * kGT * 4 + 15) & ~(size_t)15;
    L.total = L.sc + (size_t)kGW * 2 * 16 * grp_pc(K);
    return L;
}

// Whether f16 carries e2m1 times each of a lane's scales (16 halves) exactly:
// each zero or a power of two in [2^-23, 2^13].
__device__ __forceinline__ bool scales_ok(const mh_u4 (&v)[2]) {
    uint32_t bad = 0u;
#pragma unroll 1
    for (int i = 0; i < 16; ++i) {
        const uint32_t w = i < 8 ? dword_of(v[0], i >> 1) : dword_of(v[1], (i >> 1) & 3);
        const uint32_t b = i & 1 ? w >> 16 : w & 0xFFFFu;
        // normal: no mantissa bits, at most 2^13; subnormal: one bit, at least 2^-23
        bad |= b >= 0x400u ? (b & 0x3FFu) | (b > 0x7000u ? 1u : 0u) : (b & (b - 1u)) | (b == 1u ? 1u : 0u);
    }
    return bad == 0u;
}

__device__ __forceinline__ float grp_act(float g, float u, float alpha, float limit, int plain) {
    if (plain) return g / (1.0f + expf(-g)) * u;
    if (g > limit) g = limit;
    if (u > limit) u = limit;
    if (u < -limit) u = -limit;
    const float a = g / (1.0f + expf(-alpha * g));
    return a * (u + 1.0f);
}

// One tile on the vector ALUs, for any f16 scales: w[i] of lane (m, g < 2) =
// row 4 g + i's sum for assignment m / 2, before the column's scale. Lane
// (m, g) adds its chunks (first, + 8, ..) of row r8 in f32 (codes exact, the
// chunk's sum times its scale, as the GEMVs do), then the row's 8 lanes add.
__device__ __forceinline__ void grp_tile_valu(mh_rsrc rex, uint32_t row, int C, int r8, int first, const uint16_t *scr,
                                              const _Float16 *sB, int kh, int cnt, int lane, float (&w)[4]) {
    // (rolled: this runs where a model's scales leave f16's range, and must
    // not take registers from the tiles that run on the matrix cores)
#pragma unroll 1
    for (int j = 0; j < cnt; ++j) {
        float s = 0.f;
#pragma unroll 1
        for (int c = first; c < C; c += 8) {
            const mh_u4 q = __builtin_amdgcn_raw_buffer_load_b128(rex, row + 16u * (uint32_t)c, 0, 0);
            const _Float16 *col = sB + ((size_t)(c & 1) * kGCols + 2 * j) * kh + (c >> 1) * 32;
            float d = 0.f;
#pragma unroll 1
            for (int i = 0; i < 4; ++i) {
                const v8h hi = *(const v8h *)(col + 8 * i), lo = *(const v8h *)(col + kh + 8 * i);
                const v8h a = fp4x8_f16(dword_of(q, i), 1.0f);
#pragma unroll
                for (int e = 0; e < 8; ++e) d = __builtin_fmaf((float)a[e], (float)hi[e] + (float)lo[e], d);
            }
            s = __builtin_fmaf(d, mh_f16(scr[c]), s);
        }
        s += __shfl_xor(s, 8);
        s += __shfl_xor(s, 16);
        s += __shfl_xor(s, 32);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float v = __shfl(s, (4 * (lane >> 4) + i) & 7);
            if ((lane & 15) >> 1 == j) w[i] = v;
        }
    }
}

// MODE 0: gate/up (K = H, tiles of 4 pairs); MODE 1: down (K = F, tiles of
// 8 rows). CHECK: look at each tile's scales (else they are known to be
// carried by f16).
// Two blocks per CU (their LDS fits twice) at four waves per SIMD (the
// launch bound's second argument, the minimum waves per SIMD, caps the
// registers at 128): the conversion work of some waves runs under the memory
// waits of others (at 3 waves per SIMD, 101 vs 92 us per gate/up launch at
// 16 tokens of gpt-oss-120b).
template <int MODE, bool CHECK>
__global__ void __launch_bounds__(kGThreads, 4) k_grouped(GrpArgs A) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const int K = MODE == 0 ? A.H : A.F;
    const int C = K / 32;   // 16-byte chunks per row
    const int PC = grp_pc(K);
    const int NQ = grp_nq(K);   // K steps of 256 per tile (a multiple of kPD)
    const int kh = grp_kh(K);
    const GrpLds Ld = grp_lds(K);
    _Float16 *sB = (_Float16 *)(lds + Ld.b);
    float *sGs = (float *)(lds + Ld.gs);    // [kGT] the columns' output scales 2^s
    float *sMax = (float *)(lds + Ld.mx);   // [kGW][kGT] staging: per-wave column maxima
    const int t = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(t >> 6), lane = t & 63;
    const int N = A.N;
    const int NG = A.tab.head[0], vend = A.tab.head[1];
    if (MODE == 1 && vend < N) {   // unroutable assignments contribute y = 0
        const int64_t nz = (int64_t)(N - vend) * A.H;
        for (int64_t i = (int64_t)blockIdx.x * kGThreads + t; i < nz; i += (int64_t)gridDim.x * kGThreads) {
            const int r = (int)(i / A.H);
            A.out[(size_t)A.tab.order[vend + r] * A.H + (i - (int64_t)r * A.H)] = 0.f;
        }
    }
    // this block's share of the units of all groups
    const int TPG = MODE == 0 ? A.F / 4 : A.H / 8;   // tiles per group
    const int UPG = (TPG + kGW - 1) / kGW;           // units per group
    const int U = NG * UPG;                          // < 2^31: checked at launch
    const int per = U / (int)gridDim.x, rem = U % (int)gridDim.x, b = (int)blockIdx.x;
    int u = b * per + min(b, rem);
    const int u1 = u + per + (b < rem ? 1 : 0);

    const mh_rsrc rex = gemv_rsrc(A.experts, A.layer_bytes);
    const int m = lane & 15, gq = lane >> 4;
    const int r8 = m & 7, par = m >> 3;   // this lane's weight row in the tile, chunk parity
    const uint32_t rowbytes = (uint32_t)C * 16u;
    uint8_t *sScW = lds + Ld.sc + (size_t)wave * 2 * 16 * PC;   // this wave's two buffers of pieces
    // B lane (n, g): region n >> 3, column n & 7, local chunk 4 s + g
    const _Float16 *bcol = sB + ((size_t)par * kGCols + r8) * kh + 32 * gq;

    while (u < u1) {   // one group at a time; block-uniform
        const int g = u / UPG, lo = u - g * UPG;
        const int nu = min(u1 - u, UPG - lo);
        u += nu;
        const GroupEnt *ge = A.tab.ent + g;
        const int cnt = __builtin_amdgcn_readfirstlane(ge->cnt);
        const uint32_t eo = (uint32_t)__builtin_amdgcn_readfirstlane(ge->expert) * A.stride;
        // this wave's tiles: tw0, tw0 + kGW, .. below tw1
        const int tw0 = lo * kGW + wave, tw1 = min((lo + nu) * kGW, TPG);

        // this lane's row of a tile: the byte offset of its data
        auto tile_row = [&](int tile) -> uint32_t {
            uint32_t row, od;
            if constexpr (MODE == 0) {
                row = 4u * (uint32_t)tile + (uint32_t)(r8 & 3);
                od = r8 < 4 ? A.off[0] : A.off[3];
            } else {
                row = 8u * (uint32_t)tile + (uint32_t)r8;
                od = A.off[6];
            }
            return eo + od + row * rowbytes;
        };
        // a tile's pieces: C of scales (gate/up: the 4 gate rows' run, then
        // the 4 up rows'; down: the 8 rows' run; 16-aligned since C is even),
        // kept in LDS with row r8 at byte 2 C r8, then two of biases
        auto sc_load = [&](int tile, mh_u4 (&v)[2]) __attribute__((always_inline)) {
            const uint32_t ut = (uint32_t)tile, uc = (uint32_t)C;
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const uint32_t p = (uint32_t)min(lane + 64 * i, PC - 1);
                uint32_t a;
                if constexpr (MODE == 0) {
                    a = p < uc / 2 ? A.off[1] + ut * 8u * uc + 16u * p : A.off[4] + ut * 8u * uc + 16u * (p - uc / 2);
                    if (p >= uc) a = (p == uc ? A.off[2] : A.off[5]) + 16u * ut;
                } else {
                    a = p < uc ? A.off[7] + ut * 16u * uc + 16u * p : A.off[8] + 32u * ut + 16u * (p - uc);
                }
                v[i] = __builtin_amdgcn_raw_buffer_load_b128(rex, eo + a, 0, 0);
            }
        };
        auto sc_store = [&](int buf, const mh_u4 (&v)[2]) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < 2; ++i)
                if (lane + 64 * i < PC) *(mh_u4 *)(sScW + (size_t)buf * 16 * PC + 16 * (lane + 64 * i)) = v[i];
        };
        // a tile whose scales f16 cannot all carry (the bias pieces are left
        // out; lanes past the pieces hold the last one again)
        auto odd_scales = [&](mh_u4 (&v)[2]) __attribute__((always_inline)) -> bool {
            uint32_t any = 0u;
            mh_u4 s[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const bool sc = lane + 64 * i < C;
                s[i] = mh_u4{sc ? v[i].x : 0u, sc ? v[i].y : 0u, sc ? v[i].z : 0u, sc ? v[i].w : 0u};
                any |= s[i].x | s[i].y | s[i].z | s[i].w;
            }
            // no sign, no mantissa bit, no exponent above 15: zeros and powers
            // of two up to 1; else look at each
            if (__ballot((any & 0xC3FFC3FFu) != 0u) == 0ull) return false;
            return __ballot(!scales_ok(s)) != 0ull;
        };

        // the ring: step s's chunk in slot s % kPD (the cursors advance by
        // selects: stores to one of two counters under a condition would be
        // merged into a store through a chosen pointer, which keeps the
        // counters in scratch memory)
        mh_u4 qa[kPD];
        int t_p = min(tw0, TPG - 1), q_p = 0;   // (a wave with no tiles reads one, unused)
        uint32_t rd_p = tile_row(t_p);
        auto issue = [&](int j) __attribute__((always_inline)) {
            const uint32_t cc = (uint32_t)min(8 * q_p + 2 * gq + par, C - 1);   // past K: a repeat (B is zero there)
            // (cached loads: non-temporal ones were slower here, 117 vs 102 us
            // per gate/up launch at 16 tokens of gpt-oss-120b)
            qa[j] = __builtin_amdgcn_raw_buffer_load_b128(rex, rd_p + 16u * cc, 0, 0);
            const bool wrap = q_p == NQ - 1;
            const bool adv = wrap && t_p + kGW < tw1;   // past the wave's tiles: the last again
            q_p = wrap ? 0 : q_p + 1;
            t_p = adv ? t_p + kGW : t_p;
            rd_p = tile_row(t_p);
        };

        // ---------------------------------------------------------- B
        // The group's inputs are loaded first, then the ring's first steps,
        // so that staging waits for its own loads only (loads complete in
        // issue order). Then each column's scale from its max |v| (one
        // barrier), and the terms, zeros past K.
        {
            int st = t;   // opaque: else the staging's addresses are kept in registers across the groups
            asm volatile("" : "+v"(st));
            float bv[kGT][kGE];
#pragma unroll
            for (int j = 0; j < kGT; ++j) {
                if (j < cnt) {   // block-uniform
                    const int a = __builtin_amdgcn_readfirstlane(ge->a[j]);
                    const float *src = MODE == 0 ? A.in + (size_t)(a / A.k) * A.H : A.in + (size_t)a * A.F;
#pragma unroll
                    for (int e = 0; e < kGE; ++e) bv[j][e] = src[min(st + e * kGThreads, K - 1)];
                }
            }
            mh_u4 sc0[2];   // the wave's first tile's pieces
            sc_load(t_p, sc0);
            for (int j = 0; j < kPD; ++j) issue(j);
            sc_store(0, sc0);
#pragma unroll
            for (int j = 0; j < kGT; ++j) {
                if (j >= cnt) break;   // block-uniform
                float mx = 0.f;
#pragma unroll
                for (int e = 0; e < kGE; ++e)
                    if (st + e * kGThreads < K) mx = fmaxf(mx, fabsf(bv[j][e]));
                mx = wave_max(mx);
                if (lane == 0) sMax[wave * kGT + j] = mx;
            }
            __syncthreads();   // also: every wave is done with the previous group's B
            // element k: chunk c = k / 32 in region c & 1 at (c >> 1) 32 + k % 32
            // of its column; k < NQ 256 covers every step (zeros past K). The
            // columns past the group's are not written: a matrix-core output
            // column reads only its own B column, and theirs are not used.
#pragma unroll
            for (int j = 0; j < kGT; ++j) {
                if (j >= cnt) break;   // block-uniform
                float mx = 0.f;
                for (int w = 0; w < kGW; ++w) mx = fmaxf(mx, sMax[w * kGT + j]);
                // 2^s with max |v| 2^-s in [2^14, 2^15): s = e - 15 for
                // max = f 2^e, f in [0.5, 1); 2^-s no larger than f32 holds,
                // s = 0 for a zero, subnormal or infinite max
                const int be = (int)((__float_as_uint(mx) >> 23) & 255u);   // mx in [2^(be-127), 2^(be-126))
                const bool inf = be == 255;
                const int sh = be > 0 && !inf ? max(be - 126 - 15, -126) : 0;
                const float down = ldexpf(1.0f, -sh);
                if (t == 0) sGs[j] = ldexpf(1.0f, sh);
#pragma unroll
                for (int e = 0; e < kGE; ++e) {
                    const int k = st + e * kGThreads;
                    if (k < NQ * 256) {
                        float v = k < K ? bv[j][e] * down : 0.f;
                        if (inf && fabsf(v) <= 3.4028235e38f) v = 0.f;
                        const _Float16 h = (_Float16)v;
                        const int c = k >> 5;
                        _Float16 *col = sB + ((size_t)(c & 1) * kGCols + 2 * j) * kh + (c >> 1) * 32 + (k & 31);
                        col[0] = h;                                               // hi
                        col[kh] = inf ? (_Float16)0.f : (_Float16)(v - (float)h);   // lo (the next column)
                    }
                }
            }
            __syncthreads();
        }
        // ge's assignment of this lane's output column
        const int aj = min(m >> 1, cnt - 1);
        const int a_out = ge->a[aj];
        const float gs = sGs[aj];
        const bool mine = m < 2 * cnt && (m & 1) == 0;
        // A tile's steps run in groups of kPD (ring slot j = step % kPD, a
        // constant), the accumulators live in the matrix-core registers
        // across them, and the outputs follow the tile's last group.
        int buf = 0;
        for (int tile = tw0; tile < tw1; tile += kGW, buf ^= 1) {
            mh_u4 scn[2];   // the next tile's pieces (the wave's last tile re-reads its own, unused)
            sc_load(tile + kGW < tw1 ? tile + kGW : tile, scn);
            const uint8_t *pcs = sScW + (size_t)buf * 16 * PC;
            const uint16_t *scr = (const uint16_t *)pcs + r8 * C;   // this lane's row
            v4f acc[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[i] = v4f{0.f, 0.f, 0.f, 0.f};
            for (int q0 = 0; q0 < NQ; q0 += kPD) {
                uint16_t scq[kPD];
#pragma unroll
                for (int j = 0; j < kPD; ++j) scq[j] = scr[min(8 * (q0 + j) + 2 * gq + par, C - 1)];
#pragma unroll
                for (int j = 0; j < kPD; ++j) {
                    const float sc = mh_f16(scq[j]);
                    const _Float16 *bp = bcol + 128 * (q0 + j);
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const v8h hb = *(const v8h *)(bp + 8 * i);
                        acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fp4x8_f16(dword_of(qa[j], i), sc), hb, acc[i],
                                                                        0, 0, 0);
                    }
                    issue(j);
                }
            }
            // ---- the tile's outputs
            const v4f accs = (acc[0] + acc[1]) + (acc[2] + acc[3]);
            // lane (n < 8, gq < 2) holds C[4 gq + i][n]; lane + 40 holds
            // C[4 gq + i + 8][n + 8]: even plus odd chunks, then the column
            // pair (hi, lo) of assignment n / 2
            float w[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float v = accs[i] + __shfl(accs[i], (lane + 40) & 63);
                w[i] = (v + dpp_shl<1>(v)) * gs;
            }
            if constexpr (CHECK) {
                mh_u4 own[2];   // this tile's scales again, from the wave's LDS
#pragma unroll
                for (int i = 0; i < 2; ++i) own[i] = *(const mh_u4 *)(pcs + 16 * min(lane + 64 * i, PC - 1));
                if (odd_scales(own)) {   // wave-uniform
                    grp_tile_valu(rex, tile_row(tile), C, r8, 2 * gq + par, scr, sB, kh, cnt, lane, w);
#pragma unroll
                    for (int i = 0; i < 4; ++i) w[i] *= gs;
                }
            }
            sc_store(buf ^ 1, scn);   // the wave reads its own LDS in order: no barrier
            const float4 b0 = *(const float4 *)(pcs + 16 * C), b1 = *(const float4 *)(pcs + 16 * C + 16);
            if constexpr (MODE == 0) {
                // gate rows 0-3 (gq 0), up rows 4-7 (gq 1): up from lane + 16
                float up[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) up[i] = __shfl(w[i], (lane + 16) & 63);
                if (mine && gq == 0) {
                    float4 o;
                    o.x = grp_act(w[0] + b0.x, up[0] + b1.x, A.alpha, A.limit, A.act_plain);
                    o.y = grp_act(w[1] + b0.y, up[1] + b1.y, A.alpha, A.limit, A.act_plain);
                    o.z = grp_act(w[2] + b0.z, up[2] + b1.z, A.alpha, A.limit, A.act_plain);
                    o.w = grp_act(w[3] + b0.w, up[3] + b1.w, A.alpha, A.limit, A.act_plain);
                    *(float4 *)(A.out + (size_t)a_out * A.F + 4 * tile) = o;
                }
            } else {
                if (mine && gq < 2) {
                    const float4 bd = gq ? b1 : b0;
                    *(float4 *)(A.out + (size_t)a_out * A.H + 8 * tile + 4 * gq) =
                        float4{w[0] + bd.x, w[1] + bd.y, w[2] + bd.z, w[3] + bd.w};
                }
            }
        }
    }
}

}  // namespace

bool grouped_ok(const DevLayer &L, int n) {
    const int64_t N = (int64_t)n * L.top_k;
    return L.expert_dt == MH_DT_MXFP4 && n >= 2 && N * (kGMaxK / 32) < (1ll << 31) && L.hidden % 64 == 0 &&
           L.ffn % 64 == 0 && L.hidden <= kGMaxK && L.ffn <= kGMaxK &&
           L.expert_stride % 16 == 0 && L.expert_stride * (uint64_t)L.n_experts < (1ull << 32) &&
           (uintptr_t)L.experts % 16 == 0 && L.off[0] % 16 == 0 && L.off[3] % 16 == 0 && L.off[6] % 16 == 0 &&
           L.off[1] % 16 == 0 && L.off[4] % 16 == 0 && L.off[7] % 16 == 0 &&
           L.off[2] % 16 == 0 && L.off[5] % 16 == 0 && L.off[8] % 16 == 0;
}

// What they read of an expert: codes and scales of K steps in whole groups of
// kPD (past K a repeat of the row's end, as slow as the rest).
double grouped_bytes(const DevLayer &L) {
    return 18.0 * 8.0 * (2.0 * L.ffn * grp_nq((int)L.hidden) + (double)L.hidden * grp_nq((int)L.ffn));
}

// The expert FFN of n tokens (grouped_ok) from the router's table of groups:
// h (scratch [N][F]) from xb, then ye [N][H]. exact: every scale of the layer
// is known to be carried by f16 (a stack's plan has looked).
int launch_grouped(const DevLayer &L, int n, const GroupTab &tab, const float *xb, float *h, float *ye, bool exact,
                   hipStream_t s) {
    if (!grouped_ok(L, n)) return fail(MH_E_UNSUPPORTED, "grouped expert path: shape not handled");
    GrpArgs A;
    A.experts = L.experts;
    A.layer_bytes = (uint32_t)(L.expert_stride * (uint64_t)L.n_experts);
    A.stride = (uint32_t)L.expert_stride;
    for (int i = 0; i < 9; i++) A.off[i] = (uint32_t)L.off[i];
    A.H = (int)L.hidden;
    A.F = (int)L.ffn;
    A.N = n * L.top_k;
    A.k = L.top_k;
    A.alpha = L.alpha;
    A.limit = L.limit;
    A.act_plain = L.act_plain;
    A.tab = tab;
    const GrpLds l0 = grp_lds(A.H), l1 = grp_lds(A.F);
    if (l0.total > kGLdsMax || l1.total > kGLdsMax)
        return fail(MH_E_UNSUPPORTED, "grouped expert path: LDS of %zu / %zu bytes per block", l0.total, l1.total);
    static uint64_t ready = 0;   // the initialisation whose device has the attributes
    if (ready != init_epoch()) {
        for (const void *f : {(const void *)k_grouped<0, false>, (const void *)k_grouped<0, true>,
                              (const void *)k_grouped<1, false>, (const void *)k_grouped<1, true>})
            MH_HIP(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, kGLdsMax));
        ready = init_epoch();
    }
    // two blocks per CU, fewer where the units of all possible groups are fewer
    const int64_t cap = 2 * (int64_t)device_cus();
    auto grid = [&](int tiles) {
        return dim3((unsigned)std::min<int64_t>(cap, (int64_t)A.N * ((tiles + kGW - 1) / kGW)));
    };
    A.in = xb;
    A.out = h;
    if (exact)
        MH_LAUNCH("grouped_gu", (k_grouped<0, false>), grid(A.F / 4), dim3(kGThreads), l0.total, s, A);
    else
        MH_LAUNCH("grouped_gu", (k_grouped<0, true>), grid(A.F / 4), dim3(kGThreads), l0.total, s, A);
    MH_TRY(hip_check(hipGetLastError(), "grouped gate/up launch"));
    A.in = h;
    A.out = ye;
    if (exact)
        MH_LAUNCH("grouped_down", (k_grouped<1, false>), grid(A.H / 8), dim3(kGThreads), l1.total, s, A);
    else
        MH_LAUNCH("grouped_down", (k_grouped<1, true>), grid(A.H / 8), dim3(kGThreads), l1.total, s, A);
    return hip_check(hipGetLastError(), "grouped down launch");
}

}  // namespace mh
