// mh_fp6.cuh — activations as fp6 e2m3 terms: the records that the prefill's
// matrix product reads (mh_prefill.hip) and their writer, shared with the
// router that forms the normed input (mh_moe.hip).
#pragma once

#include "mh_internal.h"

namespace mh {

typedef int v6i __attribute__((ext_vector_type(6)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v32f __attribute__((ext_vector_type(32)));

constexpr int kTerms = 3;   // fp6 terms per activation

// A quantized row is a record of kRec bytes per K step of 128 columns (4
// blocks): the terms' 16-byte low pieces of the 4 blocks (codes 0..20 and a
// third of code 21), term by term, then the terms' 8-byte high pieces, then
// per block its terms' e8m0 scales in the bytes of one word. The GEMM takes
// a step's record with 16-byte loads of whole pieces.
constexpr int kRecHi = kTerms * 64, kRecSc = kTerms * 96, kRec = kTerms * 96 + 16;
static_assert(kRecSc + 16 == kRec && kTerms <= 4, "record layout");
// (two steps at least, zeros past K: the GEMM's loads run that far ahead)
__host__ __device__ inline int k_steps(int K) { return K > 128 ? (K + 127) / 128 : 2; }

// e such that m * 2^-e <= 7.5 (the largest e2m3 value), as small as possible.
__device__ __forceinline__ int fp6_block_exp(float m) {
    int km;
    const float fm = frexpf(m, &km);   // m = fm * 2^km, fm in [0.5, 1)
    return fm <= 0.9375f ? km - 3 : km - 2;
}

// Block g of a step's record from its 32 values. Each term is the previous
// residual divided by 2^e and rounded by the hardware converter, which
// interleaves its two 16-value inputs (even columns, odd columns); its values
// come back exactly from the inverse converter, so the residuals are exact.
// A zero block keeps e = 0.
__device__ __forceinline__ void quant_block(float (&v)[32], uint8_t *rec, int g) {
    uint32_t sc = 0u;
#pragma unroll
    for (int t = 0; t < kTerms; ++t) {
        float m = 0.f;
#pragma unroll
        for (int j = 0; j < 32; ++j) m = fmaxf(m, fabsf(v[j]));
        const int e = m > 0.f ? max(-126, min(127, fp6_block_exp(m))) : 0;
        const float scl = ldexpf(1.0f, e);
        v16f ev, od;
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            ev[j] = v[2 * j];
            od[j] = v[2 * j + 1];
        }
        const v6i w = __builtin_amdgcn_cvt_scalef32_2xpk16_fp6_f32(ev, od, scl);
        const v32f back = __builtin_amdgcn_cvt_scalef32_pk32_f32_fp6(w, scl);
#pragma unroll
        for (int j = 0; j < 32; ++j) v[j] -= back[j];
        *(uint4 *)(rec + 64 * t + 16 * g) = make_uint4((uint32_t)w[0], (uint32_t)w[1], (uint32_t)w[2], (uint32_t)w[3]);
        *(uint2 *)(rec + kRecHi + 32 * t + 8 * g) = make_uint2((uint32_t)w[4], (uint32_t)w[5]);
        sc |= (uint32_t)(e + 127) << (8 * t);
    }
    *(uint32_t *)(rec + kRecSc + 4 * g) = sc;
}

}  // namespace mh
