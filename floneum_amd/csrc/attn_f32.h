// Pieces shared by the prefill kernels that compute in f32 precision (attn_prefill_f32.hip, attn_prefill_f32_terms.hip).
#pragma once
#include "common.h"
#include "device_utils.h"

namespace fhip {

constexpr float PF32_LOG2E = 1.4426950408889634f;

// How a mask tensor is applied (MODE):
//   PF32_INTERVALS  by interval: analytic description, key counts, or the interval form a scan launch left in p.iv
//   PF32_BIAS       the tensor is added as it is, element by element (p.mask, no interval form): finite biases,
//                   several visible runs per row, NaN or +inf entries.  Score = (q.k * scale) + mask as in the
//                   reference (fusor flash_attention.rs:145,177), every key tile is visited.
//   PF32_EITHER     decided when the kernel starts, from the word the scan launch in front of it left in *p.iv_bad:
//                   by interval (p.iv) if every row of the mask is one, else the values are added.  No hand-over
//                   launch behind the tiled kernel; head_dim <= 64 (the register budget of both forms in one kernel).
constexpr int PF32_INTERVALS = 0, PF32_BIAS = 1, PF32_EITHER = 2;

// Probabilities are formed against a row's reference m, the maximum its scores had when it was last set: exp2(s * unit -
// m * unit) in one fused multiply-add and one exponential, `unit` being 1 where scores are exponents of two and log2(e)
// where a mask has been added to them.  (The score itself takes no log2(e): a sum of a score and a mask value that is rounded
// again at its own size has lost another bit of it.)  m * unit is the rounded product everywhere.  It overflows for references
// below -2.36e38, rows of which every score so far holds a padding value like f32's or bf16's lowest: neighbours are
// 2e31 apart there, so a score that equals m has probability 1 and every other 0.
__device__ __forceinline__ float probability(float s, float m, float unit) {
    const float m2 = m * unit;
    if (m2 == -INFINITY) return s == m && m > -INFINITY ? 1.0f : s != s ? s : 0.0f;
    return __builtin_amdgcn_exp2f(__builtin_fmaf(s, unit, -m2));
}
// what probabilities formed against m are to be multiplied by when the reference is m_new >= m
__device__ __forceinline__ float moved_reference(float m, float m_new, float unit) {
#pragma clang fp contract(off)
    const float m2 = m * unit, m2_new = m_new * unit;  // both rounded, as where probabilities are formed
    return m == m_new ? 1.0f : m2 == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m2 - m2_new);
}

// four consecutive elements of a row as f32 (16-bit storage types are widened exactly)
__device__ __forceinline__ float4_t load4(const float *p) { return *(const float4_t *)p; }
__device__ __forceinline__ float4_t load4(const half_t *p) {
    const half4_t h = *(const half4_t *)p;
    return float4_t{(float)h[0], (float)h[1], (float)h[2], (float)h[3]};
}
__device__ __forceinline__ float4_t load4(const bf16_t *p) {
    const uint2_t u = *(const uint2_t *)p;
    return float4_t{__uint_as_float(u[0] << 16), __uint_as_float(u[0] & 0xffff0000u), __uint_as_float(u[1] << 16),
                    __uint_as_float(u[1] & 0xffff0000u)};
}
// one output element: the tensors' type, or f32 when the call asks for an f32 result of 16-bit inputs
template <typename T>
__device__ __forceinline__ void store_out(const AttnParams &p, int64_t idx, float v) {
    if (sizeof(T) == 4 || p.out_f32) ((float *)p.out)[idx] = v;
    else ((T *)p.out)[idx] = from_float<T>(v);
}

__device__ __forceinline__ float half_swap_max32(float x) {
    auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float half_swap_sum32(float x) {
    auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

}  // namespace fhip
