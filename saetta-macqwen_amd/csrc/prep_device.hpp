// The step before the scores as the kernels that do it share it: attention_prep_store_kernel (prep.hip) and the
// attention kernels of a plan's token step, which take it in (decode.hip).
#pragma once
#include "common.hpp"
#include "lanes.hpp"

namespace saetta {

struct PrepArgs {
    const float *q_and_gate;  // [row][heads][2 * dim]
    const float *k, *v;       // [row][kv_heads][dim]
    const float *q_norm, *k_norm;
    float *q_out;             // [row][heads][dim]
    uint16_t *keys_half, *values_half;  // half cache [capacity][kv_heads][dim], or null
    saetta_quant_rows kq, vq;           // quantized cache (BITS 8 or 4)
    float *k_back;                      // [row][kv_heads][dim]: the normed, rotated key in f32, or null
    saetta_prep_params p;
    const saetta_token_params *tp;
    uint32_t capacity;
};

// The sum of the squares of a wavefront's 64 values, in lane 0.  Every operation is spelled out, since what is stored
// rests on its bits: the first step is a fused multiply and add, whose rounding differs between the two lanes of a pair.
__device__ __forceinline__ float square_sum(float x) {
    float y = fmaf(x, x, dpp<0xb1>(__fmul_rn(x, x)));
    y = __fadd_rn(y, dpp<0x4e>(y));
    y = __fadd_rn(y, dpp<0x141>(y));
    y = __fadd_rn(y, dpp<0x140>(y));
    return across_rows<16, 64>(y, SumOp());
}

// What the head's values are multiplied by beside the norm's weight: 1 / sqrt(mean(x^2) + eps).  `total` is the sum of the
// squares; of the four groups of 64 dims' sums as (0 + 1) + (2 + 3) where bits count.
__device__ __forceinline__ float norm_scale(float total, float eps) {
    return __fdiv_rn(1.0f, __fsqrt_rn(__fadd_rn(__fdiv_rn(total, float(SAETTA_HEAD_DIM)), eps)));
}

// Sine and cosine of rotary pair r of half_dims at a position, as on the CPU in f64 and rounded.
__device__ __forceinline__ void rope_angle(uint32_t position, uint32_t r, uint32_t half_dims, float log2_theta, float &s, float &c) {
    const double freq = exp2(-double(r) / double(half_dims) * double(log2_theta));
    const double angle = double(position) * freq;
    s = float(sin(angle)), c = float(cos(angle));
}
// Values u (index r) and w (index r + half) of a pair: the rotated first and second (one product rounded, the other fused).
__device__ __forceinline__ float rope_first(float u, float w, float s, float c) { return fmaf(u, c, -__fmul_rn(w, s)); }
__device__ __forceinline__ float rope_second(float u, float w, float s, float c) { return fmaf(u, s, __fmul_rn(w, c)); }

}  // namespace saetta
