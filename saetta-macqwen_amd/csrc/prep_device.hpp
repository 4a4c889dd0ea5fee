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

// The same for query values that nobody stores (a workgroup of the context makes its own), in a fifth of the instructions.
__device__ __forceinline__ float query_scale(float total, float eps) { return inverse_root(fmaf(total, 1.0f / float(SAETTA_HEAD_DIM), eps)); }

// Sine and cosine of rotary pair r of half_dims at a position, as on the CPU in f64 and rounded: the pair's frequency, which
// a kernel makes before it knows the position, then the two of the angle.
//
// sin() and cos() of the library, one after the other, stood in front of a token step's first scores (their code holds a
// reduction for any argument, twice).  Here the angle is reduced once: n quarter turns off it with pi / 2 as the sum of two
// doubles, fma by fma.  The first difference is exact (a multiple of the angle's or pi / 2's last place, below 2), so what is
// left is good to an ulp or so of f64 for angles up to 2^50 (frequencies of at most 1, a theta from 1 on, give angles below 2^32; any
// other theta takes library_angle); then the series of both to where the next term is below 2^-53 at pi / 4, rounded to f32.
// A layer's token step, us, with the norm below, ten layers in a graph: 8-bit 300 tokens of 8192 8.6 -> 8.4, 6000
// 10.2 -> 9.7, halves 20000 of 32768 16.3 -> 15.8, four rows over 4-bit codes at 1000 tokens 14.0 -> 13.2.
__device__ __forceinline__ double rope_frequency(uint32_t r, uint32_t half_dims, float log2_theta) {
    return exp2(-double(r) / double(half_dims) * double(log2_theta));
}
__device__ __forceinline__ void rope_angle(uint32_t position, double frequency, float &s, float &c) {
    const double angle = double(position) * frequency;
    const double n = rint(angle * 0.63661977236758134308);  // 2 / pi
    const double x = fma(-n, 6.123233995736766e-17, fma(-n, 1.5707963267948966, angle)), z = x * x;
    double sine = -1.0 / 1307674368000.0, cosine = 1.0 / 20922789888000.0;  // 1 / 15!, 1 / 16!
    sine = fma(sine, z, 1.0 / 6227020800.0), cosine = fma(cosine, z, -1.0 / 87178291200.0);
    sine = fma(sine, z, -1.0 / 39916800.0), cosine = fma(cosine, z, 1.0 / 479001600.0);
    sine = fma(sine, z, 1.0 / 362880.0), cosine = fma(cosine, z, -1.0 / 3628800.0);
    sine = fma(sine, z, -1.0 / 5040.0), cosine = fma(cosine, z, 1.0 / 40320.0);
    sine = fma(sine, z, 1.0 / 120.0), cosine = fma(cosine, z, -1.0 / 720.0);
    sine = fma(sine, z, -1.0 / 6.0), cosine = fma(cosine, z, 1.0 / 24.0);
    sine = fma(sine * z, x, x), cosine = fma(fma(cosine, z, -0.5), z, 1.0);
    const int quarter = int(n - 4.0 * floor(0.25 * n));
    const float fs = float(sine), fc = float(cosine), s0 = quarter & 1 ? fc : fs, c0 = quarter & 1 ? fs : fc;
    s = quarter & 2 ? -s0 : s0, c = (quarter + 1) & 2 ? -c0 : c0;
}
// The same for any frequency.
__device__ __forceinline__ void library_angle(uint32_t position, double frequency, float &s, float &c) {
    const double angle = double(position) * frequency;
    s = float(sin(angle)), c = float(cos(angle));
}
// Values u (index r) and w (index r + half) of a pair: the rotated first and second (one product rounded, the other fused).
__device__ __forceinline__ float rope_first(float u, float w, float s, float c) { return fmaf(u, c, -__fmul_rn(w, s)); }
__device__ __forceinline__ float rope_second(float u, float w, float s, float c) { return fmaf(u, s, __fmul_rn(w, c)); }

}  // namespace saetta
