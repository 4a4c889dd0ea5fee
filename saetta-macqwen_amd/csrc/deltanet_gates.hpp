// Shared by the Gated DeltaNet kernel files: the gates of a token and head, the conv's activation.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace saetta {

// From this many tokens on (without snapshots) saetta_deltanet_rows runs the chunked form of the
// delta rule on the matrix cores (deltanet_chunk.hip); below it the token-by-token kernels.
constexpr uint32_t DELTANET_CHUNK_FROM = 128;

// g = exp(-exp(A_log) softplus(a + dt_bias)), beta = sigmoid(b), with the hardware's exp2 and log2
// (the library routines are some 150 instructions, and in the kernels the gates sit in one wave's
// path): log1p(e) as e - e^2 / 2 below 2^-10 and log(1 + e) above; the errors stay near 1e-7.
// log_g, if asked for, is the exponent itself.
__device__ __forceinline__ void fast_gates(float a_plus_bias, float exp_a_log, float b, float &g, float &beta,
                                           float *log_g = nullptr) {
    const float e = __expf(-fabsf(a_plus_bias));
    const float log1p_e = e < 0x1p-10f ? e * (1.0f - 0.5f * e) : __logf(1.0f + e);
    const float softplus = fmaxf(a_plus_bias, 0.0f) + log1p_e;
    const float lg = -exp_a_log * softplus;
    if (log_g) *log_g = lg;
    g = __expf(lg);
    beta = __builtin_amdgcn_rcpf(1.0f + __expf(-b));
}

__device__ __forceinline__ float sigmoid_f(float x) { return 1.0f / (1.0f + expf(-x)); }
// x / (1 + e^-x): the exponent as a product and what its rounding leaves out, the hardware's exp2, and the quotient by the
// hardware's reciprocal and one step on what the product with it leaves of x (no further off than expf and a division, on the
// average nearer; zero where e^-x is beyond f32).  From e^-x = 2^64 on the divisor is taken 2^64 smaller and the quotient by as much
// too large, for from 2^126 on the hardware's reciprocal is zero.  The library's two calls, thirty instructions in a row, stood
// twice on the path of a DeltaNet token's one launch.
__device__ __forceinline__ float silu_f(float x) {
    constexpr float LOG2_E = 0x1.715476p+0f, LOG2_E_REST = 0x1.4ae0cp-26f, LN_2 = 0x1.62e43p-1f;
    const float at = -LOG2_E * x, rest = fmaf(-LOG2_E_REST, x, fmaf(-LOG2_E, x, LOG2_E * x));
    // (where e^-x is zero or infinite no rest, but not zero, which times an infinity is NaN)
    const float tail = fabsf(at) < 128.0f ? LN_2 * rest : 0x1p-64f, down = at > 64.0f ? 0x1p-64f : 1.0f;
    const float e = __builtin_amdgcn_exp2f(at), d = fmaf(fmaf(e, tail, e), down, down), r = __builtin_amdgcn_rcpf(d);
    const float y = x * r, off = fmaf(-d, y, x), y_down = y * down;
    return off == off ? fmaf(off, r * down, y_down) : y_down;
}
// silu_f of four values: where none of the wavefront's is beyond +-44, and none therefore meets a bound above, the same steps
// without the bounds (eleven instructions a value, not eighteen; the same bits).
__device__ __forceinline__ float4 silu4_f(float4 x) {
    if (__any(fmaxf(fmaxf(fabsf(x.x), fabsf(x.y)), fmaxf(fabsf(x.z), fabsf(x.w))) > 44.0f)) return make_float4(silu_f(x.x), silu_f(x.y), silu_f(x.z), silu_f(x.w));
    auto inside = [](float v) {
        constexpr float LOG2_E = 0x1.715476p+0f, LOG2_E_REST = 0x1.4ae0cp-26f, LN_2 = 0x1.62e43p-1f;
        const float at = -LOG2_E * v, rest = fmaf(-LOG2_E_REST, v, fmaf(-LOG2_E, v, LOG2_E * v));
        const float e = __builtin_amdgcn_exp2f(at), d = fmaf(e, LN_2 * rest, e) + 1.0f, r = __builtin_amdgcn_rcpf(d);
        const float y = v * r;
        return fmaf(fmaf(-d, y, v), r, y);
    };
    return make_float4(inside(x.x), inside(x.y), inside(x.z), inside(x.w));
}

}  // namespace saetta
