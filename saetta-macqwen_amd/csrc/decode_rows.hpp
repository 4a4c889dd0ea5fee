// What decode_half_rows.hpp and decode_code_rows.hpp share: counters in LDS, the norm of a computing wave's query values, the
// split of a product.  Included by decode.hip, inside its namespace.  (A workgroup's share of the context stays in both: as a
// struct of its own it changed the loops: 6 rows over halves at 57123 tokens 35.5 -> 35.9 us a layer.)

// Counters in LDS through which waves meet (see attention_partial_s_body): one lane adds, the others poll, and every wait is
// bounded.  `lost`: the counter, behind the kernel's CODE, of a wait that gave up.
template <uint32_t SPIN_LIMIT, uint32_t CODE, uint32_t COUNT_MASK = ~0u>
struct LdsCounters {
    uint32_t *counters;
    uint32_t lane, lost = 0;

    __device__ __forceinline__ void raise(uint32_t c, uint32_t by = 1) const {
        asm volatile("" ::: "memory");
        if (lane == 0) __hip_atomic_fetch_add(counters + c, by, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        asm volatile("" ::: "memory");
    }
    __device__ __forceinline__ uint32_t peek(uint32_t c) const {
        asm volatile("" ::: "memory");
        const uint32_t v = __hip_atomic_load(counters + c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        asm volatile("" ::: "memory");
        return uint32_t(__builtin_amdgcn_readfirstlane(v));
    }
    // until the counter's COUNT_MASK part has come to `want`; the whole counter
    __device__ __forceinline__ uint32_t await(uint32_t c, uint32_t want) {
        asm volatile("" ::: "memory");
        uint32_t left = SPIN_LIMIT, v;
#pragma nounroll
        do {
            v = __builtin_amdgcn_readfirstlane(__hip_atomic_load(counters + c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
            if ((v & COUNT_MASK) >= want) break;
            __builtin_amdgcn_s_sleep(1);
        } while (--left);
        if (__builtin_expect(left == 0, 0)) lost = CODE + c;
        asm volatile("" ::: "memory");
        return v;
    }
};

// The query norm of a computing wave: of its pair a lane has dims dim_of(s) .. + 7 as q[s], the other lanes of its column
// (16, 32 and 48 further) the rest.
template <typename DimOf>
__device__ __forceinline__ void norm_query(float (&q)[8][8], const PrepArgs &prep, DimOf dim_of) {
    float sum = 0.0f;
#pragma unroll
    for (int s = 0; s < 8; s++) {
#pragma unroll
        for (int e = 0; e < 8; e++) sum += q[s][e] * q[s][e];
    }
    const float scale = query_scale(across_rows<16, 64>(sum, SumOp()), prep.p.eps);
#pragma unroll
    for (int s = 0; s < 8; s++) {
        const float4 *w = reinterpret_cast<const float4 *>(prep.q_norm + dim_of(s));
        const float4 f0 = w[0], f1 = w[1];
        const float wv[8] = {f0.x, f0.y, f0.z, f0.w, f1.x, f1.y, f1.z, f1.w};
#pragma unroll
        for (int e = 0; e < 8; e++) q[s][e] *= scale * wv[e];
    }
}

// x * y as f16 hi and lo parts: hi with the product's low mantissa bits cut off, lo what that leaves of the exact product (one
// fused operation from it to the f16).
__device__ __forceinline__ void split_product(float x, float y, _Float16 &hi, _Float16 &lo) {
    hi = (_Float16)__builtin_bit_cast(float, __builtin_bit_cast(uint32_t, x * y) & 0xffffe000u);
    lo = (_Float16)fmaf(x, y, -(float)hi);
}
constexpr float NEVER = -3e38f;  // the score of a masked token: below any maximum, its probability is 0
