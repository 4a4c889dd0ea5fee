// Gated DeltaNet over the tokens of a prefill chunk on the matrix cores: the delta rule in its
// chunked form, blocks of 64 tokens.
//
// What it computes is what deltanet_rows_kernel computes token by token (the reference's definition:
// src/cpu/deltanet.rs:69-155, delta_rule :148-155; the kernels it stands for: delta_prep + delta_rows3,
// kernels/prefill.metal:788-1116): per value head, with state S [v_dim][128],
//     S <- g_t S;  u_t = beta_t (v_t - S k_t);  S += u_t k_t^T;  o_t = S q_t.
// Inside a block of C = 64 tokens, with c_t = sum_{r <= t} log g_r and S0 the state before the block,
//     S_t = e^{c_t} S0 + sum_{s <= t} e^{c_t - c_s} u_s k_s^T,
// so the u_t solve a triangular system that does not involve the state's rows one by one:
//     (I + A) U = diag(beta) (V - diag(e^c) K S0^T),   A_ts = beta_t e^{c_t - c_s} (k_t . k_s)  (s < t)
//     O = diag(e^c) Q S0^T + M U,                       M_ts = e^{c_t - c_s} (q_t . k_s)         (s <= t)
//     S1^T = e^{c_last} S0^T + K^T diag(e^{c_last - c}) U
// (U, V, O: [C][v_dim]; K, Q: [C][128], normalised as the reference does).  Two kernels:
//   deltanet_chunk_prepare_kernel   one workgroup per (block, key head) with its two value heads (or per
//       value head, for another ratio), all blocks at once: the
//       normalised q and k, A and M (64 x 64 x 128 products), T = (I + A)^-1 diag(beta) by forward
//       substitution, and the decay factors, to a workspace;
//   deltanet_chunk_chain_kernel     one workgroup per (16 value dims, value head) walks the blocks in
//       order with its slice of the state in registers: five small products per block.
// All products run on v_mfma_f32_16x16x32_f16 with every operand split into an f16 hi and lo part
// (hi * hi + hi * lo + lo * hi: about 2^-21 relative, against 2^-24 of the f32 chain; f32 MFMA has an
// eighth of the rate per k and wants one LDS read per operand element).  The exponents e^{c_t - c_s}
// never exceed 1 and come from running sums of log g kept in f64 (in f32 the difference of two sums of
// some tens loses what the product of the g themselves keeps).  The output differs from the
// token-by-token kernels' by rounding only (tests hold it to 2e-5 of the largest value, also over a
// 4096-token chunk; measured 2e-6).
#include "common.hpp"
#include "deltanet_gates.hpp"
#include "lanes.hpp"

#include <type_traits>

namespace saetta {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr int K_DIM = 128;
constexpr int C = 64;                 // tokens per block
constexpr int DV = 16;                // value dims per workgroup of the chain kernel (32: 317 against 253 us per 4096 tokens)
constexpr float Q_SCALE = 0.08838834764831845f;  // 1 / sqrt(128), the reference's factor on q
// LDS images of the prepare kernel: rows padded so that 16 rows' 16-byte reads fall on all banks
constexpr int KROW = K_DIM + 8;       // f16 per row of a q / k image: 272 bytes
constexpr int TROW = C + 8;           // f16 per row of a T / M image (and of the chain's [dv][token] images): 144 bytes
constexpr int K_IMG = C * KROW * 2;   // bytes: 17408
constexpr int T_IMG = C * TROW * 2;   // bytes: 9216

// Workspace, per block.  Everything the chain kernel reads lies in the order its waves take it as MFMA
// operands: an operand of a wave is 64 lanes x 16 bytes = 1 KB (lane (n, j): row or column n, 8 values of
// the k index from 8j), so a load instruction of a wave reads one contiguous kilobyte.
//   per key head:   K hi | K lo | Q hi | Q lo   [wave 4][k-step 4][lane]: row 16 wave + n, key dims 32 ks + 8j ..
//   per value head: T hi | T lo | M hi | M lo   [wave 4][k-step 2][lane]: row 16 wave + n, columns 32 ks + 8j ..
//                   128 floats: e^{c_t} and e^{c_last - c_t}
constexpr int OPERAND = 1024;
constexpr int K_GL = 4 * 4 * OPERAND, T_GL = 4 * 2 * OPERAND;
constexpr size_t KHEAD_BYTES = 4 * size_t(K_GL);
constexpr size_t VHEAD_BYTES = 4 * size_t(T_GL) + 2 * C * sizeof(float);
__host__ __device__ inline size_t block_bytes(uint32_t k_heads, uint32_t v_heads) { return k_heads * KHEAD_BYTES + v_heads * VHEAD_BYTES; }

struct ChunkArgs {
    const float *mixed, *a, *b, *a_log, *dt_bias;
    float *state;
    float *o;  // [tokens][v_heads][v_dim], before the gated norm
    unsigned char *ws;
    uint32_t k_heads, v_heads, v_dim, tokens, channels;
    float eps;
    // the conv before it, where the prepare kernel makes that too (`mixed` is then its output)
    const float *x, *conv_w;
    float *conv_state;
};
constexpr int CONV = 4;     // taps of the conv that the prepare kernel makes
constexpr int CONV_V = 128;  // ... and the value dim it takes

// Four values as f16 hi parts and f16 lo parts.  A lo part has to complete the hi part that is stored: where x is
// a product, the compiler may round the exact product to f16 for the one and the f32 product for the other, and
// next to a midpoint between two f16 numbers the two roundings differ by an ulp of the hi part (one value in
// some thousands: an error of 2^-11 of it instead of 2^-22).  So x is pinned as the f32 number it is, and the
// hi parts, two to a conversion, as the numbers that the lo parts are taken against.
typedef _Float16 half2_ __attribute__((ext_vector_type(2)));
template <class F>
__device__ __forceinline__ void split4(F &&value, half4 &hi, half4 &lo) {
    half2_ h[2], l[2];
    float minus = -1.0f;  // not as a constant: x - hi is then one v_fma_mix, taken from and rounded to f16, and not three instructions
    asm("" : "+s"(minus));
#pragma unroll
    for (int p = 0; p < 2; p++) {
        float x = value(2 * p), y = value(2 * p + 1);
        asm("" : "+v"(x), "+v"(y));
        uint32_t both = __builtin_bit_cast(uint32_t, half2_{(_Float16)x, (_Float16)y});
        asm("" : "+v"(both));
        h[p] = __builtin_bit_cast(half2_, both);
        l[p] = half2_{(_Float16)__builtin_fmaf((float)h[p][0], minus, x), (_Float16)__builtin_fmaf((float)h[p][1], minus, y)};
    }
    hi = __builtin_shufflevector(h[0], h[1], 0, 1, 2, 3), lo = __builtin_shufflevector(l[0], l[1], 0, 1, 2, 3);
}

// acc += A B with both operands in hi and lo parts
__device__ __forceinline__ floatx4 mma3(half8 ah, half8 al, half8 bh, half8 bl, floatx4 acc) {
    acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(al, bh, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah, bl, acc, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(ah, bh, acc, 0, 0, 0);
}

// ---- prepare: everything of a block that does not depend on the state ------------------------------
// One workgroup of eight waves takes G value heads of one key head: the q / k images and the k . k and q . k products
// belong to the key head, the gates, A, M and T to a value head.  (G = 2: the model's two value heads per key head;
// G = 1: any other ratio, one workgroup per value head, the first of a key head's writing the key head's images.)
// What bounds it: a workgroup is a chain of short phases, and with few blocks (up to 1024 tokens: a workgroup to a CU)
// that chain is the kernel's time, with many the memory (69 MB read and 118 written at 4096 tokens in 40 us: 4.7 TB/s).  So the phases are
// spread over two teams of four waves, a row tile of 16 tokens to a wave: one makes A and solves for T, the other makes M
// and stores it meanwhile; the products are taken as their transposes, so that a lane's four results lie in a row and
// leave as one 8-byte store; the solve has a lane to a column, with no sums over lanes.
// Measured, us, against four waves that did it all in order: 1000 tokens 22.7 -> 15.8, 2047 28.3 -> 26.4, 4096 57.4 -> 49.8;
// with the conv inside, 512 tokens 31.5 -> 20.3; then 4096 49.8 -> 40: of the 34 000 cycles of a block with its conv most were waits for something that
// need not be waited for, or one wave's work: without them 25 000, and 20 400 of 25 900 without the conv (whole chunk: 130
// tokens 28.9 -> 25.3, 500 38.7 -> 35.6, 1000 60.2 -> 57.9, 2300 127.2 -> 121.4, 4096 230.3 -> 223.3, with the chain's outputs
// in whole lines and the conv's and norm's short activation 219).
// LDS: the four q / k images; once the products are taken, the heads' A (f32) go over kh | kl, their M
// images and later their T images over qh | ql (and more), so that they leave as whole 16-byte stores.
constexpr int PREP_THREADS = 512, PREP_WAVES = PREP_THREADS / 64;
template <int G>
struct PrepLds {
    // per head, over kh | kl once the products are taken: the two diagonal 32 x 32 blocks of A as f32, rows of
    // DROW (their inverses go over them, the product of the off-diagonal block over those later), then the
    // block below the diagonal and the inverse of the second diagonal block as f16 images
    // (a diagonal block is 128 bytes longer than its rows: what the four 16 x 16 blocks of a solve read at once lies in different banks)
    static constexpr int DROW = 32 + 4, D_BYTES = 32 * DROW * 4 + 128;
    static constexpr int HROW = 32 + 8, H_IMG = 32 * HROW * 2;  // f16 per row of a 32 x 32 image; bytes of one part
    static constexpr int W_OFF = 0, LBA_OFF = 2 * D_BYTES, XBB_OFF = LBA_OFF + 2 * H_IMG, HEAD_BYTES = XBB_OFF + 2 * H_IMG;
    static_assert(2 * H_IMG <= 2 * D_BYTES, "the product's images fit over the diagonal blocks");
    static constexpr int M_BYTES = 2 * T_IMG;  // mh | ml (then th | tl) of a head
    static constexpr int M_OFF = G * HEAD_BYTES > 2 * K_IMG ? G * HEAD_BYTES : 2 * K_IMG;
    static constexpr int GATES = M_OFF + G * M_BYTES > 4 * K_IMG ? M_OFF + G * M_BYTES : 4 * K_IMG;  // [head]: cum f64 [C] | beta f32 [C]
    static constexpr int GATE_BYTES = C * 8 + C * 4;
    static constexpr int BYTES = GATES + G * GATE_BYTES;
    static_assert(2 * BYTES <= 160 * 1024, "two workgroups per CU");
};

// x of the lane that DPP control CTRL names, zero where there is none or the row is not in ROWS
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_or_zero(double x) {
    const u32x2 v = __builtin_bit_cast(u32x2, x);
    return __builtin_bit_cast(double, u32x2{uint32_t(__builtin_amdgcn_update_dpp(0, int(v.x), CTRL, ROWS, 0xf, false)),
                                            uint32_t(__builtin_amdgcn_update_dpp(0, int(v.y), CTRL, ROWS, 0xf, false))});
}
// The inclusive sum over the lanes of a wavefront: inside rows of 16 lanes, then row by row.
__device__ __forceinline__ double inclusive_sum(double x) {
    x += dpp_or_zero<0x111, 0xf>(x), x += dpp_or_zero<0x112, 0xf>(x);  // row_shr 1, 2
    x += dpp_or_zero<0x114, 0xf>(x), x += dpp_or_zero<0x118, 0xf>(x);  // row_shr 4, 8
    x += dpp_or_zero<0x142, 0xa>(x);                                   // row_bcast 15, to rows 1 and 3
    return x + dpp_or_zero<0x143, 0xc>(x);                             // row_bcast 31, to rows 2 and 3
}

// The B operand of a 16-column tile out of a row-major f16 image in LDS (hi part at `at`, lo part `part_bytes`
// on; `at`: the byte address of row 8j + e, column 4a of the tile for lane a + 4e of its 16): lane (n, j)
// gets column n of rows 8j .. 8j + 7.  ds_read_b64_tr_b16 works on 16 lanes: lane a + 4e of them names 8
// bytes (4 values of a row), and lane 4a + c receives value c of the lanes a, a + 4, a + 8, a + 12.
__device__ __forceinline__ void read_by_column(uint32_t at, uint32_t part_bytes, uint32_t four_rows_bytes, half8 &hi, half8 &lo) {
    u32x2 r[2][2];
    asm volatile("ds_read_b64_tr_b16 %0, %1" : "=v"(r[0][0]) : "v"(at) : "memory");
    asm volatile("ds_read_b64_tr_b16 %0, %1" : "=v"(r[0][1]) : "v"(at + four_rows_bytes) : "memory");
    asm volatile("ds_read_b64_tr_b16 %0, %1" : "=v"(r[1][0]) : "v"(at + part_bytes) : "memory");
    asm volatile("ds_read_b64_tr_b16 %0, %1" : "=v"(r[1][1]) : "v"(at + part_bytes + four_rows_bytes) : "memory");
    asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(r[0][0]), "+v"(r[0][1]), "+v"(r[1][0]), "+v"(r[1][1])::"memory");
    hi = __builtin_bit_cast(half8, u32x4{r[0][0].x, r[0][0].y, r[0][1].x, r[0][1].y});
    lo = __builtin_bit_cast(half8, u32x4{r[1][0].x, r[1][0].y, r[1][1].x, r[1][1].y});
}

// The conv of four channels c .. c + 3 for the TOKENS tokens from t0 on, in two parts: the inputs are asked for, and
// the outputs made, with the sums in the order of deltanet_conv_rows4_kernel (the results are the same bit for bit).
template <int TOKENS>
struct ConvPiece {
    static_assert(TOKENS >= CONV - 1, "every token that reads the state lies in the first piece");
    float4 taps[CONV], in[CONV - 1 + TOKENS];
    __device__ __forceinline__ void request_taps(const ChunkArgs &a, uint32_t c) {
#pragma unroll
        for (int j = 0; j < CONV; j++) taps[j] = reinterpret_cast<const float4 *>(a.conv_w + size_t(c) * CONV)[j];  // (by channel)
    }
    __device__ __forceinline__ void request_inputs(const ChunkArgs &a, uint32_t c, uint32_t t0) {
#pragma unroll
        for (int i = 0; i < CONV - 1 + TOKENS; i++) {
            const int t = int(t0) + i - (CONV - 1);
            // (a token past the end: unused)
            const float *from = t >= 0 ? a.x : a.conv_state;
            const uint32_t row = t >= 0 ? min(uint32_t(t), a.tokens - 1) : uint32_t(t + CONV - 1);
            in[i] = *reinterpret_cast<const float4 *>(from + size_t(row) * a.channels + c);
        }
    }
    __device__ __forceinline__ float4 output(int i) const {
        float4 sum = make_float4(0, 0, 0, 0);
#pragma unroll
        for (int j = 0; j < CONV; j++) {
            const float4 v = in[i + j];
            const float w[4] = {j == 0 ? taps[0].x : j == 1 ? taps[0].y : j == 2 ? taps[0].z : taps[0].w, j == 0 ? taps[1].x : j == 1 ? taps[1].y : j == 2 ? taps[1].z : taps[1].w,
                                j == 0 ? taps[2].x : j == 1 ? taps[2].y : j == 2 ? taps[2].z : taps[2].w, j == 0 ? taps[3].x : j == 1 ? taps[3].y : j == 2 ? taps[3].z : taps[3].w};
            sum.x += w[0] * v.x, sum.y += w[1] * v.y, sum.z += w[2] * v.z, sum.w += w[3] * v.w;
        }
        return silu4_f(sum);
    }
    // the first block's piece: the chunk's last inputs become the conv's state, which only that piece has read
    __device__ __forceinline__ void keep_state(const ChunkArgs &a, uint32_t c) const {
#pragma unroll
        for (int j = 0; j < CONV - 1; j++)
            *reinterpret_cast<float4 *>(a.conv_state + j * a.channels + c) = *reinterpret_cast<const float4 *>(a.x + size_t(a.tokens - (CONV - 1) + j) * a.channels + c);
    }
};
constexpr int CONV_QK = C / PREP_WAVES, CONV_VALUES = 8;  // tokens of a piece of q and k, and of the values

// CONVOLVE: the conv before the delta rule is part of the launch.  The workgroup of a block makes the q and k of its key
// head, which are nobody else's: a thread four channels' outputs for CONV_QK tokens, stored as the conv's own kernel does
// and in LDS as f32, over the place of the images, from where they go to the threads that normalise them.  The values, which
// nothing in this kernel reads, are made by workgroups of their own behind the blocks' (grid x from the number of blocks on).
template <int G, bool CONVOLVE>
__global__ __launch_bounds__(PREP_THREADS, 4) void deltanet_chunk_prepare_kernel(ChunkArgs a, float *conv_out) {
    using L = PrepLds<G>;
    constexpr int DROW = L::DROW, HROW = L::HROW;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    _Float16 *kh = reinterpret_cast<_Float16 *>(lds), *kl = kh + C * KROW, *qh = kl + C * KROW, *ql = qh + C * KROW;
    auto diag_lds = [&](int hh, int half) { return reinterpret_cast<float *>(lds + hh * L::HEAD_BYTES + half * L::D_BYTES); };
    auto half_img = [&](int hh, int off) { return reinterpret_cast<_Float16 *>(lds + hh * L::HEAD_BYTES + off); };  // hi part; lo: 32 * HROW on
    auto m_lds = [&](int hh) { return reinterpret_cast<_Float16 *>(lds + L::M_OFF + hh * L::M_BYTES); };
    // The running sums of log g are kept in f64: the decay between two tokens is e^(c_t - c_s), the sums reach
    // -100 and beyond inside a block, and an f32 difference of two of them carries the ulp of the sums (1e-5), which
    // is then the relative error of every entry of A and M: three orders above the rest of this path's arithmetic.
    auto cum_lds = [&](int hh) { return reinterpret_cast<double *>(lds + L::GATES + hh * L::GATE_BYTES); };
    auto beta_lds = [&](int hh) { return reinterpret_cast<float *>(lds + L::GATES + hh * L::GATE_BYTES + C * 8); };
    const uint32_t blk = blockIdx.x, group = a.v_heads / a.k_heads;
    const uint32_t h0 = blockIdx.y * G, khd = h0 / group;  // the workgroup's first value head, its key head
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), n = lane & 15, j = lane >> 4;
    const uint32_t key_size = a.k_heads * K_DIM;
    unsigned char *ws_blk = a.ws + size_t(blk) * block_bytes(a.k_heads, a.v_heads);
    unsigned char *ws_k = ws_blk + khd * KHEAD_BYTES;
    auto ws_v = [&](int hh) { return ws_blk + a.k_heads * KHEAD_BYTES + (h0 + hh) * VHEAD_BYTES; };
    const bool writer = h0 % group == 0;  // one workgroup of the key head's keeps the q / k images

    if constexpr (CONVOLVE) {
        const uint32_t nblocks = (a.tokens + C - 1) / C;
        if (blk >= nblocks) {  // the values' conv: four channels a thread, CONV_VALUES tokens
            const uint32_t quads = a.v_heads * a.v_dim / 4, columns = (quads + PREP_THREADS - 1) / PREP_THREADS;
            const uint32_t at = (blk - nblocks) * a.k_heads + blockIdx.y, quad = at % columns * PREP_THREADS + tid, t0 = at / columns * CONV_VALUES;
            if (quad >= quads || t0 >= a.tokens) return;
            const uint32_t cv = 2 * key_size + 4 * quad;
            ConvPiece<CONV_VALUES> values;
            values.request_taps(a, cv);
            values.request_inputs(a, cv, t0);
#pragma unroll
            for (int i = 0; i < CONV_VALUES; i++) {
                const float4 y = values.output(i);
                if (t0 + i < a.tokens) *reinterpret_cast<float4 *>(conv_out + size_t(t0 + i) * a.channels + cv) = y;
            }
            if (t0 == 0) values.keep_state(a, cv);
            return;
        }
    }
    // ---- the gates' inputs of head h0 + gate_head, one of the first G waves: asked for first, and used when the wave has made its
    // q and k: the first wave of a SIMD, which has precedence, then waits for the second ----
    const int gate_head = wave < G ? int(wave) : -1;
    const bool gate_real = blk * C + lane < a.tokens;
    float gate_a = 0.0f, gate_b = 0.0f, gate_log = 0.0f, gate_bias = 0.0f;
    if (gate_head >= 0) {
        const uint32_t tok = min(blk * C + lane, a.tokens - 1), h = h0 + gate_head;
        gate_a = a.a[size_t(tok) * a.v_heads + h], gate_b = a.b[size_t(tok) * a.v_heads + h], gate_log = a.a_log[h], gate_bias = a.dt_bias[h];
    }
    // c_t = sum of log g up to t, beta_t (tokens past the end: g = 1, beta = 0)
    auto gates = [&]() {
        if (gate_head < 0) return;
        asm volatile("" : "+v"(gate_a), "+v"(gate_b), "+v"(gate_log), "+v"(gate_bias));  // (their first use is here: the loads that follow them wait for nothing)
        float g, beta, lg;
        fast_gates(gate_a + gate_bias, __expf(gate_log), gate_b, g, beta, &lg);
        const double c = inclusive_sum(gate_real ? double(lg) : 0.0);
        cum_lds(gate_head)[lane] = c, beta_lds(gate_head)[lane] = gate_real ? beta : 0.0f;
        const double last = __shfl(c, 63, 64);
        float *gam = reinterpret_cast<float *>(ws_v(gate_head) + 4 * T_GL);
        gam[lane] = __expf(float(c)), gam[C + lane] = __expf(float(last - c));
    };

    // ---- the conv (src/cpu/deltanet.rs:69-100) of the workgroup's channels ----
    constexpr int FROW = 2 * K_DIM + 4;  // f32 per token's q | k in LDS
    static_assert(C * FROW * 4 <= 4 * K_IMG, "the f32 q and k lie over the images");
    float *qk_lds = reinterpret_cast<float *>(lds);
    if constexpr (CONVOLVE) {
        const uint32_t t0 = blk * C + CONV_QK * wave;
        const uint32_t cqk = (lane < 32 ? 0 : key_size - K_DIM) + khd * K_DIM + 4 * lane;  // q: lanes 0-31, k: lanes 32-63
        // The taps, which are the same in all waves, go through LDS: channel c's four to piece c / 4 of plane c % 4.
        constexpr int TAP_PLANE = 64 * 16 + 64;
        static_assert(C * FROW * 4 + CONV * TAP_PLANE <= L::GATES, "the taps lie behind the f32 q and k");
        unsigned char *taps_lds = lds + C * FROW * 4;
        float4 tap = make_float4(0, 0, 0, 0);
        if (tid < 2 * K_DIM) tap = reinterpret_cast<const float4 *>(a.conv_w)[(tid < K_DIM ? 0 : key_size - K_DIM) + khd * K_DIM + tid];
        ConvPiece<CONV_QK> qk;
        qk.request_inputs(a, cqk, t0);
        if (tid < 2 * K_DIM) *reinterpret_cast<float4 *>(taps_lds + (tid & 3) * TAP_PLANE + (tid >> 2) * 16) = tap;
        __syncthreads();
#pragma unroll
        for (int j = 0; j < CONV; j++) qk.taps[j] = *reinterpret_cast<const float4 *>(taps_lds + j * TAP_PLANE + lane * 16);
        // (Every token's output, and all of them before the first store: loads and stores count in one order, and a load whose value
        // nobody had taken would be waited for, behind all stores, at the next use of its registers.)
        float4 y[CONV_QK];
#pragma unroll
        for (int i = 0; i < CONV_QK; i++) {
            const float4 made = qk.output(i);
            y[i] = t0 + i < a.tokens ? made : make_float4(0, 0, 0, 0);
            *reinterpret_cast<float4 *>(qk_lds + (CONV_QK * wave + i) * FROW + 4 * lane) = y[i];
        }
#pragma unroll
        for (int i = 0; i < CONV_QK; i++) {
            if (t0 + i < a.tokens) *reinterpret_cast<float4 *>(conv_out + size_t(t0 + i) * a.channels + cqk) = y[i];
        }
        if (t0 == 0) qk.keep_state(a, cqk);
        gates();
        __syncthreads();
    }

    // ---- q and k of the block's tokens, normalised (src/cpu/deltanet.rs:133-146), as hi and lo parts ----
    {
        // thread (token t, part): the 8-value pieces part and part + 8 of the token's q and k, so that the eight threads
        // of a token read 256 bytes in a row with every pair of loads
        const uint32_t t = tid >> 3, part = tid & 7, tok = blk * C + t;
        const bool real = tok < a.tokens;
        float4 qv[4], kv[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t at = 8 * (part + 8 * (i >> 1)) + 4 * (i & 1);
            if constexpr (CONVOLVE) {
                qv[i] = *reinterpret_cast<const float4 *>(qk_lds + t * FROW + at);
                kv[i] = *reinterpret_cast<const float4 *>(qk_lds + t * FROW + K_DIM + at);
            } else {
                const float *row = a.mixed + size_t(min(tok, a.tokens - 1)) * a.channels + khd * K_DIM + at;
                qv[i] = *reinterpret_cast<const float4 *>(row);
                kv[i] = *reinterpret_cast<const float4 *>(row + key_size);
            }
        }
        if constexpr (!CONVOLVE) {
            if ((blk + 1) * C > a.tokens && !real) {
#pragma unroll
                for (int i = 0; i < 4; i++) qv[i] = kv[i] = make_float4(0, 0, 0, 0);
            }
        }
        float qs = 0.0f, ks = 0.0f;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            qs += qv[i].x * qv[i].x + qv[i].y * qv[i].y + qv[i].z * qv[i].z + qv[i].w * qv[i].w;
            ks += kv[i].x * kv[i].x + kv[i].y * kv[i].y + kv[i].z * kv[i].z + kv[i].w * kv[i].w;
        }
        if constexpr (CONVOLVE) __syncthreads();  // the f32 q and k are read: the images go over them
        qs = group_reduce<8>(qs, SumOp());
        ks = group_reduce<8>(ks, SumOp());
        // (q's factor 1 / sqrt(128) is applied to the output: at unit length the lo parts stay clear of the f16 underflow;
        // a token past the end is zeros and stays so, whatever eps is)
        const float qi = real ? __builtin_amdgcn_rsqf(qs + a.eps) : 0.0f, ki = real ? __builtin_amdgcn_rsqf(ks + a.eps) : 0.0f;
#pragma unroll
        for (int i = 0; i < 4; i += 2) {
            half4 h[2][2], l[2][2];  // [q | k][half of the piece]
#pragma unroll
            for (int e = 0; e < 2; e++) {
                const float4 qq = qv[i + e], kk = kv[i + e];
                split4([&](int c) { return (c == 0 ? qq.x : c == 1 ? qq.y : c == 2 ? qq.z : qq.w) * qi; }, h[0][e], l[0][e]);
                split4([&](int c) { return (c == 0 ? kk.x : c == 1 ? kk.y : c == 2 ? kk.z : kk.w) * ki; }, h[1][e], l[1][e]);
            }
            auto joined = [](const half4 (&x)[2]) { return __builtin_shufflevector(x[0], x[1], 0, 1, 2, 3, 4, 5, 6, 7); };
            const half8 a_qh = joined(h[0]), a_ql = joined(l[0]), a_kh = joined(h[1]), a_kl = joined(l[1]);
            const uint32_t piece = part + 4 * i;  // key dims 8 piece ..: k-step piece / 4, lane group piece % 4 of an operand
            const int at = t * KROW + 8 * piece;
            *reinterpret_cast<half8 *>(kh + at) = a_kh, *reinterpret_cast<half8 *>(kl + at) = a_kl;
            *reinterpret_cast<half8 *>(qh + at) = a_qh, *reinterpret_cast<half8 *>(ql + at) = a_ql;
        }
        if constexpr (!CONVOLVE) gates();
    }
    __syncthreads();

    // ---- k . k (first team) and q . k (second): wave tw of a team takes the rows t = 16 tw + .., the tiles of 16 columns s
    // at and below the diagonal, transposed: lane (n, j) holds columns s = 16 nt + 4j + i of row t = 16 tw + n.  The tiles go two
    // by two, the columns of the first 32 tokens and, for the rows of the last 32, those of the last; what of a pair lies above the
    // diagonal is masked.  The two waves of a SIMD, w and w + 4, have six tiles between them: the second team's rows go upwards.
    // The decays e^(c_t - c_s), which wait for no product, are made between them. ----
    const uint32_t team = wave >> 2, tw = team == 0 ? wave & 3 : 3 - (wave & 3), t_row = 16 * tw + n;
    floatx4 prod[4];
    float decay[G][4][4];
    auto products = [&](auto half) {
        constexpr int nt0 = 2 * decltype(half)::value;
        const _Float16 *rh = team == 0 ? kh : qh, *rl = team == 0 ? kl : ql;
        prod[nt0] = prod[nt0 + 1] = floatx4{0, 0, 0, 0};
#pragma unroll
        for (int ks = 0; ks < 4; ks++) {
            const int to = t_row * KROW + 32 * ks + 8 * j;
            const half8 th = *reinterpret_cast<const half8 *>(rh + to), tl = *reinterpret_cast<const half8 *>(rl + to);
            if (nt0 == 0 && writer) {  // the rows' operands are what the chain kernel reads: operand (wave tw, k-step), whole lines a store
                unsigned char *g = ws_k + team * (2 * K_GL) + ((tw * 4 + ks) * 64 + lane) * 16;
                *reinterpret_cast<half8 *>(g) = th, *reinterpret_cast<half8 *>(g + K_GL) = tl;
            }
#pragma unroll
            for (int nt = nt0; nt < nt0 + 2; nt++) {
                const int so = (16 * nt + n) * KROW + 32 * ks + 8 * j;
                prod[nt] = mma3(*reinterpret_cast<const half8 *>(kh + so), *reinterpret_cast<const half8 *>(kl + so), th, tl, prod[nt]);
            }
        }
#pragma unroll
        for (int hh = 0; hh < G; hh++) {
            const double ct = cum_lds(hh)[t_row];
#pragma unroll
            for (int nt = nt0; nt < nt0 + 2; nt++) {
#pragma unroll
                for (int i = 0; i < 4; i++) decay[hh][nt][i] = __expf(float(ct - cum_lds(hh)[16 * nt + 4 * j + i]));
            }
        }
    };
    products(std::integral_constant<int, 0>());
    if (tw >= 2) products(std::integral_constant<int, 1>());
    __syncthreads();  // the images are read: A and M go over them

    // ---- A and M.  What lies above the diagonal inside the 32 x 32 blocks is zero; the block above them is not read by
    // anybody and not written. ----
    auto matrices = [&](auto half) {
        constexpr int nt0 = 2 * decltype(half)::value;
        const bool diagonal = team == 0 && (nt0 == 2 || tw < 2);  // a diagonal 32 x 32 block of A
        const uint32_t end = t_row + team;  // A has s < t, M s <= t
#pragma unroll
        for (int hh = 0; hh < G; hh++) {
            const float beta_t = team == 0 ? beta_lds(hh)[t_row] : 1.0f;
            float x[2][4];
#pragma unroll
            for (int e = 0; e < 2; e++) {
#pragma unroll
                for (int i = 0; i < 4; i++) x[e][i] = 16 * (nt0 + e) + 4 * j + i < end ? beta_t * (decay[hh][nt0 + e][i] * prod[nt0 + e][i]) : 0.0f;
            }
            if (diagonal) {
                float *dst = diag_lds(hh, nt0 / 2) + (t_row & 31) * DROW + 4 * j;
                *reinterpret_cast<floatx4 *>(dst) = floatx4{x[0][0], x[0][1], x[0][2], x[0][3]};
                *reinterpret_cast<floatx4 *>(dst + 16) = floatx4{x[1][0], x[1][1], x[1][2], x[1][3]};
            } else {  // M | the block of A below the diagonal, as an MFMA operand
                _Float16 *dst = team == 0 ? half_img(hh, L::LBA_OFF) + (t_row - 32) * HROW : m_lds(hh) + t_row * TROW;
                const int lo_part = team == 0 ? 32 * HROW : C * TROW;
#pragma unroll
                for (int e = 0; e < 2; e++) {
                    half4 hi, lo;
                    split4([&](int i) { return x[e][i]; }, hi, lo);
                    *reinterpret_cast<half4 *>(dst + 16 * (nt0 + e) + 4 * j) = hi;
                    *reinterpret_cast<half4 *>(dst + 16 * (nt0 + e) + 4 * j + lo_part) = lo;
                }
            }
        }
    };
    matrices(std::integral_constant<int, 0>());
    if (tw >= 2) matrices(std::integral_constant<int, 1>());
    __syncthreads();
    // A staged matrix leaves in operand order, 16 bytes per piece, by `threads` threads: piece (part hi | lo, operand, lane
    // (n, j)) is row 16 w + n, columns 32 ks + 8j .. of the part's image; the operands are (w, ks) = (0, 0), (1, 0), (2, 0),
    // (2, 1), (3, 0), (3, 1): nobody reads the other two.
    auto leave = [&](int hh, unsigned char *dst, uint32_t thread, uint32_t threads) {
        for (uint32_t i = thread; i < 2 * 6 * 64; i += threads) {
            const uint32_t part = i >= 6 * 64 ? 1 : 0, op = (i >> 6) - 6 * part, w = op < 2 ? op : op < 4 ? 2 : 3, ks = op < 2 ? 0 : op & 1, nn = i & 15, jj = (i >> 4) & 3;
            reinterpret_cast<u32x4 *>(dst)[part * (T_GL / 16) + (w * 2 + ks) * 64 + (i & 63)] =
                *reinterpret_cast<const u32x4 *>(m_lds(hh) + part * C * TROW + (16 * w + nn) * TROW + 32 * ks + 8 * jj);
        }
    };

    // ---- T = (I + A)^-1 diag(beta), in 32 x 32 blocks: with L = I + A = [[L_AA, 0], [L_BA, L_BB]],
    //     T_AA = L_AA^-1 diag(beta_A),  T_BB = L_BB^-1 diag(beta_B),  T_BA = -L_BB^-1 (L_BA T_AA).
    // A diagonal block's inverse goes over it, one wave per head, in the same way from 16 x 16 blocks: lane (column c = n, block j)
    // solves x_t = [t = c] - sum_{s < t} A_ts x_s of its block, and the block below is two f32 products on the matrix cores.  The
    // second team stores M meanwhile.  Then T_BA: two products in hi and lo parts. ----
    if (wave < G) {
        float *ad = diag_lds(wave, j >> 1) + (j & 1) * (16 * DROW + 16);
        float x[16];
        floatx4 av[2][4];  // a row and the next: no row waits for its own reads
#pragma unroll
        for (int t = 0; t < 16; t++) {
#pragma unroll
            for (int s4 = 0; t < 15 && 4 * s4 <= t; s4++) av[(t + 1) & 1][s4] = *reinterpret_cast<const floatx4 *>(ad + (t + 1) * DROW + 4 * s4);
            __builtin_amdgcn_sched_barrier(0);
            floatx4 part4 = {0, 0, 0, 0};  // (four chains of sums instead of one of up to 15)
#pragma unroll
            for (int s4 = 0; 4 * s4 < t; s4++) {
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    if (4 * s4 + e < t) part4[e] += av[t & 1][s4][e] * x[4 * s4 + e];
                }
            }
            x[t] = (uint32_t(t) == n ? 1.0f : 0.0f) - ((part4[0] + part4[1]) + (part4[2] + part4[3]));
        }
#pragma unroll
        for (int t = 0; t < 16; t++) ad[t * DROW + n] = x[t];  // (behind the loop: in it, the next row's reads would wait for x_t)
        // the block below them, for both halves: k index 4j + i in step i, so that the first product's result is the second's operand
        floatx4 w[2], y[2];
#pragma unroll
        for (int half = 0; half < 2; half++) {
            const float *d = diag_lds(wave, half);
            const floatx4 below = *reinterpret_cast<const floatx4 *>(d + (16 + n) * DROW + 4 * j);
            w[half] = floatx4{0, 0, 0, 0};
#pragma unroll
            for (int i = 0; i < 4; i++) w[half] = __builtin_amdgcn_mfma_f32_16x16x4f32(below[i], d[(4 * j + i) * DROW + n], w[half], 0, 0, 0);
        }
#pragma unroll
        for (int half = 0; half < 2; half++) {
            const floatx4 second = *reinterpret_cast<const floatx4 *>(diag_lds(wave, half) + (16 + n) * DROW + 16 + 4 * j);
            y[half] = floatx4{0, 0, 0, 0};
#pragma unroll
            for (int i = 0; i < 4; i++) y[half] = __builtin_amdgcn_mfma_f32_16x16x4f32(second[i], w[half][i], y[half], 0, 0, 0);
        }
#pragma unroll
        for (int half = 0; half < 2; half++) {
#pragma unroll
            for (int i = 0; i < 4; i++) diag_lds(wave, half)[(16 + 4 * j + i) * DROW + n] = -y[half][i];
        }
    } else if (team == 1) {
#pragma unroll
        for (int hh = 0; hh < G; hh++) leave(hh, ws_v(hh) + 2 * T_GL, tid - 256, 256);
    }
    __syncthreads();  // M has left: T goes over it
    for (uint32_t i = tid; i < G * 2 * 32 * 8; i += PREP_THREADS) {
        // four columns c .. of row t of a diagonal block
        const uint32_t c = (i & 7) * 4, t = (i >> 3) & 31, half = (i >> 8) & 1, hh = G == 2 ? i >> 9 : 0;
        const floatx4 x = *reinterpret_cast<const floatx4 *>(diag_lds(hh, half) + t * DROW + c);
        const floatx4 beta = *reinterpret_cast<const floatx4 *>(beta_lds(hh) + 32 * half + c);
        half4 th, tl, xh, xl;
        split4([&](int e) { return x[e] * beta[e]; }, th, tl);
        split4([&](int e) { return x[e]; }, xh, xl);
        _Float16 *dst = m_lds(hh) + (32 * half + t) * TROW + 32 * half + c;
        *reinterpret_cast<half4 *>(dst) = th, *reinterpret_cast<half4 *>(dst + C * TROW) = tl;
        if (half) {
            _Float16 *xd = half_img(hh, L::XBB_OFF) + t * HROW + c;
            *reinterpret_cast<half4 *>(xd) = xh, *reinterpret_cast<half4 *>(xd + 32 * HROW) = xl;
        }
    }
    __syncthreads();
    {
        // W = L_BA T_AA and then T_BA = -L_BB^-1 W: a wave takes one 16 x 16 tile (rows 16 r, columns 16 ct) of its head,
        // as its transpose.  The right operands are read by column out of row-major images.
        const uint32_t hs = wave >> 2, r = (wave >> 1) & 1, ct = wave & 1, la = lane & 3, le = (lane >> 2) & 3;
        const bool takes = hs < G;
        const uint32_t lds0 = uint32_t(reinterpret_cast<uintptr_t>(lds));
        const int ao = (16 * r + n) * HROW + 8 * j, at = (16 * r + n) * HROW + 16 * ct + 4 * j;
        if (takes) {
            half8 bh, bl;
            read_by_column(lds0 + L::M_OFF + hs * L::M_BYTES + ((8 * j + le) * TROW + 16 * ct + 4 * la) * 2, C * TROW * 2, 4 * TROW * 2, bh, bl);
            const floatx4 w = mma3(bh, bl, *reinterpret_cast<const half8 *>(half_img(hs, L::LBA_OFF) + ao),
                                   *reinterpret_cast<const half8 *>(half_img(hs, L::LBA_OFF) + 32 * HROW + ao), floatx4{0, 0, 0, 0});
            // (the inverses of the diagonal blocks were last read before the barrier above)
            half4 wh, wl;
            split4([&](int i) { return w[i]; }, wh, wl);
            *reinterpret_cast<half4 *>(half_img(hs, L::W_OFF) + at) = wh, *reinterpret_cast<half4 *>(half_img(hs, L::W_OFF) + 32 * HROW + at) = wl;
        }
        __syncthreads();
        if (takes) {
            half8 bh, bl;
            read_by_column(lds0 + hs * L::HEAD_BYTES + L::W_OFF + ((8 * j + le) * HROW + 16 * ct + 4 * la) * 2, 32 * HROW * 2, 4 * HROW * 2, bh, bl);
            const floatx4 tba = mma3(bh, bl, *reinterpret_cast<const half8 *>(half_img(hs, L::XBB_OFF) + ao),
                                     *reinterpret_cast<const half8 *>(half_img(hs, L::XBB_OFF) + 32 * HROW + ao), floatx4{0, 0, 0, 0});
            half4 th, tl;
            split4([&](int i) { return -tba[i]; }, th, tl);
            _Float16 *dst = m_lds(hs) + (32 + 16 * r + n) * TROW + 16 * ct + 4 * j;
            *reinterpret_cast<half4 *>(dst) = th, *reinterpret_cast<half4 *>(dst + C * TROW) = tl;
        }
    }
    __syncthreads();
#pragma unroll
    for (int hh = 0; hh < G; hh++) leave(hh, ws_v(hh), tid, PREP_THREADS);
}

// ds_read_b64_tr_b16 of the 8 bytes at `at` in LDS
__device__ __forceinline__ half4 read_transposed(const unsigned char *at) {
    typedef __fp16 fp16x4 __attribute__((ext_vector_type(4)));
    return __builtin_bit_cast(half4, __builtin_amdgcn_ds_read_tr16_b64_v4f16((__attribute__((address_space(3))) fp16x4 *)(at)));
}

// ---- the chain over the blocks --------------------------------------------------------------------
// Per block, with S0 [dv][128] the state's slice: P = K S0^T and Q S0^T (rows: tokens); R = V - e^c P;
// U = T R; O = (e^c (Q S0^T) + M U) / sqrt(128); S1 = e^{c_last} S0 + (e^{c_last - c} U)^T K.
// A wave takes 16 tokens' rows of K, Q, T and M, and nobody else reads those: they come from the workspace
// straight into its registers, two blocks ahead, as the MFMA operands they are.  LDS holds what the
// waves hand to each other: the state's image, R, U and the scaled U, the block's values and decay
// factors, and the block's keys, which the state's update contracts over the tokens: every wave puts
// its rows there, and ds_read_b64_tr_b16 hands them out by key dim.
// What bounds it: a block is three phases between barriers, each a trip through LDS, a few dependent products and a trip back,
// and 92 KB of operands through the CU's 64 bytes a cycle, 1500 cycles of loads that a wave stands still at when they come all at
// once.  A block took 4050 cycles, a state wave 450 of them at its eight loads behind K S0^T and 580 waiting for the output waves, who
// stood at theirs.  So each team works where the other leaves LDS and the memory pipe alone: the outputs' M U and
// stores under the next block's K S0^T, their Q S0^T under U, their loads under the state's update; the state's
// loads two at a time between its dependent products.  (The output waves' loads under U: 246 us instead of 230.)
// Measured, whole chunk, us: 1000 tokens 65.4 -> 61.2, 2300 140.3 -> 128.7, 4096 253.3 -> 230.4 (this kernel 132 -> 109,
// with the outputs in whole lines); results bit for bit the same.
struct ChainLds {
    static constexpr int GAM = 0;                          // e^{c_t}, e^{c_last - c_t}: 128 f32
    static constexpr int V = GAM + 2 * C * 4;              // [token][DV] f32
    static constexpr int SROW = K_DIM + 8;                 // f16 per row of the state's operand image [dv][128]
    static constexpr int SH = V + C * DV * 4, SL = SH + DV * SROW * 2;
    static constexpr int RH = SL + DV * SROW * 2;          // [dv][64 tokens] images, rows of TROW f16: R, U, U scaled
    static constexpr int RL = RH + DV * TROW * 2, UH = RL + DV * TROW * 2, UL = UH + DV * TROW * 2;
    static constexpr int WH = UL + DV * TROW * 2, WL = WH + DV * TROW * 2;
    // the block's keys [token][128] as hi and lo images: every wave puts its 16 rows there, and the state's update reads
    // them by key dim (transposing reads).  Piece p (8 key dims) of token t lies at place p ^ key_piece(t) of the token's 256
    // bytes: 16 rows' pieces fall on all banks, and so do what half a wave reads, four tokens in a row and four 8 further.
    static constexpr int KIMG = (WL + DV * TROW * 2 + 15) / 16 * 16, K_BYTES = C * K_DIM * 2;
    static __device__ __forceinline__ uint32_t key_piece(uint32_t t) { return (t & 3) << 1 | (t & 8) | (t >> 2 & 1); }
    static constexpr int BYTES = KIMG + 2 * K_BYTES;
};

// Eight waves in two teams.  Waves 0-3 carry the state: K S0^T, R, U and the state's update, each for 16 of
// the block's tokens (the update: for 32 key dims).  Waves 4-7 make the outputs, which nothing in the chain
// waits for: Q S0^T beside the first team's U, M U and the stores beside its K S0^T of the next block.
// What a wave reads of a block: its 16 rows of K (or Q) and of T (or M), 12 operands at most, and, in the
// first team, its share of the block's values and factors.
struct ChainBlock {
    u32x4 kq[2][4];  // [hi | lo][k-step]: rows 16 w + n of K | Q
    u32x4 tm[2][2];  // [hi | lo][k-step]: rows 16 w + n of T | M
    static constexpr int V_LOADS = C * DV * 4 / 16 / 256;  // 16-byte pieces per thread of the block's [token][DV] values
    u32x4 v[V_LOADS], gam;   // ...; 16 bytes of the 128 factors (threads 0-31)
    uint32_t touched[2];     // AHEAD: what `touch` has loaded
};

// AHEAD: the operands of the block AHEAD_BLOCKS on are brought into the L2 by the workgroups that share them, each a piece
// (`touch`).  What the conv and the prepare kernel have just written is served from the memory's cache (256 MB) while it fits, fast
// enough for loads two blocks ahead, and the pieces are an eighth more traffic: whole chunk, us, without -> with: 1000 tokens 61.2
// -> 62.8, 2300 128.9 -> 133.5, 3200 180.6 -> 182.0; past it the first of a line's readers waits for memory: 3500 205.1 -> 199.9, 4096
// 248.0 -> 230.5 (6 blocks ahead 232.3, without the values' lines 238.7).  With the rest as it is now: 2300 123.8 -> 127.0, 3000 159.3 ->
// 160.9, 3150 171.7 -> 171.7, 3250 177.7 -> 176.3.
constexpr uint32_t AHEAD_BLOCKS = 3;
constexpr size_t AHEAD_FROM = size_t(208) << 20;  // bytes of `mixed` and the workspace: 3300 tokens of the model's shape
template <bool AHEAD>
__global__ __launch_bounds__(512) void deltanet_chunk_chain_kernel(ChunkArgs a) {
    using L = ChainLds;
    constexpr int NT = DV / 16;  // 16-wide tiles of value dims
    constexpr int V_LOADS = ChainBlock::V_LOADS;
    static_assert(V_LOADS >= 1 && V_LOADS * 256 * 16 == C * DV * 4, "whole 16-byte pieces of the block's values per thread");
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    // Workgroups go to the 8 XCDs in turn, and each XCD has its own L2: workgroup w of the launch runs on
    // XCD w % 8.  The slices of a value head, and the value heads of a key head, read the same operands, so
    // they are given to one XCD (v_heads / 8 value heads each, where that divides).
    const uint32_t slices = a.v_dim / DV;
    uint32_t slice = blockIdx.x % slices, h = blockIdx.x / slices;
    if (a.v_heads % 8 == 0) {
        const uint32_t xcd = blockIdx.x % 8, at = blockIdx.x / 8;  // at: the XCD's workgroups in order
        h = xcd * (a.v_heads / 8) + at / slices, slice = at % slices;
    }
    const uint32_t group = a.v_heads / a.k_heads, khd = h / group;
    const uint32_t lane = threadIdx.x & 63, wave_all = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), n = lane & 15, j = lane >> 4;
    const bool state_team = wave_all < 4;
    const uint32_t wave = wave_all & 3, tid = threadIdx.x & 255;  // the wave and the thread inside the team
    const uint32_t nblocks = (a.tokens + C - 1) / C;
    const size_t per_block = block_bytes(a.k_heads, a.v_heads);
    auto img = [&](int off) { return reinterpret_cast<const _Float16 *>(lds + off); };
    auto img_w = [&](int off) { return reinterpret_cast<_Float16 *>(lds + off); };
    const float *gam = reinterpret_cast<const float *>(lds + L::GAM);
    float *v_lds = reinterpret_cast<float *>(lds + L::V);

    // A block's operands are asked for in three lots, each when the registers it goes to have been read
    // for the block two before: the rows of K | Q, the rows of T | M, the block's values and factors.
    auto clamp_block = [&](uint32_t blk) { return blk < nblocks ? blk : nblocks - 1; };  // (past the last block: its operands again, unused)
    // (the second team's operands lie two parts on: Q behind K, M behind T)
    auto rows_of = [&](uint32_t at) {
        return reinterpret_cast<const u32x4 *>(a.ws + size_t(clamp_block(at)) * per_block + khd * KHEAD_BYTES + (state_team ? 0 : 2 * K_GL)) + wave * 4 * 64 + lane;
    };
    auto request_kq_step = [&](const u32x4 *wk, int ks, ChainBlock &b) {
#pragma unroll
        for (int part = 0; part < 2; part++) b.kq[part][ks] = wk[(part * K_GL) / 16 + ks * 64];
    };
    auto request_kq = [&](uint32_t at, ChainBlock &b) {
        const u32x4 *wk = rows_of(at);
#pragma unroll
        for (int ks = 0; ks < 4; ks++) request_kq_step(wk, ks, b);
    };
    auto request_tm = [&](uint32_t at, ChainBlock &b) {
        const uint32_t blk = clamp_block(at);
        const u32x4 *wv = reinterpret_cast<const u32x4 *>(a.ws + size_t(blk) * per_block + a.k_heads * KHEAD_BYTES + h * VHEAD_BYTES);
        const u32x4 *wt = wv + (state_team ? 0 : 2 * T_GL) / 16;
#pragma unroll
        for (int part = 0; part < 2; part++) {
#pragma unroll
            for (int ks = 0; ks < 2; ks++) {
                // (T and M are lower triangular: rows 16 wave .. have nothing in columns 32 ks .. beyond their own)
                if (ks <= int(wave) / 2) b.tm[part][ks] = wt[(part * T_GL) / 16 + (wave * 2 + ks) * 64 + lane];
            }
        }
    };
    auto request_values = [&](uint32_t at, ChainBlock &b) {  // (the first team)
        const uint32_t blk = clamp_block(at);
        const u32x4 *wv = reinterpret_cast<const u32x4 *>(a.ws + size_t(blk) * per_block + a.k_heads * KHEAD_BYTES + h * VHEAD_BYTES);
#pragma unroll
        for (int i = 0; i < V_LOADS; i++) {
            // piece p of the block's [token][DV] values: token p / (DV / 4), four dims (a token past the end: unused, see `place`)
            const uint32_t p = tid + 256 * i, tok = min(blk * C + p / (DV / 4), a.tokens - 1);
            b.v[i] = *reinterpret_cast<const u32x4 *>(a.mixed + size_t(tok) * a.channels + 2 * a.k_heads * K_DIM + h * a.v_dim + DV * slice + 4 * (p % (DV / 4)));
        }
        b.gam = wv[(4 * T_GL) / 16 + (tid & 31)];
    };
    // the block's values (tokens past the end: zeros) and factors to LDS (the first team)
    auto place = [&](uint32_t blk, const ChainBlock &b) {
#pragma unroll
        for (int i = 0; i < V_LOADS; i++) {
            const uint32_t p = tid + 256 * i;
            const bool real = blk * C + p / (DV / 4) < a.tokens;
            reinterpret_cast<u32x4 *>(v_lds)[p] = real ? b.v[i] : u32x4{0, 0, 0, 0};
        }
        if (tid < 32) reinterpret_cast<u32x4 *>(lds + L::GAM)[tid] = b.gam;
    };

    // ---- the state's slice: S [dv][128]; wave w of the first team keeps columns 32 w .. + 31: lane (n, j) the four
    // columns 32 w + 16 nt + 4j + i of row dv = 16 mt + n.  Its image for the products lies in LDS as hi and lo parts. ----
    float *state = a.state + (size_t(h) * a.v_dim + DV * slice) * K_DIM;
    floatx4 s_reg[NT][2];
    auto publish_state = [&]() {
#pragma unroll
        for (int mt = 0; mt < NT; mt++) {
#pragma unroll
            for (int nt = 0; nt < 2; nt++) {
                half4 sh, sl;
                split4([&](int i) { return s_reg[mt][nt][i]; }, sh, sl);
                const int at = (16 * mt + n) * L::SROW + 32 * wave + 16 * nt + 4 * j;
                *reinterpret_cast<half4 *>(img_w(L::SH) + at) = sh, *reinterpret_cast<half4 *>(img_w(L::SL) + at) = sl;
            }
        }
    };
#pragma unroll
    for (int mt = 0; mt < NT; mt++) {
#pragma unroll
        for (int nt = 0; nt < 2; nt++) {
            s_reg[mt][nt] = state_team ? *reinterpret_cast<const floatx4 *>(state + (16 * mt + n) * K_DIM + 32 * wave + 16 * nt + 4 * j) : floatx4{0, 0, 0, 0};
        }
    }

    // One block: `cur` holds its operands, `next` those of the block after it (asked for during the block before
    // this one).  Each lot of `cur`, once read, is asked for again for the block after next: a load has two
    // blocks' time to come back (one block's time is less than the 2.9 us a wave's batch takes under this load).
    // (the team is a type, so that a team's blocks are one piece of code: what one team asks for is not taken to be
    // in flight where the other team waits)
    // AHEAD: the lines of a block's operands that this workgroup brings into its XCD's L2 for all that read them: a sixteenth of
    // the key head's rows (an eighth per value head), an eighth of T and M, and of the values, whose lines two slices share,
    // half of its own.  One load names a line every four (values: eight) lanes.
    auto touch = [&](uint32_t at, ChainBlock &b) {
        asm volatile("" ::"v"(b.touched[0]), "v"(b.touched[1]));  // (two blocks old: there)
        const uint32_t blk = clamp_block(at), line = (wave & 1) * 16 + (lane >> 2);
        const unsigned char *base = a.ws + size_t(blk) * per_block;
        const unsigned char *rows = base + khd * KHEAD_BYTES + (((h % group) * slices + slice) * 32 + line) * 128 % KHEAD_BYTES;
        const unsigned char *tm = base + a.k_heads * KHEAD_BYTES + h * VHEAD_BYTES + (slice * 32 + line) * 128 % (4 * T_GL);
        b.touched[0] = *reinterpret_cast<const uint32_t *>(wave < 2 ? rows : tm);
        const uint32_t tok = min(blk * C + (slice & 1) * 32 + wave * 8 + (lane >> 3), a.tokens - 1);
        b.touched[1] = *reinterpret_cast<const uint32_t *>(a.mixed + size_t(tok) * a.channels + 2 * a.k_heads * K_DIM + h * a.v_dim + DV * slice);
    };
    // ---- O = (e^c (Q S0^T) + M U) / sqrt(128) of block `blk`, whose Q S0^T and e^c the second team's waves hold ----
    floatx4 held[NT];
    float held_gam = 0.0f;
#pragma unroll
    for (int vt = 0; vt < NT; vt++) held[vt] = floatx4{0, 0, 0, 0};
    auto outputs = [&](uint32_t blk, bool real, ChainBlock &b) {
        floatx4 mu[NT];
#pragma unroll
        for (int vt = 0; vt < NT; vt++) {
            mu[vt] = floatx4{0, 0, 0, 0};
#pragma unroll
            for (int ks = 0; ks < 2; ks++) {
                if (ks > int(wave) / 2) continue;
                const int bo = (16 * vt + n) * TROW + 32 * ks + 8 * j;
                mu[vt] = mma3(*reinterpret_cast<const half8 *>(img(L::UH) + bo), *reinterpret_cast<const half8 *>(img(L::UL) + bo),
                              __builtin_bit_cast(half8, b.tm[0][ks]), __builtin_bit_cast(half8, b.tm[1][ks]), mu[vt]);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        request_tm(blk + 2, b);
        __builtin_amdgcn_sched_barrier(0);
        // AHEAD: lane 4t + p takes piece p of token t's 64 bytes, so that four lanes store them in a row (a store of 64 lanes that
        // are apart takes the memory pipe 64 cycles and not 16, and leaves in more pieces: 4096 tokens 224.2 -> 220.6 us, 3500 192.7 ->
        // 190.3; where the memory's cache takes the stores it gives nothing, 2300 121.2 -> 121.3, 130 25.5 -> 25.6)
        const uint32_t row = AHEAD ? lane >> 2 : n, piece = AHEAD ? lane & 3 : j, tok = blk * C + 16 * wave + row;
        floatx4 out[NT];
#pragma unroll
        for (int vt = 0; vt < NT; vt++) {
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float x = Q_SCALE * (held_gam * held[vt][i] + mu[vt][i]);
                out[vt][i] = AHEAD ? __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(int(4 * (16 * piece + row)), __builtin_bit_cast(int, x))) : x;
            }
        }
        if (real && tok < a.tokens) {
            float *o = a.o + (size_t(tok) * a.v_heads + h) * a.v_dim + DV * slice + 4 * piece;
#pragma unroll
            for (int vt = 0; vt < NT; vt++) *reinterpret_cast<floatx4 *>(o + 16 * vt) = out[vt];
        }
    };

    auto step = [&](auto team, uint32_t blk, ChainBlock &cur, ChainBlock &next) {
        constexpr bool STATE = decltype(team)::value;
        const uint32_t nxt = blk + 1 < nblocks ? blk + 1 : blk;
        if constexpr (STATE) request_values(blk + 2, cur);  // (this block's values went to LDS during the block before)
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();  // the block's values and factors and the state's image are in LDS

        // K S0^T (first team): rows t = 16 wave + n, columns dv = 16 vt + n' | (Q S0^T)^T (second team): the other way round,
        // so that a lane's results are four value dims of a token, one 16-byte store.  As a k-step's rows have been read, the first
        // team puts them into LDS (the image was last read two barriers ago) and asks for the block after next's.
        floatx4 pkq[NT];
        const u32x4 *const wk = rows_of(blk + 2);
        auto by_state = [&]() {
            half8 image[4][NT][2];
#pragma unroll
            for (int ks = 0; ks < 4; ks++) {
#pragma unroll
                for (int vt = 0; vt < NT; vt++) {
                    const int bo = (16 * vt + n) * L::SROW + 32 * ks + 8 * j;
                    image[ks][vt][0] = *reinterpret_cast<const half8 *>(img(L::SH) + bo), image[ks][vt][1] = *reinterpret_cast<const half8 *>(img(L::SL) + bo);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int ks = 0; ks < 4; ks++) {
#pragma unroll
                for (int vt = 0; vt < NT; vt++) {
                    const half8 bh = image[ks][vt][0], bl = image[ks][vt][1];
                    const half8 ah = __builtin_bit_cast(half8, cur.kq[0][ks]), al = __builtin_bit_cast(half8, cur.kq[1][ks]);
                    pkq[vt] = STATE ? mma3(ah, al, bh, bl, pkq[vt]) : mma3(bh, bl, ah, al, pkq[vt]);
                }
                if constexpr (STATE) {
#pragma unroll
                    for (int part = 0; part < 2; part++)
                        *reinterpret_cast<u32x4 *>(lds + L::KIMG + part * L::K_BYTES + (16 * wave + n) * 256 + ((4 * ks + j) ^ L::key_piece(n)) * 16) = cur.kq[part][ks];
                    __builtin_amdgcn_sched_barrier(0);
                    request_kq_step(wk, ks, cur);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        };
#pragma unroll
        for (int vt = 0; vt < NT; vt++) pkq[vt] = floatx4{0, 0, 0, 0};
        // C layout: lane (n, j) holds dv = 16 vt + n of tokens t = 16 wave + 4j + i (second team: dv = 16 vt + 4j + i of
        // token 16 wave + n)
        floatx4 gk4 = {0, 0, 0, 0};
        float glast = 0.0f;
        if constexpr (STATE) {
            const floatx4 gam4 = *reinterpret_cast<const floatx4 *>(gam + 16 * wave + 4 * j);
            gk4 = *reinterpret_cast<const floatx4 *>(gam + C + 16 * wave + 4 * j);
            glast = gam[C - 1];
            float v4[NT][4];
#pragma unroll
            for (int vt = 0; vt < NT; vt++)
#pragma unroll
                for (int i = 0; i < 4; i++) v4[vt][i] = v_lds[(16 * wave + 4 * j + i) * DV + 16 * vt + n];
            by_state();
#pragma unroll
            for (int vt = 0; vt < NT; vt++) {
                // R = V - e^c (K S0^T), as the [dv][token] image
                half4 rh, rl;
                split4([&](int i) { return v4[vt][i] - gam4[i] * pkq[vt][i]; }, rh, rl);
                const int at = (16 * vt + n) * TROW + 16 * wave + 4 * j;
                *reinterpret_cast<half4 *>(img_w(L::RH) + at) = rh, *reinterpret_cast<half4 *>(img_w(L::RL) + at) = rl;
            }
        }
        if constexpr (!STATE) {
            outputs(blk - 1, blk > 0, next);
            if constexpr (AHEAD) touch(blk + AHEAD_BLOCKS, cur);
        }
        __syncthreads();  // R and the block's keys are whole
        // The left operands of the state's update, K by key dim: lane (n, j) wants key dim 32 wave + 16 nt + n, tokens
        // 32 ks + 8j .. + 7.  The transposing read works on 16 lanes: lane a + 4e of them names 8 bytes (4 values of a row),
        // and lane 4a + c receives value c of the lanes a, a + 4, a + 8, a + 12.  So lane a + 4e names token .. + e, key
        // dims .. + 4a .. + 3, and lane n = 4a + c receives key dim .. + n of four tokens in a row; two reads an operand.
        // They are asked for behind R, a barrier before their use.
        half4 xr[2][2][2][2];  // [hi | lo][nt][k-step][tokens + 0 | + 4]
        auto read_keys = [&]() {
            const uint32_t la = lane & 3, le = (lane >> 2) & 3, x = (4 * wave + (la >> 1)) ^ L::key_piece(8 * (j & 1) + le);
            const unsigned char *kbase = lds + L::KIMG + (8 * j + le) * 256 + (la & 1) * 8;
#pragma unroll
            for (int part = 0; part < 2; part++) {
#pragma unroll
                for (int nt = 0; nt < 2; nt++) {
#pragma unroll
                    for (int ks = 0; ks < 2; ks++) {
#pragma unroll
                        for (int hf = 0; hf < 2; hf++) {
                            xr[part][nt][ks][hf] = read_transposed(kbase + part * L::K_BYTES + (32 * ks + 4 * hf) * 256 + (x ^ (2 * nt + hf)) * 16);
                        }
                    }
                }
            }
        };

        if constexpr (STATE) {
            // ---- U = T R (T is lower triangular: k-steps up to the row tile's own) ----
#pragma unroll
            for (int vt = 0; vt < NT; vt++) {
                floatx4 u = {0, 0, 0, 0};
                half8 r[2][2];  // [k-step][hi | lo]
#pragma unroll
                for (int ks = 0; ks < 2; ks++) {
                    if (ks > int(wave) / 2) continue;
                    const int bo = (16 * vt + n) * TROW + 32 * ks + 8 * j;
                    r[ks][0] = *reinterpret_cast<const half8 *>(img(L::RH) + bo), r[ks][1] = *reinterpret_cast<const half8 *>(img(L::RL) + bo);
                }
                if (vt == 0) {
                    __builtin_amdgcn_sched_barrier(0);
                    read_keys();
                    __builtin_amdgcn_sched_barrier(0);
                }
#pragma unroll
                for (int ks = 0; ks < 2; ks++) {
                    if (ks > int(wave) / 2) continue;
                    u = mma3(__builtin_bit_cast(half8, cur.tm[0][ks]), __builtin_bit_cast(half8, cur.tm[1][ks]), r[ks][0], r[ks][1], u);
                }
                half4 uh, ul, wh, wl;
                split4([&](int i) { return u[i]; }, uh, ul);
                split4([&](int i) { return u[i] * gk4[i]; }, wh, wl);  // scaled by e^{c_last - c_t} for the state
                const int at = (16 * vt + n) * TROW + 16 * wave + 4 * j;
                *reinterpret_cast<half4 *>(img_w(L::UH) + at) = uh, *reinterpret_cast<half4 *>(img_w(L::UL) + at) = ul;
                *reinterpret_cast<half4 *>(img_w(L::WH) + at) = wh, *reinterpret_cast<half4 *>(img_w(L::WL) + at) = wl;
            }
            __builtin_amdgcn_sched_barrier(0);
            request_tm(blk + 2, cur);
            __builtin_amdgcn_sched_barrier(0);
        } else {
            // (here, where the first team does not want the LDS that both teams' reads of the state's image would share)
            by_state();
            held_gam = gam[16 * wave + n];
#pragma unroll
            for (int vt = 0; vt < NT; vt++) held[vt] = pkq[vt];
        }
        __syncthreads();  // U is whole; every wave is through with the state's image, the values and the factors

        if constexpr (STATE) {
            // ---- S1 = e^{c_last} S0 + (U scaled)^T K, over the 64 tokens, taken as its transpose: rows are the key dims
            // 32 wave + 16 nt + .., columns dv, so that a lane's four results are four columns of a row of S in a row ----
            auto x_operand = [&](int part, int nt, int ks) {
                return __builtin_shufflevector(xr[part][nt][ks][0], xr[part][nt][ks][1], 0, 1, 2, 3, 4, 5, 6, 7);
            };
#pragma unroll
            for (int nt = 0; nt < 2; nt++) {
                floatx4 acc[NT];
#pragma unroll
                for (int mt = 0; mt < NT; mt++) acc[mt] = floatx4{0, 0, 0, 0};
#pragma unroll
                for (int ks = 0; ks < 2; ks++) {
#pragma unroll
                    for (int mt = 0; mt < NT; mt++) {
                        const int ao = (16 * mt + n) * TROW + 32 * ks + 8 * j;
                        acc[mt] = mma3(x_operand(0, nt, ks), x_operand(1, nt, ks), *reinterpret_cast<const half8 *>(img(L::WH) + ao),
                                       *reinterpret_cast<const half8 *>(img(L::WL) + ao), acc[mt]);
                    }
                }
#pragma unroll
                for (int mt = 0; mt < NT; mt++) s_reg[mt][nt] = s_reg[mt][nt] * glast + acc[mt];
            }
            // the next block's state image, values and factors: their places were last read before the barrier above
            publish_state();
            place(nxt, next);
        } else {
            request_kq(blk + 2, cur);
        }
    };
    // (two sets of operand registers that change roles, so that nothing is copied from one to the other)
    auto walk = [&](auto team) {
        constexpr bool STATE = decltype(team)::value;
        ChainBlock even, odd;
        even.touched[0] = even.touched[1] = odd.touched[0] = odd.touched[1] = 0;
        // (in the order the blocks ask in, so that the first blocks' waits are those of every block)
        if constexpr (STATE) request_values(0, even);
        request_kq(0, even), request_tm(0, even);
        if constexpr (STATE) request_values(1, odd);
        request_kq(1, odd);
        if constexpr (STATE) request_tm(1, odd);
        else odd.tm[0][0] = odd.tm[0][1] = odd.tm[1][0] = odd.tm[1][1] = u32x4{0, 0, 0, 0};
        if constexpr (STATE) {
            publish_state();
            place(0, even);
        }
        // (pairs of blocks without a branch between them, so that the loads asked for in one block are known to be
        // behind those of the block before wherever a wait is placed)
        uint32_t blk = 0;
        for (; blk + 1 < nblocks; blk += 2) {
            step(team, blk, even, odd);
            step(team, blk + 1, odd, even);
        }
        if (blk < nblocks) step(team, blk, even, odd);
        if constexpr (!STATE) outputs(nblocks - 1, true, nblocks % 2 ? even : odd);
    };
    // (the first team is the chain: where both teams' waves of a SIMD are ready, its go first)
    if (state_team) {
        __builtin_amdgcn_s_setprio(2);
        walk(std::true_type{});
    } else {
        walk(std::false_type{});
    }
    if (state_team) {
#pragma unroll
        for (int mt = 0; mt < NT; mt++) {
#pragma unroll
            for (int nt = 0; nt < 2; nt++) {
                *reinterpret_cast<floatx4 *>(state + (16 * mt + n) * K_DIM + 32 * wave + 16 * nt + 4 * j) = s_reg[mt][nt];
            }
        }
    }
}

}  // namespace

int setup_deltanet_chunk() {
    const std::pair<const void *, int> prepares[] = {{reinterpret_cast<const void *>(deltanet_chunk_prepare_kernel<1, false>), PrepLds<1>::BYTES},
                                                     {reinterpret_cast<const void *>(deltanet_chunk_prepare_kernel<2, false>), PrepLds<2>::BYTES},
                                                     {reinterpret_cast<const void *>(deltanet_chunk_prepare_kernel<2, true>), PrepLds<2>::BYTES}};
    for (const auto &[kernel, bytes] : prepares) {
        if (int rc = int(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes))) return rc;
    }
    for (const void *kernel : {reinterpret_cast<const void *>(deltanet_chunk_chain_kernel<false>), reinterpret_cast<const void *>(deltanet_chunk_chain_kernel<true>)}) {
        if (int rc = int(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, ChainLds::BYTES))) return rc;
    }
    return 0;
}

size_t deltanet_chunk_workspace_bytes(const saetta_rows_step_params &p) {
    if (p.snapshots || p.tokens < DELTANET_CHUNK_FROM || p.v_dim % DV != 0 || p.k_heads == 0 || p.v_heads % p.k_heads != 0) return 0;
    return size_t((p.tokens + C - 1) / C) * block_bytes(p.k_heads, p.v_heads);
}

namespace {
// Whether the launch recorded last is the conv that made `mixed` for this call; it is then taken off the list and the
// prepare kernel makes it too.  For a call of its own the conv has run before this call is known.  The conv's inputs
// are read beside what this call writes and reads here, so buffers that a program lays over each other (a workspace in
// the place of x, gates in the place of `mixed`) keep the two launches.
bool take_conv(LaunchList &list, ChunkArgs &args, float *&conv_out) {
    if (list.launches.empty() || list.launches.back().kind != LAUNCH_CONV) return false;
    const LaunchRecord &conv = list.launches.back();
    const float *x = list.arg<const float *>(conv, 0), *w = list.arg<const float *>(conv, 1);
    float *conv_state = list.arg<float *>(conv, 2), *out = list.arg<float *>(conv, 3);
    const saetta_conv_rows_params &c = list.arg<saetta_conv_rows_params>(conv, 5);
    if (c.kernel_size != CONV || c.snapshots || c.channels != args.channels || c.tokens != args.tokens || out != args.mixed) return false;
    const size_t rows = size_t(args.tokens) * args.channels * sizeof(float), gates = size_t(args.tokens) * args.v_heads * sizeof(float);
    const Span inputs[] = {{x, rows}, {w, size_t(CONV) * args.channels * sizeof(float)}, {args.a, gates}, {args.b, gates},
                                                      {args.a_log, args.v_heads * sizeof(float)}, {args.dt_bias, args.v_heads * sizeof(float)}},
        outputs[] = {{out, rows}, {conv_state, size_t(CONV - 1) * args.channels * sizeof(float)},
                     {args.ws, size_t((args.tokens + C - 1) / C) * block_bytes(args.k_heads, args.v_heads)}};
    for (const auto &o : outputs) {
        for (const auto &i : inputs) {
            if (!apart(o, i)) return false;
        }
        for (const auto &other : outputs) {
            if (&other != &o && !apart(o, other)) return false;
        }
    }
    args.x = x, args.conv_w = w, args.conv_state = conv_state, conv_out = out;
    list.launches.pop_back();
    return true;
}
}  // namespace

int run_deltanet_chunk(hipStream_t stream, const float *mixed, const float *a, const float *b, const float *a_log,
                       const float *dt_bias, float *state, float *o, const saetta_rows_step_params &p, uint32_t channels,
                       void *workspace) {
    const uint32_t nblocks = (p.tokens + C - 1) / C;
    ChunkArgs args{mixed, a, b, a_log, dt_bias, state, o, static_cast<unsigned char *>(workspace), p.k_heads, p.v_heads, p.v_dim, p.tokens, channels, p.eps, nullptr, nullptr, nullptr};
    const bool two_heads = p.v_heads == 2 * p.k_heads;
    LaunchList *list = recording();
    float *conv_out = nullptr;
    // The conv inside: while every workgroup, the blocks' and the values', has a CU to itself.  Where they share one, a
    // block's chain of phases is held up by the conv beside it, and the conv's own launch is the better one (whole chunk,
    // us, inside against apart: 512 tokens 35.8 and 39.3; 513 41.8 and 39.3, 640 45.2 and 43.4, 800 50.7 and 50.4, 1000 58.3 and 58.1,
    // 2047 126 and 120; the values' conv alone as a launch of its own: 513 41.8, 1000 57.4, 2300 124.7 instead of 122.0, 4096 226.7
    // instead of 222.6).
    const uint32_t columns = (p.v_heads * p.v_dim / 4 + PREP_THREADS - 1) / PREP_THREADS, value_groups = columns * ((p.tokens + CONV_VALUES - 1) / CONV_VALUES);
    const bool conv_inside = two_heads && p.v_dim == CONV_V && nblocks * p.k_heads + value_groups <= cu_count();
    if (conv_inside && list && take_conv(*list, args, conv_out)) {
        launch(deltanet_chunk_prepare_kernel<2, true>, dim3(nblocks + (value_groups + p.k_heads - 1) / p.k_heads, p.k_heads), PREP_THREADS, PrepLds<2>::BYTES, stream, args, conv_out);
    } else if (two_heads) {
        launch(deltanet_chunk_prepare_kernel<2, false>, dim3(nblocks, p.k_heads), PREP_THREADS, PrepLds<2>::BYTES, stream, args, conv_out);
    } else {
        launch(deltanet_chunk_prepare_kernel<1, false>, dim3(nblocks, p.v_heads), PREP_THREADS, PrepLds<1>::BYTES, stream, args, conv_out);
    }
    const bool ahead = size_t(p.tokens) * channels * sizeof(float) + deltanet_chunk_workspace_bytes(p) >= AHEAD_FROM;
    launch(ahead ? deltanet_chunk_chain_kernel<true> : deltanet_chunk_chain_kernel<false>, dim3(p.v_dim / DV * p.v_heads), 512, ChainLds::BYTES, stream, args);
    return SAETTA_OK;
}

}  // namespace saetta
