// Gated DeltaNet (linear attention): the conv and the step after it, for one token, for up to 8
// rows of a verify step, and for the tokens of a prefill chunk in order.
//
// Kernels:
//   deltanet_conv_kernel, deltanet_step_kernel          one token, the reference's two ops
//   deltanet_conv_rows_kernel, deltanet_rows_kernel,
//   deltanet_gated_norm_rows_kernel   any number of tokens in order (prefill chunks)
//   deltanet_rows_small_kernel, deltanet_rows_small_tail_kernel
//                                                       conv and step together for 1..8 tokens
//
// Reference: kernels deltanet_conv and deltanet_step (kernels/layers.metal:198-226,290-357),
// recorded by GpuDeltaNet (src/gpu_layers.rs:573-1000); CPU definition src/cpu/deltanet.rs:69-155:
//   conv:  out[c] = silu(sum_t w[c][t] * past[t][c] + w[c][K-1] * x[c]); x shifts into the state
//   step, per value head h (key head h / (v_heads / k_heads)), key dim 128:
//     q, k L2-normalised (eps inside the root), q also times 1 / sqrt(128)
//     g = exp(-exp(A_log[h]) * softplus(a[h] + dt_bias[h])),  beta = sigmoid(b[h])
//     per state row i:  S_i <- g S_i;  d = (v[i] - S_i . k) beta;  S_i += d k;  o[i] = S_i . q
//     y = o / sqrt(mean(o^2) + eps) * norm_w * silu(z)
//
// The step is a stream over the recurrent state: 32 heads x 128 x 128 f32 = 2 MB read and 2 MB
// written per layer and token, everything else is small.  One workgroup of 1024 threads per value
// head; a state row is 128 floats = 32 lanes x float4, so a wavefront takes two rows at a time
// (whole 512-byte rows per half wave: reads and writes are full cache lines), all of a wave's
// rows are requested before the first is used, and the dot products are reductions over 32 lanes
// by DPP moves (no LDS).
#include "common.hpp"
#include "deltanet_gates.hpp"
#include "lanes.hpp"

#include <type_traits>

namespace saetta {
namespace {

constexpr int K_DIM = 128;
constexpr int STEP_THREADS = 1024;
constexpr int MAX_ROWS_PER_LANE = 8;  // v_dim up to 256

__device__ __forceinline__ float dot4(float4 a, float4 b) { return a.x * b.x + a.y * b.y + a.z * b.z + a.w * b.w; }

__global__ __launch_bounds__(256) void deltanet_conv_kernel(const float *__restrict__ x, const float *__restrict__ w,
                                                            float *__restrict__ state, float *__restrict__ out,
                                                            saetta_conv_params p) {
    const uint32_t c = blockIdx.x * 256 + threadIdx.x;
    if (c >= p.channels) return;
    const uint32_t past = p.kernel_size - 1;
    const float *wc = w + size_t(c) * p.kernel_size;
    const float xc = x[c];
    // the CPU adds the stored inputs oldest first and the new one last (src/cpu/deltanet.rs:122-126)
    float old = 0.0f;
    for (uint32_t t = 0; t < past; t++) old += wc[t] * state[size_t(t) * p.channels + c];
    for (uint32_t t = 0; t + 1 < past; t++) state[size_t(t) * p.channels + c] = state[size_t(t + 1) * p.channels + c];
    state[size_t(past - 1) * p.channels + c] = xc;
    out[c] = silu_f(old + wc[past] * xc);
}

struct StepArgs {
    const float *q, *k, *v, *a, *b, *a_log, *dt_bias;
    float *state;
    const float *z, *norm_w;
    float *y;
    saetta_step_params p;
};

__global__ __launch_bounds__(STEP_THREADS) void deltanet_step_kernel(StepArgs a) {
    __shared__ float o_lds[MAX_ROWS_PER_LANE * 32];
    __shared__ float partial[STEP_THREADS / 64];
    const uint32_t h = blockIdx.x, tid = threadIdx.x;
    const uint32_t lane32 = tid & 31, half_wave = tid >> 5;  // 32 half waves, one state row each at a time
    const uint32_t v_dim = a.p.v_dim;
    const uint32_t kh = h / (a.p.v_heads / a.p.k_heads);

    // the state rows of this half wave: i = half_wave, half_wave + 32, ... all requested up front
    float4 s[MAX_ROWS_PER_LANE];
    float *rows = a.state + size_t(h) * v_dim * K_DIM;
#pragma unroll
    for (int r = 0; r < MAX_ROWS_PER_LANE; r++) {
        const uint32_t i = half_wave + 32 * r;
        if (i < v_dim) s[r] = reinterpret_cast<const float4 *>(rows + size_t(i) * K_DIM)[lane32];
    }
    float4 qv = reinterpret_cast<const float4 *>(a.q + size_t(kh) * K_DIM)[lane32];
    float4 kv = reinterpret_cast<const float4 *>(a.k + size_t(kh) * K_DIM)[lane32];
    // normalize_qk (src/cpu/deltanet.rs:133-146): x * (scale / sqrt(x . x + eps))
    const float qi = (1.0f / sqrtf(float(K_DIM))) / sqrtf(group_reduce<32>(dot4(qv, qv), SumOp()) + a.p.eps);
    const float ki = 1.0f / sqrtf(group_reduce<32>(dot4(kv, kv), SumOp()) + a.p.eps);
    qv.x *= qi, qv.y *= qi, qv.z *= qi, qv.w *= qi;
    kv.x *= ki, kv.y *= ki, kv.z *= ki, kv.w *= ki;

    const float xg = a.a[h] + a.dt_bias[h];
    const float softplus = fmaxf(xg, 0.0f) + log1pf(expf(-fabsf(xg)));
    const float g = expf(-expf(a.a_log[h]) * softplus);
    const float beta = sigmoid_f(a.b[h]);
    const float *vh = a.v + size_t(h) * v_dim;

#pragma unroll
    for (int r = 0; r < MAX_ROWS_PER_LANE; r++) {
        const uint32_t i = half_wave + 32 * r;
        if (i < v_dim) {  // the same for the 32 lanes of a row
            float4 x = s[r];
            x.x *= g, x.y *= g, x.z *= g, x.w *= g;
            const float delta = (vh[i] - group_reduce<32>(dot4(x, kv), SumOp())) * beta;
            x.x += kv.x * delta, x.y += kv.y * delta, x.z += kv.z * delta, x.w += kv.w * delta;
            reinterpret_cast<float4 *>(rows + size_t(i) * K_DIM)[lane32] = x;
            const float o = group_reduce<32>(dot4(x, qv), SumOp());
            if (lane32 == 0) o_lds[i] = o;
        }
    }
    __syncthreads();

    // gated RMSNorm over the head's v_dim outputs, times silu(z)
    const float o = tid < v_dim ? o_lds[tid] : 0.0f;
    const float sq = group_reduce<64>(o * o, SumOp());
    if ((tid & 63) == 0) partial[tid >> 6] = sq;
    __syncthreads();
    float total = 0.0f;
#pragma unroll
    for (int w = 0; w < STEP_THREADS / 64; w++) total += partial[w];
    const float inv = 1.0f / sqrtf(total / float(v_dim) + a.p.eps);
    if (tid < v_dim) {
        const size_t nidx = size_t(h) * v_dim + tid;
        a.y[nidx] = o * (inv * a.norm_w[tid]) * silu_f(a.z[nidx]);
    }
}


// ---- several tokens in one launch: verify rows and prefill chunks ------------------------------
//
// Reference: conv_rows2 + conv_state, delta_prep + delta_rows3 and the gated norm after them
// (kernels/prefill.metal:734-1116, recorded by src/prefill.rs:1433-1578), and for verify rows
// deltanet_conv_rows + deltanet_step_rows (kernels/layers.metal:510-635, src/gpu_layers.rs:686-786).
// Token t + 1 sees the state token t left, exactly as t single-token calls would.

// One thread per (channel, tile of CONV_TILE tokens).  Input i of the window of token t is
// x[i] for i >= 0 and the stored state row i + kernel_size - 1 before that; the taps are added
// oldest first, as the single-token kernel does.  The window slides in registers (KS taps known
// at compile time for the common sizes), so every x is loaded once per tile.
constexpr uint32_t CONV_TILE = 32;

__device__ __forceinline__ float conv_input(const float *x, const float *state, int i, uint32_t c,
                                            const saetta_conv_rows_params &p) {
    return i >= 0 ? x[size_t(i) * p.channels + c] : state[size_t(i + int(p.kernel_size) - 1) * p.channels + c];
}

// After the outputs the last kernel_size - 1 inputs become the state.  Only the tokens before the window's length
// read it, and those lie in the first tile: its thread of the channel has read what it needs and moves the rows
// itself, where a launch of its own took 2.5 us.  Rows are written in ascending order and row j only reads rows above
// it (or x), so the shift is safe in place.
__device__ __forceinline__ void conv_state_move(const float *x, float *state, uint32_t c, const saetta_conv_rows_params &p) {
    const int past = int(p.kernel_size) - 1;
    for (int j = 0; j < past; j++) state[size_t(j) * p.channels + c] = conv_input(x, state, int(p.tokens) - past + j, c, p);
}

// The same for four channels a thread (16-byte loads and stores, a tile's loads all in flight), four taps: every channel's
// sums are taken in the same order as above, so the results are the same bit for bit.  Bound by memory over a long chunk,
// by one trip through memory and the instructions behind it over a short one, so the tiles are short: a tile of 4 tokens
// reads 7 rows, 3 of them a second time out of the L2, and is done 8 times as soon as one of 32.  Conv alone, tiles of 32
// -> 4: 40 tokens 13.9 -> 4.6 us, 2100 34.6 -> 27, 4096 50.6 -> 49.9 (268 MB at 5.4 TB/s); whole layer, us, tiles of
// 32 / 16 / 8 / 4: 40 tokens 25.7 / 21.1 / 18.8 / 17.6, 2100 150 / 147 / 145 / 142, 4095 269 / 273 / 269 / 267.
// Vector instructions are issued for half of its time: the activation's short form takes 0.2 to 1 us of the layer (40 tokens 16.85 -> 16.65,
// 513 39.3 -> 39.1, 2300 121.7 -> 120.9, 4096 221.6 -> 220.5; the norm's 2300 120.9 -> 120.7).  The taps by way of LDS, whole lines to a load
// instead of 64 bytes to a lane, give nothing (40 tokens 16.9, 2300 121.5).
constexpr uint32_t CONV4_TILE = 4;
constexpr uint32_t CONV4_TAPS = 4, CONV4_FROM = SAETTA_MAX_ROWS + 1;  // (taps it is made for; tokens from which it is taken)
static_assert(CONV4_TILE >= CONV4_TAPS - 1, "every token that reads the state lies in the first tile");
__global__ __launch_bounds__(256) void deltanet_conv_rows4_kernel(const float *__restrict__ x, const float *__restrict__ w,
                                                                  float *state, float *__restrict__ out,
                                                                  float *__restrict__ snaps, saetta_conv_rows_params p) {
    constexpr int KS = CONV4_TAPS;
    const uint32_t c4 = blockIdx.x * 256 + threadIdx.x, quads = p.channels / 4;
    if (c4 >= quads) return;
    const float4 *x4 = reinterpret_cast<const float4 *>(x);
    float4 *o4 = reinterpret_cast<float4 *>(out), *s4 = reinterpret_cast<float4 *>(state);
    // taps[j] holds tap j of the four channels (w is [channel][4]: the thread's 16 floats lie in a row)
    float4 taps[KS];
    {
        const float4 *w4 = reinterpret_cast<const float4 *>(w) + size_t(c4) * 4;
        const float4 a = w4[0], b = w4[1], c = w4[2], d = w4[3];
        taps[0] = make_float4(a.x, b.x, c.x, d.x), taps[1] = make_float4(a.y, b.y, c.y, d.y);
        taps[2] = make_float4(a.z, b.z, c.z, d.z), taps[3] = make_float4(a.w, b.w, c.w, d.w);
    }
    const uint32_t t0 = blockIdx.y * CONV4_TILE;
    float4 win[KS - 1], xt[CONV4_TILE];
#pragma unroll
    for (int j = 0; j < KS - 1; j++) {
        const int i = int(t0) - (KS - 1) + j;
        win[j] = i >= 0 ? x4[size_t(i) * quads + c4] : s4[size_t(i + KS - 1) * quads + c4];
    }
#pragma unroll
    for (uint32_t u = 0; u < CONV4_TILE; u++) xt[u] = x4[size_t(min(t0 + u, p.tokens - 1)) * quads + c4];
#pragma unroll
    for (uint32_t u = 0; u < CONV4_TILE; u++) {
        const uint32_t t = t0 + u;
        if (t >= p.tokens) break;
        float4 acc = make_float4(0, 0, 0, 0);
#pragma unroll
        for (int j = 0; j < KS - 1; j++) {
            acc.x += taps[j].x * win[j].x, acc.y += taps[j].y * win[j].y, acc.z += taps[j].z * win[j].z, acc.w += taps[j].w * win[j].w;
        }
        o4[size_t(t) * quads + c4] = silu4_f(make_float4(acc.x + taps[KS - 1].x * xt[u].x, acc.y + taps[KS - 1].y * xt[u].y,
                                                         acc.z + taps[KS - 1].z * xt[u].z, acc.w + taps[KS - 1].w * xt[u].w));
#pragma unroll
        for (int j = 0; j + 1 < KS - 1; j++) win[j] = win[j + 1];
        win[KS - 2] = xt[u];
        if (p.snapshots) {
            float4 *snap = reinterpret_cast<float4 *>(snaps) + size_t(t) * (KS - 1) * quads;
#pragma unroll
            for (int j = 0; j < KS - 1; j++) snap[size_t(j) * quads + c4] = win[j];
        }
    }
    if (blockIdx.y == 0) {  // (CONV4_FROM tokens at least: the new state is all inputs)
#pragma unroll
        for (int j = 0; j < KS - 1; j++) s4[size_t(j) * quads + c4] = x4[size_t(p.tokens - (KS - 1) + j) * quads + c4];
    }
}

template <int KS>  // taps; 0: any number (read from p), the window is re-read from memory
__global__ __launch_bounds__(256) void deltanet_conv_rows_kernel(const float *__restrict__ x,
                                                                 const float *__restrict__ w,
                                                                 float *state, float *__restrict__ out,
                                                                 float *__restrict__ snaps,
                                                                 saetta_conv_rows_params p) {
    const uint32_t c = blockIdx.x * 256 + threadIdx.x;
    if (c >= p.channels) return;
    const int past = int(p.kernel_size) - 1;
    const float *wc = w + size_t(c) * p.kernel_size;
    const uint32_t t_begin = blockIdx.y * CONV_TILE, t_end = min(p.tokens, t_begin + CONV_TILE);
    if constexpr (KS > 0) {
        float taps[KS], win[KS - 1];
#pragma unroll
        for (int j = 0; j < KS; j++) taps[j] = wc[j];
#pragma unroll
        for (int j = 0; j < KS - 1; j++) win[j] = conv_input(x, state, int(t_begin) - (KS - 1) + j, c, p);
        for (uint32_t t = t_begin; t < t_end; t++) {
            const float xt = x[size_t(t) * p.channels + c];
            float acc = 0.0f;
#pragma unroll
            for (int j = 0; j < KS - 1; j++) acc += taps[j] * win[j];
            out[size_t(t) * p.channels + c] = silu_f(acc + taps[KS - 1] * xt);
#pragma unroll
            for (int j = 0; j + 1 < KS - 1; j++) win[j] = win[j + 1];
            win[KS - 2] = xt;
            if (p.snapshots) {
                float *snap = snaps + size_t(t) * (KS - 1) * p.channels;
#pragma unroll
                for (int j = 0; j < KS - 1; j++) snap[size_t(j) * p.channels + c] = win[j];
            }
        }
    } else {
        for (uint32_t t = t_begin; t < t_end; t++) {
            float acc = 0.0f;
            for (int j = 0; j < past; j++) acc += wc[j] * conv_input(x, state, int(t) - past + j, c, p);
            out[size_t(t) * p.channels + c] = silu_f(acc + wc[past] * x[size_t(t) * p.channels + c]);
            if (p.snapshots) {
                float *snap = snaps + size_t(t) * past * p.channels;
                for (int j = 0; j < past; j++) {
                    snap[size_t(j) * p.channels + c] = conv_input(x, state, int(t) - past + 1 + j, c, p);
                }
            }
        }
    }
    if (blockIdx.y == 0) conv_state_move(x, state, c, p);
}

// The delta rule over the tokens, in order.  A workgroup owns a few rows of one value head's state
// for the whole launch: LANES lanes per row, 128 / LANES state values per lane in registers.  The
// chain from one token to the next (decay, S_i . k, its sum over the row's lanes, delta, update)
// cannot be shortened, so the rows are spread as wide as the chip: 32 lanes per row make the 4096
// rows of 32 heads two wavefronts on every SIMD, one running while the other waits on its chain.
// The q and k of the head's key head are the same for all its rows: they are staged per block of 16
// tokens in LDS (double buffered; the next block's loads are in flight while this one runs),
// normalised on the way in; g, beta and v of a block sit in the lanes (lane p of each 16 holds
// token p's) and reach the others by DPP row broadcasts.
constexpr int ROWS_TB = 16;  // tokens per staged block
#ifndef ROWS_LANES_PER_ROW
#define ROWS_LANES_PER_ROW 16
#endif

struct RowsArgs {
    const float *mixed, *a, *b, *a_log, *dt_bias;
    float *state;
    float *o;      // [tokens][v_heads][v_dim], before the gated norm
    float *snaps;  // [tokens] copies of the state, or unused
    saetta_rows_step_params p;
    uint32_t channels;
};

template <int I>
__device__ __forceinline__ float row_lane(float x) {
    // value of lane I of every row of 16 lanes
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x150 + I, 0xf, 0xf, true));
}

template <int I>
struct TokenLoop {
    template <class F>
    static __device__ __forceinline__ void run(F &&f) {
        f(std::integral_constant<int, I>{});
        if constexpr (I + 1 < ROWS_TB) TokenLoop<I + 1>::run(f);
    }
};

// sum of N float4 products as a tree (N = 1 or 2): two or three dependent additions after the products
template <int N>
__device__ __forceinline__ float dot_tree(const float4 (&a)[N], const float4 (&b)[N]) {
    float sum = (a[0].x * b[0].x + a[0].y * b[0].y) + (a[0].z * b[0].z + a[0].w * b[0].w);
    if constexpr (N == 2) sum += (a[1].x * b[1].x + a[1].y * b[1].y) + (a[1].z * b[1].z + a[1].w * b[1].w);
    return sum;
}

template <bool SNAPS, int LANES>
__global__ __launch_bounds__(256) void deltanet_rows_kernel(RowsArgs a) {
    constexpr int PER_LANE = K_DIM / LANES;  // state values per lane: 8 or 4
    constexpr int F4 = PER_LANE / 4;         // as float4s
    constexpr int ROWS_PER_WG = 256 / LANES;
    static_assert(LANES == 16 || LANES == 32, "a row is one or two DPP rows");
    // a token's q and k: [q | k][float4 of the lane][lane][4] floats, so that the lanes of a row read
    // contiguous bytes
    __shared__ __attribute__((aligned(16))) float qk_lds[2][ROWS_TB][2 * K_DIM];
    __shared__ float gb_lds[2][ROWS_TB][2];
    __shared__ float o_lds[ROWS_TB][ROWS_PER_WG];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint32_t h = blockIdx.y, part = tid % LANES, row_in_wg = tid / LANES;
    const uint32_t tok_lane = tid & 15;  // the token of a block whose g, beta and v this lane holds
    const uint32_t row = blockIdx.x * ROWS_PER_WG + row_in_wg;
    const uint32_t v_dim = a.p.v_dim, v_heads = a.p.v_heads, tokens = a.p.tokens;
    const bool live = row < v_dim;
    const uint32_t kh = h / (v_heads / a.p.k_heads);
    const uint32_t key_size = a.p.k_heads * K_DIM;
    const size_t value_size = size_t(v_heads) * v_dim;

    float4 st[F4];
    float *sp = a.state + (size_t(h) * v_dim + (live ? row : 0)) * K_DIM + part * PER_LANE;
#pragma unroll
    for (int c = 0; c < F4; c++) st[c] = live ? reinterpret_cast<const float4 *>(sp)[c] : make_float4(0, 0, 0, 0);

    const float exp_a = expf(a.a_log[h]);
    const float bias = a.dt_bias[h];
    const float q_scale = 1.0f / sqrtf(float(K_DIM));

    // ---- one block's inputs, as loaded (registers) --------------------------------------------
    // thread -> float4 `lane` of token wave + 4 j of the block: lanes 0-31 are q, 32-63 are k
    float4 raw[ROWS_TB / 4];
    float ga = 0.0f, gbv = 0.0f;  // a and b of token `tid` (threads 0-15)
    bool g_real = false;          // that token exists
    float nv = 0.0f;              // v of token `tok_lane`, this thread's row
    auto load_block = [&](uint32_t t0) {
        const uint32_t off = (lane < 32 ? 0 : key_size) + kh * K_DIM + 4 * (lane & 31);
#pragma unroll
        for (int j = 0; j < ROWS_TB / 4; j++) {
            const uint32_t t = t0 + wave + 4 * j;
            raw[j] = make_float4(0, 0, 0, 0);
            if (t < tokens) raw[j] = *reinterpret_cast<const float4 *>(a.mixed + size_t(t) * a.channels + off);
        }
        g_real = t0 + tid < tokens;
        if (tid < ROWS_TB && g_real) {
            ga = a.a[size_t(t0 + tid) * v_heads + h];
            gbv = a.b[size_t(t0 + tid) * v_heads + h];
        }
        nv = 0.0f;
        if (live && t0 + tok_lane < tokens) {
            nv = a.mixed[size_t(t0 + tok_lane) * a.channels + 2 * key_size + h * v_dim + row];
        }
    };
    // normalise (src/cpu/deltanet.rs:133-146), compute the gates, and put the block into buffer `buf`
    auto store_block = [&](int buf) {
#pragma unroll
        for (int j = 0; j < ROWS_TB / 4; j++) {
            const float4 x = raw[j];
            const float ss = group_reduce<32>(dot4(x, x), SumOp());
            const float inv = (lane < 32 ? q_scale : 1.0f) * __builtin_amdgcn_rsqf(ss + a.p.eps);
            const uint32_t f = lane & 31;  // float4 f of the vector belongs to lane f / F4, its float4 f % F4
            float *dst = &qk_lds[buf][wave + 4 * j][(lane < 32 ? 0 : K_DIM) + (f % F4) * (LANES * 4) + (f / F4) * 4];
            *reinterpret_cast<float4 *>(dst) = make_float4(x.x * inv, x.y * inv, x.z * inv, x.w * inv);
        }
        if (tid < ROWS_TB) {
            float g, beta;
            fast_gates(ga + bias, exp_a, gbv, g, beta);
            gb_lds[buf][tid][0] = g_real ? g : 1.0f;
            gb_lds[buf][tid][1] = g_real ? beta : 0.0f;
        }
    };

    load_block(0);
    store_block(0);
    float v_cur = nv;
    __syncthreads();

    int cur = 0;
    for (uint32_t t0 = 0; t0 < tokens; t0 += ROWS_TB) {
        const bool more = t0 + ROWS_TB < tokens;
        if (more) load_block(t0 + ROWS_TB);
        const float g_mine = gb_lds[cur][tok_lane][0], b_mine = gb_lds[cur][tok_lane][1];
        const float v_mine = v_cur;

        // Tokens past the end of a ragged last block are staged as q = k = 0, g = 1, beta = 0: they
        // leave the state as it is, so the 16 steps run without a branch between them, and token
        // I + 1's q and k are read from LDS while token I is computed.
        float4 q_next[F4], k_next[F4];
        auto read_qk = [&](int i) {
            const float *qk = qk_lds[cur][i];
#pragma unroll
            for (int c = 0; c < F4; c++) {
                q_next[c] = *reinterpret_cast<const float4 *>(qk + c * (LANES * 4) + part * 4);
                k_next[c] = *reinterpret_cast<const float4 *>(qk + K_DIM + c * (LANES * 4) + part * 4);
            }
        };
        read_qk(0);
        float out_mine = 0.0f;  // lane `tok_lane` keeps the output of that token
        float out_part = 0.0f;  // this lane's share of the previous token's output: its sum over the
                                // row is not needed by the next token, so it runs beside that token's chain
        auto token = [&](auto index) {
            constexpr int I = decltype(index)::value;
            float4 q[F4], k[F4];
#pragma unroll
            for (int c = 0; c < F4; c++) q[c] = q_next[c], k[c] = k_next[c];
            if constexpr (I + 1 < ROWS_TB) read_qk(I + 1);
            __builtin_amdgcn_sched_barrier(0);  // the reads stay here, a token ahead of their use
            if constexpr (I > 0) {
                const float out = group_reduce<LANES>(out_part, SumOp());
                out_mine = tok_lane == I - 1 ? out : out_mine;
            }
            const float gt = row_lane<I>(g_mine), bt = row_lane<I>(b_mine), vt = row_lane<I>(v_mine);
#pragma unroll
            for (int c = 0; c < F4; c++) st[c].x *= gt, st[c].y *= gt, st[c].z *= gt, st[c].w *= gt;
            const float mem = group_reduce<LANES>(dot_tree<F4>(st, k), SumOp());
            const float delta = (vt - mem) * bt;
#pragma unroll
            for (int c = 0; c < F4; c++) {
                st[c].x += k[c].x * delta, st[c].y += k[c].y * delta, st[c].z += k[c].z * delta, st[c].w += k[c].w * delta;
            }
            out_part = dot_tree<F4>(st, q);
            if constexpr (SNAPS) {
                if (live && t0 + I < tokens) {
                    float *snap = a.snaps + size_t(t0 + I) * v_heads * v_dim * K_DIM +
                                  (size_t(h) * v_dim + row) * K_DIM + part * PER_LANE;
#pragma unroll
                    for (int c = 0; c < F4; c++) reinterpret_cast<float4 *>(snap)[c] = st[c];
                }
            }
        };
        TokenLoop<0>::run(token);
        {
            const float out = group_reduce<LANES>(out_part, SumOp());
            out_mine = tok_lane == ROWS_TB - 1 ? out : out_mine;
        }
        if (part < ROWS_TB) o_lds[part][row_in_wg] = out_mine;

        if (more) {
            store_block(cur ^ 1);
            v_cur = nv;
        }
        __syncthreads();  // the block's outputs are in o_lds; the next block is staged
        if (tid < ROWS_TB * ROWS_PER_WG) {
            // thread -> (token, row): the rows of a token are contiguous
            const uint32_t ti = tid / ROWS_PER_WG, ri = tid % ROWS_PER_WG;
            const uint32_t t = t0 + ti, r = blockIdx.x * ROWS_PER_WG + ri;
            if (t < tokens && r < v_dim) a.o[size_t(t) * value_size + size_t(h) * v_dim + r] = o_lds[ti][ri];
        }
        __syncthreads();  // o_lds is free again
        cur ^= 1;
    }
    if (live) {
#pragma unroll
        for (int c = 0; c < F4; c++) reinterpret_cast<float4 *>(sp)[c] = st[c];
    }
}

// The same for the chunks of a prefill, which are held to a tolerance and not to the single-token kernels'
// bits: LP = v_dim / 4 lanes per pair, four values each (16-byte loads and stores, two pairs per wavefront at
// the model's 128), the sum of squares over the LP lanes.
template <int LP>
__global__ __launch_bounds__(256) void deltanet_gated_norm_wide_kernel(float *y, const float *__restrict__ z,
                                                                       const float *__restrict__ norm_w, uint32_t pairs, float eps) {
    const uint32_t at = blockIdx.x * 256 + threadIdx.x, pair = at / LP, part = at % LP;
    if (pair >= pairs) return;  // (whole groups of LP lanes: 256 is a multiple of LP)
    float4 *yp = reinterpret_cast<float4 *>(y) + size_t(pair) * LP + part;
    const float4 o = *yp, g = reinterpret_cast<const float4 *>(z)[size_t(pair) * LP + part], w = reinterpret_cast<const float4 *>(norm_w)[part];
    const float total = group_reduce<LP>(o.x * o.x + o.y * o.y + o.z * o.z + o.w * o.w, SumOp());
    const float inv = 1.0f / sqrtf(total / float(4 * LP) + eps);
    const float4 open = silu4_f(g);
    *yp = make_float4(o.x * (inv * w.x) * open.x, o.y * (inv * w.y) * open.y, o.z * (inv * w.z) * open.z, o.w * (inv * w.w) * open.w);
}

// y = o / sqrt(mean(o^2) + eps) * norm_w * silu(z) per (token, value head), in place on y:
// one wavefront per pair, v_dim up to 256.
__global__ __launch_bounds__(256) void deltanet_gated_norm_rows_kernel(float *y, const float *__restrict__ z,
                                                                       const float *__restrict__ norm_w,
                                                                       uint32_t pairs, uint32_t v_dim, float eps) {
    const uint32_t pair = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (pair >= pairs) return;
    float *yp = y + size_t(pair) * v_dim;
    const float *zp = z + size_t(pair) * v_dim;
    float o[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const uint32_t d = lane + 64 * i;
        o[i] = d < v_dim ? yp[d] : 0.0f;
    }
    // the single-token kernel sums 64-lane partials in the same order: lanes first, then the groups of 64
    float total = 0.0f;
    {
        float part_sum[4];
#pragma unroll
        for (int i = 0; i < 4; i++) part_sum[i] = group_reduce<64>(o[i] * o[i], SumOp());
#pragma unroll
        for (int i = 0; i < 4; i++) total += part_sum[i];
    }
    const float inv = 1.0f / sqrtf(total / float(v_dim) + eps);
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const uint32_t d = lane + 64 * i;
        if (d < v_dim) yp[d] = o[i] * (inv * norm_w[d]) * silu_f(zp[d]);
    }
}


// ---- up to 8 tokens, conv and step together (the verify step) -----------------------------------
//
// Reference: kernel deltanet_rows (kernels/layers.metal, recorded by GpuDeltaNet::record_rows with
// DN_SIMDS = 0, src/gpu_layers.rs:737-757): conv, q/k norm, gates, delta rule, gated norm for m rows
// in one op, with the states after every row to the snapshot buffers; with one row, what
// GpuDeltaNet::record does (src/gpu_layers.rs:633-684).  The separate conv and step kernels above
// cost a launch each and the step runs on 32 workgroups.  Here a workgroup takes 16 rows of one value
// head's state (grid 8 x 32 at the model's shape), computes the conv outputs it needs itself for all
// the tokens (q and k of its key head, v of its rows: the conv state is only read) and walks the
// tokens; what needs the whole head or the whole layer is a small second launch: the gated norm over
// a head's outputs, the new conv state and the conv snapshots.
constexpr int SMALL_ROWS_MAX = 8;

struct SmallRowsArgs {
    const float *x, *w;
    float *conv_state;
    const float *a, *b, *a_log, *dt_bias;
    float *state;
    const float *z, *norm_w;
    float *y, *conv_snaps, *state_snaps;
    saetta_rows_fused_params p;
    uint32_t channels;
};

// out[t] of channel c for t < tokens.  The stored inputs and the new ones are one sequence in
// registers, the stored ones ending at index 14, x[t] at 15 + t; the taps are right-aligned the same
// way (the newest at 15), so that out[t] = sum_k taps[k] * seq[t + k] with constant indices: the
// unused leading taps are zeros, which leaves the sum (oldest first, the new input last, as the
// single-token kernel adds them) unchanged.  Every load is requested before the first is used.
template <typename F>
__device__ __forceinline__ void conv_small(const SmallRowsArgs &a, uint32_t c, F &&emit) {
    const uint32_t past = a.p.kernel_size - 1, tokens = a.p.rows;
    const float *wc = a.w + size_t(c) * a.p.kernel_size;
    float taps[16], seq[15 + SMALL_ROWS_MAX];
#pragma unroll
    for (uint32_t k = 0; k < 16; k++) taps[k] = k + past >= 15 ? wc[k + past - 15] : 0.0f;
#pragma unroll
    for (uint32_t k = 0; k < 15; k++) seq[k] = k + past >= 15 ? a.conv_state[size_t(k + past - 15) * a.channels + c] : 0.0f;
#pragma unroll
    for (uint32_t t = 0; t < SMALL_ROWS_MAX; t++) seq[15 + t] = t < tokens ? a.x[size_t(t) * a.channels + c] : 0.0f;
#pragma unroll
    for (uint32_t t = 0; t < SMALL_ROWS_MAX; t++) {
        if (t < tokens) {
            float acc = 0.0f;
#pragma unroll
            for (uint32_t k = 0; k < 15; k++) acc += taps[k] * seq[t + k];
            emit(t, silu_f(acc + taps[15] * seq[t + 15]));
        }
    }
}

// Waves 0-3 hold the 16 state rows (16 lanes a row) and compute the conv of the key head's q and k
// channels; wave 4 computes the conv of the 16 value channels and wave 5 the gates, so that no wave
// waits for memory twice before the first barrier.  Then the q/k norms of every token at once (one
// group of 16 lanes per token and vector), and the tokens in order with the next token's operands
// fetched from LDS while the current one's chain of sums runs.
constexpr int SMALL_THREADS = 384;

template <bool SNAPS>
__global__ __launch_bounds__(SMALL_THREADS) void deltanet_rows_small_kernel(SmallRowsArgs a) {
    __shared__ __attribute__((aligned(16))) float qk_lds[SMALL_ROWS_MAX][2 * K_DIM];  // per token: q then k, as [half][part][4]
    __shared__ float v_lds[SMALL_ROWS_MAX][16];
    __shared__ float gb_lds[SMALL_ROWS_MAX][2];   // decay, beta
    __shared__ float inv_lds[SMALL_ROWS_MAX][2];  // what q and k are multiplied by
    const uint32_t tid = threadIdx.x, part = tid & 15, row_in_wg = (tid >> 4) & 15;
    const uint32_t h = blockIdx.y, r0 = blockIdx.x * 16, row = r0 + row_in_wg;
    const uint32_t v_dim = a.p.v_dim, v_heads = a.p.v_heads, tokens = a.p.rows;
    const uint32_t kh = h / (v_heads / a.p.k_heads), key_size = a.p.k_heads * K_DIM;
    const bool live = tid < 256 && row < v_dim;
    float *sp = a.state + (size_t(h) * v_dim + (live ? row : 0)) * K_DIM + part * 8;
    float4 st[2];
    st[0] = live ? reinterpret_cast<const float4 *>(sp)[0] : make_float4(0, 0, 0, 0);
    st[1] = live ? reinterpret_cast<const float4 *>(sp)[1] : make_float4(0, 0, 0, 0);
    if (tid < 256) {
        const uint32_t e = tid & 127;
        const uint32_t slot = (tid < 128 ? 0 : K_DIM) + ((e & 7) >> 2) * 64 + (e >> 3) * 4 + (e & 3);
        conv_small(a, (tid < 128 ? 0 : key_size) + kh * K_DIM + e, [&](uint32_t t, float v) { qk_lds[t][slot] = v; });
    } else if (tid < 320) {
        const uint32_t i = tid - 256;
        if (i < 16 && r0 + i < v_dim) {
            conv_small(a, 2 * key_size + h * v_dim + r0 + i, [&](uint32_t t, float v) { v_lds[t][i] = v; });
        }
    } else {
        const uint32_t t = tid - 320;
        if (t < tokens) {
            fast_gates(a.a[size_t(t) * v_heads + h] + a.dt_bias[h], __expf(a.a_log[h]), a.b[size_t(t) * v_heads + h],
                       gb_lds[t][0], gb_lds[t][1]);
        }
    }
    __syncthreads();
    if (tid < 256) {
        // normalize_qk (src/cpu/deltanet.rs:133-146): group (tid / 16) takes token (group % 8), q or k
        const uint32_t t = row_in_wg & 7, which = row_in_wg >> 3;
        if (t < tokens) {
            const float4 lo = *reinterpret_cast<const float4 *>(qk_lds[t] + which * K_DIM + part * 4);
            const float4 hi = *reinterpret_cast<const float4 *>(qk_lds[t] + which * K_DIM + 64 + part * 4);
            const float sum = group_reduce<16>(dot4(lo, lo) + dot4(hi, hi), SumOp());
            const float scale = which == 0 ? 1.0f / sqrtf(float(K_DIM)) : 1.0f;
            if (part == 0) inv_lds[t][which] = scale * __builtin_amdgcn_rsqf(sum + a.p.eps);
        }
    }
    __syncthreads();
    if (tid >= 256) return;
    const size_t value_size = size_t(v_heads) * v_dim;
    float4 qn[2], kn[2];
    float gn, bn, vn, qin, kin;
    auto fetch = [&](uint32_t t) {
        qn[0] = *reinterpret_cast<const float4 *>(qk_lds[t] + part * 4);
        qn[1] = *reinterpret_cast<const float4 *>(qk_lds[t] + 64 + part * 4);
        kn[0] = *reinterpret_cast<const float4 *>(qk_lds[t] + K_DIM + part * 4);
        kn[1] = *reinterpret_cast<const float4 *>(qk_lds[t] + K_DIM + 64 + part * 4);
        gn = gb_lds[t][0], bn = gb_lds[t][1], vn = v_lds[t][row_in_wg];
        qin = inv_lds[t][0], kin = inv_lds[t][1];
    };
    fetch(0);
    for (uint32_t t = 0; t < tokens; t++) {
        float4 q[2], k[2];
        const float g = gn, beta = bn, v = vn, qi = qin, ki = kin;
#pragma unroll
        for (int c = 0; c < 2; c++) q[c] = qn[c], k[c] = kn[c];
        if (t + 1 < tokens) fetch(t + 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int c = 0; c < 2; c++) {
            q[c].x *= qi, q[c].y *= qi, q[c].z *= qi, q[c].w *= qi;
            k[c].x *= ki, k[c].y *= ki, k[c].z *= ki, k[c].w *= ki;
            st[c].x *= g, st[c].y *= g, st[c].z *= g, st[c].w *= g;
        }
        const float mem = group_reduce<16>(dot4(st[0], k[0]) + dot4(st[1], k[1]), SumOp());
        const float delta = (v - mem) * beta;
#pragma unroll
        for (int c = 0; c < 2; c++) {
            st[c].x += k[c].x * delta, st[c].y += k[c].y * delta, st[c].z += k[c].z * delta, st[c].w += k[c].w * delta;
        }
        const float o = group_reduce<16>(dot4(st[0], q[0]) + dot4(st[1], q[1]), SumOp());
        if (live) {
            if (part == 0) a.y[size_t(t) * value_size + size_t(h) * v_dim + row] = o;  // before the norm
            if constexpr (SNAPS) {
                float *snap = a.state_snaps + size_t(t) * v_heads * v_dim * K_DIM + (size_t(h) * v_dim + row) * K_DIM + part * 8;
                reinterpret_cast<float4 *>(snap)[0] = st[0];
                reinterpret_cast<float4 *>(snap)[1] = st[1];
            }
        }
    }
    if (live) reinterpret_cast<float4 *>(sp)[0] = st[0], reinterpret_cast<float4 *>(sp)[1] = st[1];
}

// After it.  Block b owns 16 channels of the conv: entry j of the conv state after token t is place
// t + 1 + j of (stored inputs, new inputs); the snapshots are written first, then, past a barrier
// (the entries are moved in place), the state after the last token.  The first blocks also norm the
// (token, head) pairs, one wave each, in place on y.
constexpr int TAIL_CHANNELS = 16;

__global__ __launch_bounds__(256) void deltanet_rows_small_tail_kernel(SmallRowsArgs a) {
    const uint32_t tid = threadIdx.x, lane = tid & 63;
    const uint32_t v_dim = a.p.v_dim, tokens = a.p.rows, past = a.p.kernel_size - 1, channels = a.channels;
    const uint32_t pair = blockIdx.x * 4 + (tid >> 6), pairs = tokens * a.p.v_heads;
    const bool has_pair = pair < pairs;
    float o[4];
    if (has_pair) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t d = lane + 64 * i;
            o[i] = d < v_dim ? a.y[size_t(pair) * v_dim + d] : 0.0f;
        }
    }
    const uint32_t c = blockIdx.x * TAIL_CHANNELS + (tid & 15);
    const float *stored = a.conv_state, *fresh = a.x;
    auto place = [&](uint32_t at) {  // `at` in (stored inputs, new inputs)
        return at < past ? stored[size_t(at) * channels + c] : fresh[size_t(at - past) * channels + c];
    };
    if (c < channels) {
        if (a.p.snapshots) {
            float *__restrict__ snaps = a.conv_snaps;
#pragma unroll 2
            for (uint32_t e = tid >> 4; e < tokens * past; e += 16) {  // e = t * past + j
                snaps[size_t(e) * channels + c] = place(e / past + 1 + e % past);
            }
        }
    }
    const uint32_t j = tid >> 4;  // past <= 15 < 16 entries a block can move at once
    const bool moves = c < channels && j < past;
    const float moved = moves ? place(tokens + j) : 0.0f;
    __syncthreads();
    if (moves) a.conv_state[size_t(j) * channels + c] = moved;
    if (has_pair) {
        float *yp = a.y + size_t(pair) * v_dim;
        const float *zp = a.z + size_t(pair) * v_dim;
        float total = 0.0f;
#pragma unroll
        for (int i = 0; i < 4; i++) total += group_reduce<64>(o[i] * o[i], SumOp());
        const float inv = 1.0f / sqrtf(total / float(v_dim) + a.p.eps);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t d = lane + 64 * i;
            if (d < v_dim) yp[d] = o[i] * (inv * a.norm_w[d]) * silu_f(zp[d]);
        }
    }
}

// ---- the same in one launch: a workgroup per value head ------------------------------------------
//
// Everything after the conv belongs to one value head, so with the head's whole state in one workgroup (64 KB in the
// registers of 1024 threads) the gated norm needs no second launch.  32 workgroups pull the 2.1 MB of the model's states
// through 32 CUs: reading and writing them back takes 3.5 us with the launch, against 2.5 us with 256 workgroups, and a
// second launch in a graph 1.6 us before it does anything.
// What is left over is the conv state, which is moved in place: the q and k channels of a key head are read by the
// workgroups of all of its value heads, and may be written only when the last of them has read.  Each of the four waves
// that hold these channels adds one to a counter of its own when its loads have come back (it has the inputs in registers,
// and nobody waits); the wave that finds the others there before it is the last and writes the channels and the zero back.
// The counters (4 per key head, zero before the first call, left at zero) come with the call: see
// saetta_deltanet_fused_sync_bytes.
// The snapshots are stored past the caches: as plain stores their lines, 2 MB of dirty data in the L2s per token, are
// written back when the kernel ends (4 rows 10.7 instead of 8.8 us).  More workgroups to a head, each writing a part of
// the snapshots, are no faster (9.2 us).
// A further token is vector instructions, sixteen waves' on one CU (without the snapshots' stores 8 rows take as long); a third
// of them were the three sums of q and k, which every group of lanes made for itself.  From SHARED_SCALES_FROM rows on a wave
// makes them for a token, for all, at the price of a barrier (4 rows with snapshots 8.62 -> 8.21 us, 8 rows 12.55 -> 10.94); one and
// two rows' are made by the waves of the conv.  (A head by 512 threads, 8 lanes a row: 11.27 for 8 rows, 2 rows slower.  The
// loop over the tokens rolled: 8.44, 11.55.)
// A launch this short is its chain of latencies, so what the chain waits for is looked at in the compiled code: the arguments
// come in one fetch, no load's use moves up between the requests, and nobody waits for a counter's answer but at the end.
// Measured per layer (30 layers in a graph, with the two-launch form before it): one token 7.1 -> 4.2 us (3.1 of them in the kernel, by
// clock stamps: 1.2 until the last wave has asked for its rows, 0.5 of which is their 64 KB at 64 bytes a cycle, 1.0 in the loop, 0.3
// for the norm, 0.3 until the stores are out), 4 rows with snapshots 11.3 -> 7.3; 8 rows 14.2 -> 10.3.
typedef float nt4 __attribute__((ext_vector_type(4)));
constexpr int HEAD_THREADS = 1024, HEAD_V_DIM = 128, HEAD_TAPS = 4;
constexpr int SHARED_SCALES_FROM = 3;
constexpr int HEAD_QK_WAVES = 2 * K_DIM / 64;  // waves that hold a key head's q and k channels

// M tokens (1..8), 128 value dims, 4 taps.
template <int M>
__global__ __launch_bounds__(HEAD_THREADS) void deltanet_head_kernel(SmallRowsArgs a, uint32_t *sync) {
    constexpr int PAST = HEAD_TAPS - 1;
    __shared__ __attribute__((aligned(16))) float in_lds[M][2 * K_DIM + HEAD_V_DIM];  // conv outputs: q, k, v
    __shared__ float gb_lds[M][2];                                                    // decay, beta
    __shared__ float o_lds[M][HEAD_V_DIM];
    __shared__ __attribute__((aligned(16))) float scale_lds[M][4];                    // a token's factors, see Factors
    __shared__ __attribute__((aligned(16))) float sum_lds[M][2][4];                   // PAIRED: |q|^2, |k|^2 and q.k of a wave's channels
    // One and two rows: a thread has the q and the k channel of a dim, so that the waves of the conv make the sums of q and k
    // too, half of a key head's channels each (made in the loop by every group of lanes they were a quarter of its instructions).
    constexpr bool PAIRED = M < SHARED_SCALES_FROM;
    constexpr uint32_t QK_WAVES = PAIRED ? HEAD_QK_WAVES / 2 : HEAD_QK_WAVES;
    const uint32_t tid = threadIdx.x, lane = tid & 63, part = lane & 15;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t v_heads = a.p.v_heads, per_key = gridDim.y, kh = blockIdx.x, h = kh * per_key + blockIdx.y;
    // (the arguments at once: left alone the compiler fetches them in four lots, each waited for)
    asm volatile("" ::"s"(a.x), "s"(a.w), "s"(a.conv_state), "s"(a.a), "s"(a.b), "s"(a.a_log), "s"(a.dt_bias), "s"(a.state), "s"(a.z), "s"(a.norm_w), "s"(sync),
                 "s"(a.p.k_heads), "s"(v_heads), "s"(per_key), "s"(a.channels), "s"(a.p.snapshots), "s"(a.p.eps));
    const uint32_t key_size = a.p.k_heads * K_DIM;
    const size_t value_size = size_t(v_heads) * HEAD_V_DIM;
    constexpr uint32_t CONV_WAVES = QK_WAVES + HEAD_V_DIM / 64;
    const bool conv = wave < CONV_WAVES;  // thread = channel: q (the first two waves), k (the next two; PAIRED: q and k), v (two)
    const uint32_t k_channel = key_size + kh * K_DIM + (tid & 127);
    const uint32_t c = wave < 2 ? kh * K_DIM + tid : wave < QK_WAVES ? k_channel : 2 * key_size + h * HEAD_V_DIM + (tid & 127);
    const uint32_t slot = wave < QK_WAVES ? tid : 2 * K_DIM + (tid & 127);

    // Everything is requested before anything is used, the conv's inputs first: loads return in order.
    struct Channel {
        float seq[PAST + M];  // stored inputs, oldest first, then the new ones
        float4 taps;
        __device__ __forceinline__ void request(const SmallRowsArgs &a, uint32_t c) {
            taps = *reinterpret_cast<const float4 *>(a.w + size_t(c) * HEAD_TAPS);
#pragma unroll
            for (int k = 0; k < PAST; k++) seq[k] = a.conv_state[size_t(k) * a.channels + c];
#pragma unroll
            for (int t = 0; t < M; t++) seq[PAST + t] = a.x[size_t(t) * a.channels + c];
        }
        __device__ __forceinline__ float output(int t) const {  // (the sum as the single-token conv adds it: oldest first)
            float acc = taps.x * seq[t];
            acc += taps.y * seq[t + 1];
            acc += taps.z * seq[t + 2];
            return silu_f(acc + taps.w * seq[t + 3]);
        }
        __device__ __forceinline__ void keep_snapshots(const SmallRowsArgs &a, uint32_t c) const {
            // after token t the conv state is the inputs t + 1 .. t + PAST of the sequence
#pragma unroll
            for (int t = 0; t < M; t++) {
#pragma unroll
                for (int j = 0; j < PAST; j++) __builtin_nontemporal_store(seq[t + 1 + j], a.conv_snaps + (size_t(t) * PAST + j) * a.channels + c);
            }
        }
        __device__ __forceinline__ void keep_state(const SmallRowsArgs &a, uint32_t c) const {
#pragma unroll
            for (int j = 0; j < PAST; j++) a.conv_state[size_t(j) * a.channels + c] = seq[M + j];
        }
    };
    Channel own, key;  // (key: PAIRED, the k channel beside the q channel)
    const bool paired = PAIRED && wave < QK_WAVES;
    if (conv) own.request(a, c);
    if (paired) key.request(a, k_channel);
    float gate_a, gate_b, gate_log, gate_bias;
    asm("" : "=v"(gate_a), "=v"(gate_b), "=v"(gate_log), "=v"(gate_bias));  // (no constants: sums of them would move into the branch, behind a wait)
    const bool gates = wave == CONV_WAVES && lane < M;
    if (gates) {
        // (vector loads: a scalar load is waited for on the spot, and the wave's rows of the state are asked for behind it)
        uint32_t gate_h = h;
        asm volatile("" : "+v"(gate_h));
        gate_a = a.a[size_t(lane) * v_heads + gate_h], gate_b = a.b[size_t(lane) * v_heads + gate_h];
        gate_log = a.a_log[gate_h], gate_bias = a.dt_bias[gate_h];
    }
    // 16 lanes a row of the state, dims 4 part .. + 3 and 64 + 4 part .. + 3; rows 8 wave + lane / 16 and four further
    const uint32_t row = 8 * wave + (lane >> 4);
    float *sp = a.state + (size_t(h) * HEAD_V_DIM + row) * K_DIM + part * 4;
    float4 st[2][2];
#pragma unroll
    for (int r = 0; r < 2; r++) {
#pragma unroll
        for (int i = 0; i < 2; i++) st[r][i] = *reinterpret_cast<const float4 *>(sp + r * 4 * K_DIM + i * 64);
    }
    const uint32_t out_t = tid / HEAD_V_DIM, out_d = tid % HEAD_V_DIM;  // the output this thread finishes (out_t < M)
    float z = 0.0f, norm = 0.0f;
    if (out_t < M) {
        z = a.z[size_t(out_t) * value_size + size_t(h) * HEAD_V_DIM + out_d];
        norm = a.norm_w[out_d];
    }

    if (paired) {
#pragma unroll
        for (int t = 0; t < M; t++) {
            const float y = own.output(t), k = key.output(t);
            in_lds[t][slot] = y, in_lds[t][K_DIM + slot] = k;
            const float qq = group_reduce<64>(y * y, SumOp()), kk = group_reduce<64>(k * k, SumOp()), kq = group_reduce<64>(y * k, SumOp());
            if (lane == 0) *reinterpret_cast<float4 *>(sum_lds[t][wave]) = make_float4(qq, kk, kq, 0.0f);
        }
    } else if (conv) {
#pragma unroll
        for (int t = 0; t < M; t++) in_lds[t][slot] = own.output(t);
    }
    if (gates) fast_gates(gate_a + gate_bias, __expf(gate_log), gate_b, gb_lds[lane][0], gb_lds[lane][1]);
    __syncthreads();

    // This wave's conv inputs are in registers (its outputs above were made of them).
    // (The counter's place as a lane's own: where it is known to be the wave's the compiler adds for all lanes at once and
    // hands the answer out right there, which makes the wave wait for it.)
    uint32_t before = 0, counter = kh * HEAD_QK_WAVES + wave;
    asm volatile("" : "+v"(counter));
    if (wave < QK_WAVES && lane == 0) before = atomicAdd(sync + counter, 1u);

    // With q and k as the conv gives them, ki and qi what they are multiplied by:  delta / ki = (v - x S.k) y,
    // o = z S.q + w delta,  S = g S + delta k  for x = g ki, y = beta ki, z = qi g, w = qi (k.q)  (o of the updated state: (g S +
    // delta k^T) q = g S q + delta (k.q)).
    auto factors = [&](float qq, float kk, float kq, float g, float beta) {
        const float qi = (1.0f / sqrtf(float(K_DIM))) * __builtin_amdgcn_rsqf(qq + a.p.eps), ki = __builtin_amdgcn_rsqf(kk + a.p.eps);
        return make_float4(g * ki, beta * ki, qi * g, qi * kq);
    };
    // |q|^2, |k|^2 and q.k of token t by wave 15 - t (the first have the counters' answers to wait for), for all
    if constexpr (M >= SHARED_SCALES_FROM) {
        const uint32_t t = HEAD_THREADS / 64 - 1 - wave;
        if (t < uint32_t(M)) {
            const float2 q = *reinterpret_cast<const float2 *>(&in_lds[t][2 * lane]), k = *reinterpret_cast<const float2 *>(&in_lds[t][K_DIM + 2 * lane]);
            const float qq = group_reduce<64>(q.x * q.x + q.y * q.y, SumOp()), kk = group_reduce<64>(k.x * k.x + k.y * k.y, SumOp());
            const float kq = group_reduce<64>(q.x * k.x + q.y * k.y, SumOp());
            if (lane == 0) *reinterpret_cast<float4 *>(scale_lds[t]) = factors(qq, kk, kq, gb_lds[t][0], gb_lds[t][1]);
        }
        __syncthreads();
    }

#pragma unroll
    for (int t = 0; t < M; t++) {
        float4 q[2], k[2];
#pragma unroll
        for (int i = 0; i < 2; i++) {
            q[i] = *reinterpret_cast<const float4 *>(&in_lds[t][64 * i + part * 4]);
            k[i] = *reinterpret_cast<const float4 *>(&in_lds[t][K_DIM + 64 * i + part * 4]);
        }
        const float g = gb_lds[t][0];
        float4 f;
        if constexpr (PAIRED) {
            const float4 x = *reinterpret_cast<const float4 *>(sum_lds[t][0]), y = *reinterpret_cast<const float4 *>(sum_lds[t][1]);
            f = factors(x.x + y.x, x.y + y.y, x.z + y.z, g, gb_lds[t][1]);
        } else {
            f = *reinterpret_cast<const float4 *>(scale_lds[t]);
        }
        // One round of 16-lane sums per token: S.k and S.q of both rows, S before the decay and the update.
        auto along = [&](const float4 (&s)[2], const float4 (&x)[2]) { return group_reduce<16>(dot4(s[0], x[0]) + dot4(s[1], x[1]), SumOp()); };
        float o[2];
#pragma unroll
        for (int r = 0; r < 2; r++) {
            const float sk = along(st[r], k), sq = along(st[r], q);
            const float delta = (in_lds[t][2 * K_DIM + row + 4 * r] - f.x * sk) * f.y;
            o[r] = f.z * sq + f.w * delta;
#pragma unroll
            for (int i = 0; i < 2; i++) {
                st[r][i].x = g * st[r][i].x + delta * k[i].x, st[r][i].y = g * st[r][i].y + delta * k[i].y;
                st[r][i].z = g * st[r][i].z + delta * k[i].z, st[r][i].w = g * st[r][i].w + delta * k[i].w;
            }
        }
        if (part < 2) o_lds[t][row + 4 * part] = part == 0 ? o[0] : o[1];
        if (a.p.snapshots) {
            float *snap = a.state_snaps + size_t(t) * value_size * K_DIM + (size_t(h) * HEAD_V_DIM + row) * K_DIM + part * 4;
#pragma unroll
            for (int r = 0; r < 2; r++) {
#pragma unroll
                for (int i = 0; i < 2; i++) __builtin_nontemporal_store(__builtin_bit_cast(nt4, st[r][i]), reinterpret_cast<nt4 *>(snap + r * 4 * K_DIM + i * 64));
            }
        }
    }
#pragma unroll
    for (int r = 0; r < 2; r++) {
#pragma unroll
        for (int i = 0; i < 2; i++) *reinterpret_cast<float4 *>(sp + r * 4 * K_DIM + i * 64) = st[r][i];
    }
    float gate = silu_f(z);
    asm volatile("" : "+v"(gate));  // (here, and not behind the barrier)
    __syncthreads();
    if (out_t < M) {
        // the head's outputs of the token, two per lane of either of its waves
        const float o0 = o_lds[out_t][lane], o1 = o_lds[out_t][lane + 64];
        const float total = group_reduce<64>(o0 * o0 + o1 * o1, SumOp());
        const float inv = inverse_root(total * (1.0f / float(HEAD_V_DIM)) + a.p.eps);
        a.y[size_t(out_t) * value_size + size_t(h) * HEAD_V_DIM + out_d] = (out_d < 64 ? o0 : o1) * (inv * norm) * gate;
    }
    if (conv) {
        const bool mine = wave >= QK_WAVES;
        if (a.p.snapshots && (mine || h == kh * per_key)) {
            own.keep_snapshots(a, c);
            if (paired) key.keep_snapshots(a, k_channel);
        }
        if (mine || uint32_t(__builtin_amdgcn_readfirstlane(before)) == per_key - 1) {
            own.keep_state(a, c);
            if (paired) key.keep_state(a, k_channel);
            if (!mine && lane == 0) __hip_atomic_store(sync + kh * HEAD_QK_WAVES + wave, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
}

template <int M>
void launch_head_rows(const SmallRowsArgs &args, uint32_t *sync, hipStream_t stream) {
    if (args.p.rows == uint32_t(M)) {
        launch(deltanet_head_kernel<M>, dim3(args.p.k_heads, args.p.v_heads / args.p.k_heads), HEAD_THREADS, 0, stream, args, sync);
    } else if constexpr (M < SMALL_ROWS_MAX) {
        launch_head_rows<M + 1>(args, sync, stream);
    }
}

void launch_small_rows(const SmallRowsArgs &args, uint32_t *sync, hipStream_t stream) {
    const saetta_rows_fused_params &p = args.p;
    if (sync && p.v_dim == HEAD_V_DIM && p.kernel_size == HEAD_TAPS && aligned(args.w, 16) && p.v_heads / p.k_heads < 65536 && p.eps >= INVERSE_ROOT_FROM) {
        launch_head_rows<1>(args, sync, stream);
        return;
    }
    const dim3 grid((p.v_dim + 15) / 16, p.v_heads);
    if (p.snapshots) {
        launch(deltanet_rows_small_kernel<true>, grid, SMALL_THREADS, 0, stream, args);
    } else {
        launch(deltanet_rows_small_kernel<false>, grid, SMALL_THREADS, 0, stream, args);
    }
    const uint32_t pair_blocks = (p.rows * p.v_heads + 3) / 4, chan_blocks = (args.channels + TAIL_CHANNELS - 1) / TAIL_CHANNELS;
    launch(deltanet_rows_small_tail_kernel, pair_blocks > chan_blocks ? pair_blocks : chan_blocks, 256, 0, stream, args);
}

}  // namespace

int setup_deltanet() {
    if (int rc = load_kernel(reinterpret_cast<const void *>(deltanet_step_kernel))) return rc;
    return setup_deltanet_chunk();
}
}  // namespace saetta

using namespace saetta;

extern "C" int saetta_deltanet_conv(saetta_stream_t stream, const float *x, const float *w, float *state, float *out,
                                    saetta_conv_params p) {
    SAETTA_REQUIRE(x && w && state && out, SAETTA_E_NULL, "deltanet_conv: null buffer");
    // (a kernel of one tap has no state; the reference's conv_step cannot run it either)
    SAETTA_REQUIRE(p.kernel_size >= 2 && p.kernel_size <= 16, SAETTA_E_SHAPE, "deltanet_conv: kernel size %u (2..16)",
                   p.kernel_size);
    if (int rc = ensure_device()) return rc;
    if (p.channels == 0) return SAETTA_OK;
    launch(deltanet_conv_kernel, (p.channels + 255) / 256, 256, 0, as_stream(stream), x, w, state, out, p);
    return launch_status("deltanet_conv");
}

extern "C" int saetta_deltanet_step(saetta_stream_t stream, const float *q, const float *k, const float *v,
                                    const float *a, const float *b, const float *a_log, const float *dt_bias,
                                    float *state, const float *z, const float *norm_w, float *y,
                                    saetta_step_params p) {
    SAETTA_REQUIRE(q && k && v && a && b && a_log && dt_bias && state && z && norm_w && y, SAETTA_E_NULL,
                   "deltanet_step: null buffer");
    SAETTA_REQUIRE(p.k_heads > 0 && p.v_heads > 0 && p.v_heads % p.k_heads == 0, SAETTA_E_SHAPE,
                   "deltanet_step: %u value heads over %u key heads", p.v_heads, p.k_heads);
    SAETTA_REQUIRE(p.v_dim >= 1 && p.v_dim <= 32 * MAX_ROWS_PER_LANE, SAETTA_E_SHAPE,
                   "deltanet_step: value dim %u (1..256); the key dim is 128", p.v_dim);
    SAETTA_REQUIRE(aligned(q, 16) && aligned(k, 16) && aligned(state, 16), SAETTA_E_ALIGN,
                   "deltanet_step: q, k and the state must be 16-byte aligned");
    if (int rc = ensure_device()) return rc;
    // q, k and v as the conv leaves them (one array, q | k | v: what the reference's layer passes,
    // src/cpu/deltanet.rs:80-83) take the kernels of saetta_deltanet_rows with one token: 8 workgroups
    // per value head instead of one.  deltanet_step_kernel is kept for vectors that lie apart.
    const size_t key_size = size_t(p.k_heads) * K_DIM;
    if (k == q + key_size && v == k + key_size && p.v_dim % 4 == 0) {
        const saetta_rows_step_params rp{p.k_heads, p.v_heads, p.v_dim, 1, p.eps, 0};
        return saetta_deltanet_rows(stream, q, a, b, a_log, dt_bias, state, z, norm_w, y, nullptr, rp);
    }
    StepArgs args{q, k, v, a, b, a_log, dt_bias, state, z, norm_w, y, p};
    launch(deltanet_step_kernel, p.v_heads, STEP_THREADS, 0, as_stream(stream), args);
    return launch_status("deltanet_step");
}

extern "C" int saetta_deltanet_conv_rows(saetta_stream_t stream, const float *x, const float *w, float *state,
                                         float *out, float *snaps, saetta_conv_rows_params p) {
    SAETTA_REQUIRE(x && w && state && out, SAETTA_E_NULL, "deltanet_conv_rows: null buffer");
    SAETTA_REQUIRE(!p.snapshots || snaps, SAETTA_E_NULL, "deltanet_conv_rows: snapshots asked for, no buffer");
    SAETTA_REQUIRE(p.kernel_size >= 2 && p.kernel_size <= 16, SAETTA_E_SHAPE,
                   "deltanet_conv_rows: kernel size %u (2..16)", p.kernel_size);
    SAETTA_REQUIRE(p.tokens <= (1u << 20), SAETTA_E_SHAPE, "deltanet_conv_rows: %u tokens", p.tokens);
    if (int rc = ensure_device()) return rc;
    if (p.channels == 0 || p.tokens == 0) return SAETTA_OK;
    const dim3 grid((p.channels + 255) / 256, (p.tokens + CONV_TILE - 1) / CONV_TILE);
    // (four channels a thread: a verify step's few rows want the workgroups; 16 tokens take 4.1 us this way and 6.1 the other)
    const bool by_four = p.tokens >= CONV4_FROM && p.channels % 4 == 0 && aligned(x, 16) && aligned(w, 16) && aligned(state, 16) && aligned(out, 16) &&
                         (!p.snapshots || aligned(snaps, 16));
    if (p.kernel_size == CONV4_TAPS && by_four) {
        launch(deltanet_conv_rows4_kernel, dim3((p.channels / 4 + 255) / 256, (p.tokens + CONV4_TILE - 1) / CONV4_TILE), 256, 0, as_stream(stream), x, w, state, out, snaps, p);
        tag_launch(LAUNCH_CONV, 0, 0);
    } else if (p.kernel_size == 4) {
        launch(deltanet_conv_rows_kernel<4>, grid, 256, 0, as_stream(stream), x, w, state, out, snaps, p);
    } else if (p.kernel_size == 2) {
        launch(deltanet_conv_rows_kernel<2>, grid, 256, 0, as_stream(stream), x, w, state, out, snaps, p);
    } else {
        launch(deltanet_conv_rows_kernel<0>, grid, 256, 0, as_stream(stream), x, w, state, out, snaps, p);
    }
    return launch_status("deltanet_conv_rows");
}

extern "C" size_t saetta_deltanet_rows_workspace_bytes(saetta_rows_step_params p) { return deltanet_chunk_workspace_bytes(p); }

extern "C" int saetta_deltanet_rows(saetta_stream_t stream, const float *mixed, const float *a, const float *b,
                                    const float *a_log, const float *dt_bias, float *state, const float *z,
                                    const float *norm_w, float *y, float *snaps, saetta_rows_step_params p) {
    return saetta_deltanet_rows_ws(stream, mixed, a, b, a_log, dt_bias, state, z, norm_w, y, snaps, p, nullptr, 0);
}

extern "C" int saetta_deltanet_rows_ws(saetta_stream_t stream, const float *mixed, const float *a, const float *b,
                                       const float *a_log, const float *dt_bias, float *state, const float *z,
                                       const float *norm_w, float *y, float *snaps, saetta_rows_step_params p,
                                       void *workspace, size_t workspace_size) {
    SAETTA_REQUIRE(mixed && a && b && a_log && dt_bias && state && z && norm_w && y, SAETTA_E_NULL,
                   "deltanet_rows: null buffer");
    SAETTA_REQUIRE(!p.snapshots || snaps, SAETTA_E_NULL, "deltanet_rows: snapshots asked for, no buffer");
    SAETTA_REQUIRE(p.k_heads > 0 && p.v_heads > 0 && p.v_heads % p.k_heads == 0, SAETTA_E_SHAPE,
                   "deltanet_rows: %u value heads over %u key heads", p.v_heads, p.k_heads);
    SAETTA_REQUIRE(p.v_dim >= 1 && p.v_dim <= 256 && p.v_dim % 4 == 0, SAETTA_E_SHAPE,
                   "deltanet_rows: value dim %u (a multiple of 4 up to 256); the key dim is 128", p.v_dim);
    SAETTA_REQUIRE(p.tokens <= (1u << 20), SAETTA_E_SHAPE, "deltanet_rows: %u tokens", p.tokens);
    SAETTA_REQUIRE(aligned(mixed, 16) && aligned(state, 16) && (!p.snapshots || aligned(snaps, 16)), SAETTA_E_ALIGN,
                   "deltanet_rows: mixed, the state and the snapshots must be 16-byte aligned");
    if (int rc = ensure_device()) return rc;
    if (p.tokens == 0) return SAETTA_OK;
    const uint32_t channels = 2 * p.k_heads * K_DIM + p.v_heads * p.v_dim;
    // A prefill chunk (128 tokens and more, no snapshots) whose caller brings a workspace: the delta rule in
    // blocks of 64 tokens on the matrix cores.  Without a workspace the call keeps to the token-by-token
    // kernels: the library holds no buffer of its own here, so calls on different streams share nothing.
    const size_t need = deltanet_chunk_workspace_bytes(p);
    const bool blocks = need > 0 && workspace != nullptr;
    if (blocks) {
        SAETTA_REQUIRE(workspace_size >= need && aligned(workspace, 16), SAETTA_E_SCRATCH,
                       "deltanet_rows: workspace of %zu bytes, %zu needed (16-byte aligned)", workspace_size, need);
        if (int rc = run_deltanet_chunk(as_stream(stream), mixed, a, b, a_log, dt_bias, state, y, p, channels, workspace)) return rc;
    } else {
        RowsArgs args{mixed, a, b, a_log, dt_bias, state, y, snaps, p, channels};
        constexpr int LANES = ROWS_LANES_PER_ROW, ROWS_PER_WG = 256 / LANES;
        const dim3 grid((p.v_dim + ROWS_PER_WG - 1) / ROWS_PER_WG, p.v_heads);
        if (p.snapshots) {
            launch(deltanet_rows_kernel<true, LANES>, grid, 256, 0, as_stream(stream), args);
        } else {
            launch(deltanet_rows_kernel<false, LANES>, grid, 256, 0, as_stream(stream), args);
        }
    }
    const uint32_t pairs = p.tokens * p.v_heads;
    const bool wide = blocks && aligned(y, 16) && aligned(z, 16) && aligned(norm_w, 16);
    if (wide && p.v_dim == 128) {
        launch(deltanet_gated_norm_wide_kernel<32>, (pairs * 32 + 255) / 256, 256, 0, as_stream(stream), y, z, norm_w, pairs, p.eps);
    } else if (wide && p.v_dim == 64) {
        launch(deltanet_gated_norm_wide_kernel<16>, (pairs * 16 + 255) / 256, 256, 0, as_stream(stream), y, z, norm_w, pairs, p.eps);
    } else if (wide && p.v_dim == 256) {
        launch(deltanet_gated_norm_wide_kernel<64>, (pairs * 64 + 255) / 256, 256, 0, as_stream(stream), y, z, norm_w, pairs, p.eps);
    } else {
        launch(deltanet_gated_norm_rows_kernel, (pairs + 3) / 4, 256, 0, as_stream(stream), y, z, norm_w, pairs, p.v_dim, p.eps);
    }
    return launch_status("deltanet_rows");
}

extern "C" size_t saetta_deltanet_fused_sync_bytes(uint32_t k_heads) { return size_t(k_heads) * HEAD_QK_WAVES * sizeof(uint32_t); }

extern "C" int saetta_deltanet_token(saetta_stream_t stream, const float *x, const float *w, float *conv_state,
                                     const float *a, const float *b, const float *a_log, const float *dt_bias,
                                     float *state, const float *z, const float *norm_w, float *y,
                                     saetta_conv_params cp, saetta_step_params sp) {
    return saetta_deltanet_token_sync(stream, x, w, conv_state, a, b, a_log, dt_bias, state, z, norm_w, y, cp, sp, nullptr);
}

extern "C" int saetta_deltanet_token_sync(saetta_stream_t stream, const float *x, const float *w, float *conv_state,
                                          const float *a, const float *b, const float *a_log, const float *dt_bias,
                                          float *state, const float *z, const float *norm_w, float *y,
                                          saetta_conv_params cp, saetta_step_params sp, uint32_t *sync) {
    SAETTA_REQUIRE(x && w && conv_state && a && b && a_log && dt_bias && state && z && norm_w && y, SAETTA_E_NULL,
                   "deltanet_token: null buffer");
    SAETTA_REQUIRE(cp.kernel_size >= 2 && cp.kernel_size <= 16, SAETTA_E_SHAPE, "deltanet_token: kernel size %u (2..16)",
                   cp.kernel_size);
    SAETTA_REQUIRE(sp.k_heads > 0 && sp.v_heads > 0 && sp.v_heads % sp.k_heads == 0, SAETTA_E_SHAPE,
                   "deltanet_token: %u value heads over %u key heads", sp.v_heads, sp.k_heads);
    SAETTA_REQUIRE(sp.v_dim >= 1 && sp.v_dim <= 256, SAETTA_E_SHAPE, "deltanet_token: value dim %u (1..256); the key dim is 128",
                   sp.v_dim);
    SAETTA_REQUIRE(cp.channels == 2 * sp.k_heads * K_DIM + sp.v_heads * sp.v_dim, SAETTA_E_SHAPE,
                   "deltanet_token: %u channels, the heads make %u", cp.channels, 2 * sp.k_heads * K_DIM + sp.v_heads * sp.v_dim);
    SAETTA_REQUIRE(aligned(state, 16) && aligned(sync, 4), SAETTA_E_ALIGN, "deltanet_token: the state must be 16-byte aligned");
    if (int rc = ensure_device()) return rc;
    const saetta_rows_fused_params p{sp.k_heads, sp.v_heads, sp.v_dim, cp.kernel_size, sp.eps, 1, 0};
    SmallRowsArgs args{x, w, conv_state, a, b, a_log, dt_bias, state, z, norm_w, y, nullptr, nullptr, p, cp.channels};
    launch_small_rows(args, sync, as_stream(stream));
    return launch_status("deltanet_token");
}

extern "C" int saetta_deltanet_rows_fused(saetta_stream_t stream, const float *x, const float *w, float *conv_state,
                                          const float *a, const float *b, const float *a_log, const float *dt_bias,
                                          float *state, const float *z, const float *norm_w, float *y,
                                          float *conv_snaps, float *state_snaps, saetta_rows_fused_params p) {
    return saetta_deltanet_rows_fused_sync(stream, x, w, conv_state, a, b, a_log, dt_bias, state, z, norm_w, y, conv_snaps,
                                           state_snaps, p, nullptr);
}

extern "C" int saetta_deltanet_rows_fused_sync(saetta_stream_t stream, const float *x, const float *w, float *conv_state,
                                               const float *a, const float *b, const float *a_log, const float *dt_bias,
                                               float *state, const float *z, const float *norm_w, float *y,
                                               float *conv_snaps, float *state_snaps, saetta_rows_fused_params p,
                                               uint32_t *sync) {
    SAETTA_REQUIRE(x && w && conv_state && a && b && a_log && dt_bias && state && z && norm_w && y, SAETTA_E_NULL,
                   "deltanet_rows_fused: null buffer");
    SAETTA_REQUIRE(!p.snapshots || (conv_snaps && state_snaps), SAETTA_E_NULL,
                   "deltanet_rows_fused: snapshots asked for, no buffers");
    SAETTA_REQUIRE(p.rows <= SMALL_ROWS_MAX, SAETTA_E_SHAPE, "deltanet_rows_fused: %u rows (up to 8)", p.rows);
    SAETTA_REQUIRE(p.kernel_size >= 2 && p.kernel_size <= 16, SAETTA_E_SHAPE,
                   "deltanet_rows_fused: kernel size %u (2..16)", p.kernel_size);
    SAETTA_REQUIRE(p.k_heads > 0 && p.v_heads > 0 && p.v_heads % p.k_heads == 0, SAETTA_E_SHAPE,
                   "deltanet_rows_fused: %u value heads over %u key heads", p.v_heads, p.k_heads);
    SAETTA_REQUIRE(p.v_dim >= 1 && p.v_dim <= 256, SAETTA_E_SHAPE,
                   "deltanet_rows_fused: value dim %u (1..256); the key dim is 128", p.v_dim);
    SAETTA_REQUIRE(aligned(state, 16) && (!p.snapshots || aligned(state_snaps, 16)) && aligned(sync, 4), SAETTA_E_ALIGN,
                   "deltanet_rows_fused: the state and its snapshots must be 16-byte aligned");
    if (int rc = ensure_device()) return rc;
    if (p.rows == 0) return SAETTA_OK;
    const uint32_t channels = 2 * p.k_heads * K_DIM + p.v_heads * p.v_dim;
    SmallRowsArgs args{x, w, conv_state, a, b, a_log, dt_bias, state, z, norm_w, y, conv_snaps, state_snaps, p, channels};
    launch_small_rows(args, sync, as_stream(stream));
    return launch_status("deltanet_rows_fused");
}
