// Flash-style causal prefill attention for gfx950 (MI355X).
//
// What it computes (reference: attention_prefill::encode,
// src/attention_prefill.rs:39-72, kernel attention_fa<TQ>,
// kernels/attention_prefill.metal:38-169; over a quantized cache
// src/prefill.rs:1735-1776, kernels/attention_rows_q.metal:55-344): for the
// chunk's token i and each of the 16 q heads
//     out[i, h] = softmax(q[i, h] K^T * scale) V * sigmoid(gate[i, h])
// over keys 0 ..= pos + i, 8 q heads sharing one kv head, head dim 256.
// q is f16; the cache is f16 or 8/4-bit codes read in place.  A quantized
// cache is seen "through half": every value is f16(f32(s)*code + f32(z)),
// exactly what round_trip_as_half (src/kv_quant.rs:119-125) gives the CPU path.
//
// Two kernels, and a third where a tile's keys are taken in parts; prefill_small_kernel instead of them for short chunks (further down: the passes of the reference's other
// route to the same output, AttGemm of src/attention_gemm.rs, on the same images, block by block of 1024 keys).
//
// prefill_prepare_kernel<16|8|4> turns the keys and values the chunk can see into
// f16 tile images in a workspace, one image per (kv head, block of 32 keys): the K tile
// [32 keys][256 dims] and the transposed V^T tile [256 dims][32 keys], laid out byte for
// byte as the attention kernel wants them in LDS (padded rows, V^T keys in the order the
// MFMA accumulator hands them out).  The dequantization happens here, once per key, with
// exactly the arithmetic of round_trip_as_half, instead of once per workgroup that walks
// the key; it costs one pass over the cache (a few microseconds).
//
// attention_prefill_kernel: workgroup (token tile of 16 or 32, kv head), 8 waves, two to a SIMD; a row group is 4 tokens x 8 heads =
// 32 query rows, one 32-row MFMA tile, and belongs to two waves that take alternate key blocks, or, in a tile of 32, to one.  Keys are
// walked in blocks of 32 whose images are copied global -> LDS by global_load_lds_dwordx4 (no vector registers, no vector ALU) into a
// ring of four places for K parts and four for V^T parts.  Every wave computes with v_mfma_f32_32x32x16_f16
//     S^T = K Q^T      (A = K rows from LDS, B = Q^T held in registers)
//     O^T += V^T P^T   (A = V^T rows from LDS, B = P^T from the S^T registers)
// Both products are transposed so that a lane always owns one query row: in the 32x32
// accumulator layout a lane holds column l % 32, so the row's running max and sum, the
// rescale of O and the final 1/l and gate are plain per-lane values and the softmax needs one
// cross-lane exchange per block.  A wave's step is its block's softmax (vector ALU) and one stream of MFMAs that adds the block to
// O and makes the scores of its next; the two waves of a SIMD take them in opposite order, so that one's softmax runs
// under the other's MFMAs, with one barrier per step.  The running max is only raised when a block exceeds it by
// more than 2^8 (lazy rescale), so O is rarely rescaled.  Tiles are taken heaviest first, one workgroup per CU, on demand.
#include "common.hpp"
#include "lanes.hpp"
#include "owned_workspace.hpp"

#include <algorithm>
#include <initializer_list>
#include <map>
#include <mutex>
#include <utility>

namespace saetta {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2_ __attribute__((ext_vector_type(2)));
typedef float float2_ __attribute__((ext_vector_type(2)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr int DIM = SAETTA_HEAD_DIM;
constexpr int PREP_THREADS = 256;       // the prepare kernel's workgroup
constexpr int WAVES = 8;                // 4 row groups x 2 waves that take alternate key blocks
constexpr int THREADS = 64 * WAVES;
constexpr int TQ = 16;                  // tokens per workgroup: a row group is 4 tokens x 8 heads = 32 rows
constexpr int WIDE_TQ = 32;             // ... of a wide tile, a row group a wave
constexpr int BK = 32;                  // keys per block
// One key block's image: the K tile and the V^T tile in MFMA fragment order, 16 KB each.  A
// fragment is what one ds_read_b128 of a wave fetches: 64 lanes x 16 bytes, lane (col, hf) at
// byte 512 hf + 16 col, so every fragment read is one contiguous kilobyte.
//   K fragment stp (0..15):           lane holds dims 16 stp + 8 hf .. + 7 of key col
//   V^T fragment 2 mt + sp (0..15):   lane holds key positions 16 sp + 8 hf .. + 7 of dim 32 mt + col
constexpr int PART_BYTES = BK * DIM * 2;
constexpr int IMG_BYTES = 2 * PART_BYTES;
constexpr float NO_SCORE = -1e30f;
// (EXACT: not in the first EXACT_BLOCKS blocks of a row's keys, see prefill_tile)
constexpr uint32_t EXACT_BLOCKS = 8;
constexpr float TAU = 8.0f;  // the reference max is raised only past this many powers of two

struct PrepareArgs {
    const void *kdata;
    const void *vdata;
    const uint16_t *kscales, *kbiases, *vscales, *vbiases;
    unsigned char *images;  // [kv head][block][IMG_BYTES]
    uint32_t kv_heads, nblocks;
    uint32_t key_limit;  // pos + tokens: rows the cache holds; keys from here on are zeros
    uint32_t *tiles_taken;  // behind the images (or nullptr): the attention kernel's count of tiles handed out, set to 0 here
};

struct PrefillArgs {
    const uint16_t *q;  // f16 [tokens][heads][256]
    const unsigned char *images;
    const float *q_and_gate;
    float *out;
    uint32_t heads, kv_heads, pos, tokens;
    float scale;
    uint32_t nblocks;  // images per kv head
    uint32_t *tiles_taken;  // tiles handed out past every workgroup's first (zero at the start: the prepare kernel's doing)
    // Split keys (attention_prefill_kernel<true, ..>): a tile's keys are taken in parts of `part_blocks` blocks, each of which
    // leaves its unnormalised O and (m, l) in the workspace for prefill_merge_kernel.
    uint32_t part_blocks;
    float *part_o;   // [part][tile][kv head][8 waves][16][64 lanes][4]: the accumulators as they are
    float *part_ml;  // [part][tile][kv head][4 row groups][32 rows][m, l]
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void *p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, int(bytes), 0x00020000);
}

template <int BITS>
constexpr int row_bytes() {
    return BITS == 16 ? 512 : BITS * 32;
}

__device__ __forceinline__ uint32_t pack_half2(float a, float b) {
    half2_ h = {(_Float16)a, (_Float16)b};
    return __builtin_bit_cast(uint32_t, h);
}

// f16(f32(s) * code + f32(z)): s * code is exact in f32, so the fma rounds as the CPU's
// multiply-then-add does, and the conversion rounds to nearest even.
__device__ __forceinline__ float dequant(float s, float z, uint32_t code) { return fmaf(s, float(code), z); }

// Code i (0..) of a little-endian packed word.
template <int BITS>
__device__ __forceinline__ uint32_t code_of(uint32_t w, int i) {
    return BITS == 8 ? ((w >> (8 * i)) & 0xffu) : ((w >> (4 * i)) & 0xfu);
}

// ---- staging registers: what one thread fetches for one key block ----------------
// K: thread (key = t / 8, piece = t % 8) takes 32 dims of one key.
// V: thread (dq = t % 64, kq = t / 64) takes 4 dims of 8 keys.
template <int BITS>
struct Stage {
    uint32_t k[BITS == 16 ? 16 : BITS];     // 32 dims: 64 B (f16), 32 B (8-bit), 16 B (4-bit)
    uint32_t v[8][BITS == 16 ? 2 : 1];      // per key 4 dims: 8 B (f16), 4 B (8-bit), 2 B (4-bit)
};

// Scales and biases of a block's 32 keys, staged in LDS by the first 128 threads (8 bytes each: the four f16
// of a key's groups) and read from there: per array [key][groups (0, 1) | groups (2, 3)] as pairs of f16.
struct BlockScales {
    uint32_t w[4][BK][2];  // [k scales | k biases | v scales | v biases]
    __device__ __forceinline__ float get(int arr, int key, int group) const {
        return (float)__builtin_bit_cast(_Float16, uint16_t(w[arr][key][group >> 1] >> (16 * (group & 1))));
    }
};

struct Rsrc {
    __amdgpu_buffer_rsrc_t k, v, ks, kz, vs, vz;
};

template <int BITS>
__device__ __forceinline__ void stage_load(Stage<BITS> &st, const Rsrc &r, uint32_t kvh, uint32_t key0, uint32_t kv,
                                           int tid) {
    constexpr int RB = row_bytes<BITS>();
    {
        const int key = tid >> 3, piece = tid & 7;
        const int row = int((key0 + key) * kvh + kv);
        const int off = row * RB + piece * (RB / 8);
        if constexpr (BITS == 8) {
            const u32x4 x = __builtin_amdgcn_raw_buffer_load_b128(r.k, off, 0, 0);
            const u32x4 y = __builtin_amdgcn_raw_buffer_load_b128(r.k, off + 16, 0, 0);
            st.k[0] = x.x, st.k[1] = x.y, st.k[2] = x.z, st.k[3] = x.w;
            st.k[4] = y.x, st.k[5] = y.y, st.k[6] = y.z, st.k[7] = y.w;
        } else if constexpr (BITS == 4) {
            const u32x4 x = __builtin_amdgcn_raw_buffer_load_b128(r.k, off, 0, 0);
            st.k[0] = x.x, st.k[1] = x.y, st.k[2] = x.z, st.k[3] = x.w;
        } else {
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const u32x4 x = __builtin_amdgcn_raw_buffer_load_b128(r.k, off + 16 * i, 0, 0);
                st.k[4 * i] = x.x, st.k[4 * i + 1] = x.y, st.k[4 * i + 2] = x.z, st.k[4 * i + 3] = x.w;
            }
        }
    }
    {
        const int dq = tid & 63, kq = tid >> 6;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int row = int((key0 + 8 * kq + i) * kvh + kv);
            const int off = row * RB + dq * (RB / 64);
            if constexpr (BITS == 8) {
                st.v[i][0] = __builtin_amdgcn_raw_buffer_load_b32(r.v, off, 0, 0);
            } else if constexpr (BITS == 4) {
                st.v[i][0] = uint16_t(__builtin_amdgcn_raw_buffer_load_b16(r.v, off, 0, 0));
            } else {
                const u32x2 x = __builtin_amdgcn_raw_buffer_load_b64(r.v, off, 0, 0);
                st.v[i][0] = x.x, st.v[i][1] = x.y;
            }
        }
    }
}

__device__ __forceinline__ float h2f(uint32_t bits16) {
    return (float)__builtin_bit_cast(_Float16, uint16_t(bits16));
}

// Where key `key` (0..31) of the block sits inside a V^T row: the order in which the
// S^T accumulator hands its keys to the P^T operand (see the kernel).
__device__ __forceinline__ constexpr int vt_pos(int key) {
    const int s = key >> 4, u = key & 15;
    return 16 * s + 8 * ((u & 7) >> 2) + 4 * (u >> 3) + (u & 3);
}

// Dequantizes the staged registers into the two parts of the block's image.  Keys at or past key_limit
// (the end of the chunk) are written as zeros: their probabilities are 0, and 0 * 0
// stays 0 whatever the cache rows hold.
template <int BITS>
__device__ __forceinline__ void stage_store(const Stage<BITS> &st, const BlockScales &sb, unsigned char *k_img, unsigned char *v_img,
                                            uint32_t key0, uint32_t key_limit, int tid) {
    {
        const int key = tid >> 3, piece = tid & 7;
        uint32_t o[16];
        if constexpr (BITS == 16) {
#pragma unroll
            for (int i = 0; i < 16; i++) o[i] = st.k[i];
        } else {
            const float s = sb.get(0, key, piece >> 1), z = sb.get(1, key, piece >> 1);
            constexpr int PER = 32 / BITS;
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const uint32_t w = st.k[(2 * i) / PER];
                o[i] = pack_half2(dequant(s, z, code_of<BITS>(w, (2 * i) % PER)),
                                  dequant(s, z, code_of<BITS>(w, (2 * i + 1) % PER)));
            }
        }
        if (key0 + key >= key_limit) {
#pragma unroll
            for (int i = 0; i < 16; i++) o[i] = 0;
        }
        // dims 32 piece + 8 j .. + 7 are the (hf = j % 2) half of fragment 2 piece + j / 2
#pragma unroll
        for (int j = 0; j < 4; j++) {
            *reinterpret_cast<u32x4 *>(k_img + (4 * piece + j) * 512 + key * 16) =
                u32x4{o[4 * j], o[4 * j + 1], o[4 * j + 2], o[4 * j + 3]};
        }
    }
    {
        const int dq = tid & 63, kq = tid >> 6;
        // keys 8kq..8kq+7: two runs of 4 neighbours in the row's key order
        const int p0 = vt_pos(8 * kq), p1 = vt_pos(8 * kq + 4);
        uint32_t w[4][4];  // [dim][pair of keys]
#pragma unroll
        for (int i = 0; i < 8; i += 2) {
            float x[2][4];
#pragma unroll
            for (int u = 0; u < 2; u++) {
                const bool live = key0 + 8 * kq + i + u < key_limit;
                if constexpr (BITS == 16) {
#pragma unroll
                    for (int d = 0; d < 4; d++) x[u][d] = live ? h2f(st.v[i + u][d >> 1] >> (16 * (d & 1))) : 0.0f;
                } else {
                    const float s = sb.get(2, 8 * kq + i + u, dq >> 4), z = sb.get(3, 8 * kq + i + u, dq >> 4);
#pragma unroll
                    for (int d = 0; d < 4; d++) x[u][d] = live ? dequant(s, z, code_of<BITS>(st.v[i + u][0], d)) : 0.0f;
                }
            }
#pragma unroll
            for (int d = 0; d < 4; d++) w[d][i / 2] = pack_half2(x[0][d], x[1][d]);
        }
#pragma unroll
        for (int d = 0; d < 4; d++) {
            const int dim = 4 * dq + d;
            unsigned char *frag = v_img + (dim >> 5) * 2048 + (dim & 31) * 16;  // position 0 of the dim
            *reinterpret_cast<u32x2 *>(frag + (p0 >> 3) * 512 + (p0 & 7) * 2) = u32x2{w[d][0], w[d][1]};
            *reinterpret_cast<u32x2 *>(frag + (p1 >> 3) * 512 + (p1 & 7) * 2) = u32x2{w[d][2], w[d][3]};
        }
    }
}

// One workgroup per (block of 32 keys, kv head).  The K tile goes out as it is made (a wave's store is eight runs
// of 128 bytes); the V^T tile is a transposition (a thread holds 4 dims of 8 keys, the image wants 8 keys of a dim
// side by side), so it is put together in LDS and copied out as whole lines.
template <int BITS>
__global__ __launch_bounds__(PREP_THREADS) void prefill_prepare_kernel(PrepareArgs a) {
    constexpr int RB = row_bytes<BITS>();
    __shared__ __attribute__((aligned(16))) unsigned char vt_lds[PART_BYTES];
    __shared__ BlockScales sb;
    const uint32_t block = blockIdx.x, kv = blockIdx.y, kvh = a.kv_heads;
    const int tid = threadIdx.x;
    if (a.tiles_taken && block == 0 && kv == 0 && tid == 0) *a.tiles_taken = 0;
    const uint32_t cap_rows = a.key_limit * kvh;
    Rsrc rs;
    rs.k = make_rsrc(a.kdata, cap_rows * RB);
    rs.v = make_rsrc(a.vdata, cap_rows * RB);
    rs.ks = make_rsrc(a.kscales, BITS == 16 ? 0 : cap_rows * 8);
    rs.kz = make_rsrc(a.kbiases, BITS == 16 ? 0 : cap_rows * 8);
    rs.vs = make_rsrc(a.vscales, BITS == 16 ? 0 : cap_rows * 8);
    rs.vz = make_rsrc(a.vbiases, BITS == 16 ? 0 : cap_rows * 8);
    if constexpr (BITS != 16) {
        if (tid < 4 * BK) {
            // (a key past the cache's end reads as zeros: its values are written as zeros whatever the scales are)
            const int arr = tid / BK, key = tid % BK;
            const int off = int((block * BK + key) * kvh + kv) * 8;
            const __amdgpu_buffer_rsrc_t r = arr == 0 ? rs.ks : arr == 1 ? rs.kz : arr == 2 ? rs.vs : rs.vz;
            const u32x2 x = __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0);
            sb.w[arr][key][0] = x.x, sb.w[arr][key][1] = x.y;
        }
    }
    Stage<BITS> st;
    stage_load<BITS>(st, rs, kvh, block * BK, kv, tid);
    __syncthreads();  // the scales are in LDS
    unsigned char *img = a.images + (size_t(kv) * a.nblocks + block) * IMG_BYTES;
    stage_store<BITS>(st, sb, img, vt_lds, block * BK, a.key_limit, tid);
    __syncthreads();  // the V^T tile is in LDS
#pragma unroll
    for (int i = 0; i < PART_BYTES / 16 / PREP_THREADS; i++) {
        const int at = (i * PREP_THREADS + tid) * 16;
        *reinterpret_cast<u32x4 *>(img + PART_BYTES + at) = *reinterpret_cast<const u32x4 *>(vt_lds + at);
    }
}

#include "prefill_stream.hpp"  // Copy, copy_plain, scores_block, stream_block, settle

// max over the two lanes l and l ^ 32, without a trip through LDS
__device__ __forceinline__ float max_across_halves(float x) {
    uint32_t u = __builtin_bit_cast(uint32_t, x), v = u;
    // Swaps the upper half of u with the lower half of v: u = (lo, lo), v = (hi, hi).  The
    // instruction may not read a register a vector instruction wrote in the two cycles before.
    asm volatile("s_nop 1\nv_permlane32_swap_b32 %0, %1\n" : "+v"(u), "+v"(v));
    return fmaxf(__builtin_bit_cast(float, u), __builtin_bit_cast(float, v));
}

// A workgroup barrier for data that went through LDS only: waits for this wave's LDS accesses, not for its
// loads and stores to memory (__syncthreads waits for those too: behind the gate loads of a tile's end, or
// the output stores, that is microseconds with nothing else to run).
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// LDS: four K slots, then four V^T slots; block b uses slot b % 4 of each.
constexpr int MERGE_WAVE_BYTES = (4 * 16 + 2) * 64 * 4;  // half of a wave's O, its m and l, on their way to its partner
constexpr int LDS_BYTES = 8 * MERGE_WAVE_BYTES > 8 * PART_BYTES ? 8 * MERGE_WAVE_BYTES : 8 * PART_BYTES;
__device__ __forceinline__ uint32_t k_slot(uint32_t b) { return (b & 3) * PART_BYTES; }
__device__ __forceinline__ uint32_t v_slot(uint32_t b) { return (4 + (b & 3)) * PART_BYTES; }

// Blocks of keys that tile `tile` of `tq` tokens sees.
__device__ __host__ __forceinline__ uint32_t tile_blocks(uint32_t pos, uint32_t tokens, uint32_t tile, uint32_t tq = TQ) {
    const uint32_t end = tile * tq + tq < tokens ? tile * tq + tq : tokens;
    return (pos + end + BK - 1) / BK;
}

// One tile of TQ tokens x 8 heads of kv head `kv` against the keys it sees, or (SPLIT) against part `part` of them.
// WIDE: of WIDE_TQ tokens.  A wave has a row group of its own and takes every block, a block a step, and what the workgroup
// copies for a step, 32 KB instead of 64, serves twice the rows.  The copies are what the clock pays for most after the products: the kernel's
// streams by themselves run at 1370 to 1384 TFLOP/s with half of them and at 1290 with all.  Where a wide tile is taken: tiles_plan.
// EXACT: in the first EXACT_BLOCKS blocks the reference maximum is the maximum itself, so that a row's largest probability
// there is 1, which f16 holds exactly; relative to a maximum up to 2^TAU below it is rounded like the others, which shows
// in rows of few keys.  For AttGemm, whose passes took every tile's probabilities relative to the tile's own maximum
// (largest error over the output's r.m.s., 1712 tokens at 37: passes 0.8e-2 to 1.3e-2, without EXACT 1.5e-2, with 0.6e-2; 1 us
// a tile).
template <bool SPLIT, bool EXACT, bool WIDE>
__device__ __forceinline__ void prefill_tile(const PrefillArgs &a, unsigned char *tiles, uint32_t tile, uint32_t kv, uint32_t part_index, bool ask, uint32_t *next_tile) {
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 31, hf = lane >> 5;
    static_assert(SPLIT || !WIDE, "wide tiles leave parts");
    constexpr uint32_t TILE = WIDE ? WIDE_TQ : TQ, STRIDE = WIDE ? 1 : 2;  // tokens; blocks from one of a wave's to its next
    const int group = WIDE ? wave : wave & 3, parity = wave >> 2;  // the wave's rows; which key blocks it takes (WIDE: all), and its order
    const uint32_t tok0 = tile * TILE + 4 * group;  // this wave's first token
    const float c = a.scale * 1.4426950408889634f;  // scores are kept in units of log2(e)

    // Row of this lane: token tok0 + col / 8, head col % 8.
    const uint32_t tok = tok0 + (col >> 3);

    // Keys this workgroup walks: up to what its last token sees; what this wave needs.  A part's keys count from its
    // first block on: key0 is that block's first key, and a row of the tile may see none of the part (the tile's tokens
    // cross a block's end where the last part begins).
    const uint32_t block0 = SPLIT ? part_index * a.part_blocks : 0, key_base = block0 * BK;
    const uint32_t all_blocks = tile_blocks(a.pos, a.tokens, tile, TILE) - block0;
    const uint32_t nblocks = SPLIT ? min(all_blocks, a.part_blocks) : all_blocks;
    auto from_base = [&](uint32_t keys) { return SPLIT ? (keys > key_base ? keys - key_base : 0) : keys; };
    const uint32_t wave_first_len = from_base(a.pos + tok0 + 1);            // keys the wave's first token sees
    const uint32_t wave_keys = from_base(a.pos + min(tok0 + 4, a.tokens));  // keys its last token sees
    const uint32_t wave_blocks = tok0 < a.tokens ? min((wave_keys + BK - 1) / BK, nblocks) : 0;
    const uint32_t full_blocks = min(wave_first_len / BK, wave_blocks);  // blocks that need no mask

    const uint32_t lds0 = uint32_t(reinterpret_cast<uintptr_t>(tiles));
    const uint32_t lane16 = lane * 16;
    const unsigned char *images = a.images + (size_t(kv) * a.nblocks + block0) * IMG_BYTES;
    // Half `half` (8 KB) of part `v` (0 = K, 1 = V^T) of block b.  Blocks past the cache's end
    // are read from the last image instead; nobody looks at their slots.
    auto piece = [&](uint32_t b, int v, int half) {
        const uint32_t bb = min(b, a.nblocks - block0 - 1);
        Copy cp;
        cp.src = reinterpret_cast<uint64_t>(images) + uint64_t(bb) * IMG_BYTES + v * PART_BYTES + half * 8192;
        cp.dst = lds0 + (v ? v_slot(b) : k_slot(b)) + half * 8192;
        return cp;
    };

    // Step s works on blocks 2s (waves 0..3: parity 0) and 2s + 1 (waves 4..7: parity 1).  A
    // wave's step is a softmax (vector ALU) and an MFMA stream that adds the block to O and
    // computes the scores of the wave's next block; the two waves of a SIMD run them in opposite
    // order, so that one's softmax runs under the other's MFMAs:
    //   parity 0:  softmax(2s)               | O(2s) + S(2s+2)
    //   parity 1:  O(2s+1) + S(2s+3)         | softmax(2s+3)
    // During step s the workgroup copies what step s + 1 reads: K(2s+4), K(2s+5), V(2s+2),
    // V(2s+3); wave w takes half (w % 2) of part w / 2 of that list.  Before the loop: K(0..3),
    // V(0), V(1), in front of them the queries.  K(2s+4) and K(2s+5) land on K(2s) and K(2s+1), which step s - 1 read, V(2s+2) and
    // V(2s+3) on V(2s-2) and V(2s-1), the same: the barrier between the steps is all they wait for.
    // WIDE: step s works on block s, in all eight waves:
    //   parity 0:  softmax(s)                | O(s) + S(s+1)
    //   parity 1:  O(s) + S(s+1)             | softmax(s+1)
    // During step s, which reads V(s) and K(s+1), the workgroup copies V(s+1) and K(s+2), a quarter a wave, parity 0 the keys.  They
    // land on V(s-3) and K(s-2), last read in step s - 3.  Before the loop: K(0), K(1) and V(0), behind the queries, which
    // had all of the places.
    auto copy2k = [&](uint64_t src, uint32_t dst) {
        asm volatile(
            "s_mov_b32 m0, %[dst]\n"
            "s_nop 0\n"
            "global_load_lds_dwordx4 %[off], %[src]\n"
            "global_load_lds_dwordx4 %[off], %[src] offset:1024\n"
            :
            : [off] "v"(lane16), [src] "s"(src), [dst] "s"(dst)
            : "memory", "m0");
    };
    // Q^T operands: lane (col, hf), k-step st: dims 16 st + 8 hf .. + 7 of its row.  They come through LDS, in the places of
    // V(0..3): a load of 16 bytes of each of 32 rows is taken a row a cycle, and 16 of them in eight waves were 4 us in front of a
    // tile (1470 tokens from 0: first keys and queries there after 5.2 us, now 2.7).  A row group's 16 KB as they lie in memory, half
    // by each of its two waves; place p of row r holds the row's 16-byte piece (p - 4 (r / 4) mod 32) ^ (r % 4), which puts what
    // 16 lanes read on different banks and keeps every 64 bytes of memory together.
    uint32_t at = lane;  // (what depends on the lane is made where it is used, not kept in registers from tile to tile)
    asm volatile("" : "+v"(at));
    // (WIDE: eight row groups fill all places, the keys' too, and come before them)
    const uint32_t q_at = (WIDE ? 0 : v_slot(0)) + group * (32 * DIM * 2), q_place = lds0 + q_at;
#pragma unroll
    for (int i = 0; i < (WIDE ? 16 : 8); i++) {
        const uint32_t k = WIDE ? i : 8 * parity + i;  // rows 2k and 2k + 1
        const uint32_t tk = min(tok0 + k / 4, a.tokens - 1);
        const uint64_t src = reinterpret_cast<uint64_t>(a.q) + ((size_t(tk) * a.heads + kv * SAETTA_GQA_GROUP + 2 * k % 8) * DIM) * 2;
        const uint32_t off = (at >> 5) * 512 + (((at - 4 * (i >> 1 & 3)) & 31) ^ (2 * (i & 1) + (at >> 5))) * 16;
        asm volatile(
            "s_mov_b32 m0, %[dst]\n"
            "s_nop 0\n"
            "global_load_lds_dwordx4 %[off], %[src]\n"
            :
            : [off] "v"(off), [src] "s"(src), [dst] "s"(q_place + k * 1024)
            : "memory", "m0");
    }
    if constexpr (!WIDE) {
#pragma unroll
        for (int i = 0; i < 4; i++) {  // K(0..3): wave w takes 2 KB of each
            const Copy cp = piece(i, 0, 0);
            copy2k(cp.src + wave * 2048, cp.dst + wave * 2048);
        }
        asm volatile("s_waitcnt vmcnt(8)\n\ts_barrier" ::: "memory");  // (the keys stay on their way)
    } else {
        asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
    }
    half8 qb[16];
#pragma unroll
    for (int st = 0; st < 16; st++) {
        const uint32_t place = 4 * (((st >> 1) + (at >> 2 & 3)) & 7) + ((2 * (st & 1) + (at >> 5)) ^ (at & 3));
        qb[st] = *reinterpret_cast<const half8 *>(tiles + q_at + (at & 31) * (DIM * 2) + place * 16);
    }
    lds_barrier();  // the queries have been read: the values may land there
    if constexpr (WIDE) {
#pragma unroll
        for (int i = 0; i < 2; i++) {  // K(0), K(1)
            const Copy cp = piece(i, 0, 0);
            copy2k(cp.src + wave * 2048, cp.dst + wave * 2048);
        }
    }
#pragma unroll
    for (int i = 0; i < (WIDE ? 1 : 2); i++) {
        const Copy cp = piece(i, 1, 0);
        copy2k(cp.src + wave * 2048, cp.dst + wave * 2048);
    }

    floatx16 acc[8];
#pragma unroll
    for (int mt = 0; mt < 8; mt++) {
#pragma unroll
        for (int r = 0; r < 16; r++) acc[mt][r] = 0.0f;
    }
    // The reference maximum starts above what a block of masked scores gives (NO_SCORE * c), so that a row that sees
    // none of a wave's first block never takes that for its maximum: with m_ref equal to the rounded NO_SCORE * c the
    // exponent s * c - m_ref of a masked score is the product's rounding error, 1e21 either way, not minus infinity.
    // (The second wave of a row group starts at block 1: rows that end inside block 0 have nothing in it.)
    float m_ref = 0.25f * NO_SCORE * c, l_sum = 0.0f;

    // Row maximum of a block's scaled scores (first half of the softmax).  Register r of the
    // accumulator is key 4 hf + r % 4 + 8 (r / 4) of the block; masked scores become NO_SCORE (NO_SCORE * c in the units of the maximum).
    auto mask_max = [&](floatx16 &s, uint32_t key0, bool masked) {
        float bm = NO_SCORE;
        if (masked) {
            const uint32_t len = from_base(a.pos + tok + 1);   // keys this row sees
            const uint32_t vis = len > key0 ? len - key0 : 0;  // of which in this block
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const uint32_t key = 4 * hf + (r & 3) + 8 * (r >> 2);
                s[r] = key < vis ? s[r] : NO_SCORE;
            }
        }
#pragma unroll
        for (int r = 0; r < 16; r++) bm = fmaxf(bm, s[r]);
        bm = max_across_halves(bm);
        return fmaxf(bm * c, NO_SCORE);
    };
    // Raises the reference maximum when a block tops it by more than 2^TAU, rescaling O and l.
    auto raise_max = [&](float bm, uint32_t kb) {
        const float slack = EXACT && block0 + kb < EXACT_BLOCKS ? 0.0f : TAU;
        if (__any(bm > m_ref + slack)) {
            const float m_new = bm > m_ref + slack ? bm : m_ref;
            const float alpha = __builtin_amdgcn_exp2f(m_ref - m_new);
            m_ref = m_new;
            l_sum *= alpha;
#pragma unroll
            for (int mt = 0; mt < 8; mt++) {
#pragma unroll
                for (int r = 0; r < 16; r++) acc[mt][r] *= alpha;
            }
        }
    };
    // Second half of the softmax: probabilities 2^(s c - m), their sum, and the P^T operands
    // (k-step sp takes registers 8 sp .. 8 sp + 7, the order vt_pos mirrors).
    auto exp_pack = [&](const floatx16 &s, half8 (&pb)[2]) {
        float p[16];
        float sum = 0.0f;
#pragma unroll
        for (int r = 0; r < 16; r++) {
            p[r] = __builtin_amdgcn_exp2f(fmaf(s[r], c, -m_ref));
            sum += p[r];
        }
        l_sum += sum;
#pragma unroll
        for (int sp = 0; sp < 2; sp++) {
            u32x4 w = {pack_half2(p[8 * sp], p[8 * sp + 1]), pack_half2(p[8 * sp + 2], p[8 * sp + 3]),
                       pack_half2(p[8 * sp + 4], p[8 * sp + 5]), pack_half2(p[8 * sp + 6], p[8 * sp + 7])};
            pb[sp] = __builtin_bit_cast(half8, w);
        }
    };

    // K(0..3) are in LDS, V(0) and V(1) on their way (WIDE: K(0) and K(1), V(0))
    if constexpr (WIDE) asm volatile("s_waitcnt vmcnt(2)\n\ts_barrier" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(4)\n\ts_barrier" ::: "memory");

    const uint32_t nsteps = WIDE ? nblocks : (nblocks + 1) / 2;
    const int part = wave >> 1, half = wave & 1;  // what the wave copies in every step
    auto copy_of = [&](uint32_t step) {
        if constexpr (WIDE) {  // a quarter of K(s + 2) or of V(s + 1)
            Copy cp = piece(step + 2 - parity, parity, 0);
            cp.src += (wave & 3) * 4096, cp.dst += (wave & 3) * 4096;
            return cp;
        }
        const uint32_t cb = part == 0 ? 2 * step + 4 : part == 1 ? 2 * step + 5 : part == 2 ? 2 * step + 2 : 2 * step + 3;
        return piece(cb, part >= 2, half);
    };
    if (parity == 0) {
        floatx16 s;
#pragma unroll
        for (int r = 0; r < 16; r++) s[r] = 0.0f;
        if (0 < wave_blocks) scores_block(s, qb, lds0 + k_slot(0) + lane16);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();  // V(0) and V(1) are there; the first step's copies overwrite K(0) and K(1) (WIDE: V(0); nothing)
        for (uint32_t step = 0; step < nsteps; step++) {
            const Copy cp = copy_of(step);
            const uint32_t kb = STRIDE * step;
            if (kb < wave_blocks) {
                raise_max(mask_max(s, kb * BK, kb >= full_blocks), kb);
                half8 pb[2];
                exp_pack(s, pb);
                // (past the wave's last block the scores are of stale keys and never looked at)
                stream_block<WIDE>(s, acc, qb, pb, lds0 + k_slot(kb + STRIDE) + lane16, lds0 + v_slot(kb) + lane16, cp, lane16);
            } else {
                copy_plain<WIDE>(cp, lane16);
            }
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
        }
    } else {
        constexpr uint32_t FIRST = WIDE ? 0 : 1;
        half8 pb[2] = {};
        if (FIRST < wave_blocks) {
            floatx16 s;
            scores_block(s, qb, lds0 + k_slot(FIRST) + lane16);
            raise_max(mask_max(s, FIRST * BK, FIRST >= full_blocks), FIRST);
            exp_pack(s, pb);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        for (uint32_t step = 0; step < nsteps; step++) {
            const Copy cp = copy_of(step);
            const uint32_t kb = STRIDE * step + FIRST;
            if (kb < wave_blocks) {
                // This wave's stream comes before its softmax, the other wave's of the SIMD after: let
                // this one's MFMAs go first, so that its softmax still finds the other's to run under.
                floatx16 s;
                __builtin_amdgcn_s_setprio(2);
                stream_block<WIDE>(s, acc, qb, pb, lds0 + k_slot(kb + STRIDE) + lane16, lds0 + v_slot(kb) + lane16, cp, lane16);
                __builtin_amdgcn_s_setprio(0);
                if (kb + STRIDE < wave_blocks) {
                    raise_max(mask_max(s, (kb + STRIDE) * BK, kb + STRIDE >= full_blocks), kb + STRIDE);
                    exp_pack(s, pb);
                }
            } else {
                copy_plain<WIDE>(cp, lane16);
            }
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
        }
    }

    settle(acc);
    // Which tile this workgroup takes next: asked for here, where the workgroups are apart in time (their tiles differ in
    // length; at the kernel's start every one of them would ask at once, and the adds on one word come one after the
    // other), and looked at when the tile has ended.  (Before the gate loads: behind them the one more register that is
    // live with them costs 150 bytes of spills.)
    uint32_t got = ask ? 0u : 0xffffffffu;
    if (ask && tid == 0) got = gridDim.x + atomicAdd(a.tiles_taken, 1u);
    if constexpr (WIDE) {
        // Nothing to join: the part's O, m and l leave as two tiles of TQ tokens would leave them (a second one past the chunk's end
        // has no place).
        const float l = l_sum + __shfl_xor(l_sum, 32);
        const uint32_t ntiles = (a.tokens + TQ - 1) / TQ, narrow = 2 * tile + (group >> 2);
        if (narrow < ntiles) {
            const size_t item = (size_t(part_index) * ntiles + narrow) * a.kv_heads + kv;
#pragma unroll
            for (int i = 0; i < 32; i++) {
                float *po = a.part_o + ((item * WAVES + (group & 3) * 2 + (i >> 4)) * 16 * 64 + lane) * 4;
                const int mt = i >> 2, q4 = i & 3;
                *reinterpret_cast<float4 *>(po + (i & 15) * 64 * 4) = float4{acc[mt][4 * q4], acc[mt][4 * q4 + 1], acc[mt][4 * q4 + 2], acc[mt][4 * q4 + 3]};
            }
            if (hf == 0) *reinterpret_cast<float2 *>(a.part_ml + ((item * 4 + (group & 3)) * 32 + col) * 2) = float2{m_ref, l};
        }
        if (tid == 0) *next_tile = got;
        return;
    }

    // The gate values of this wave's half of the dims, asked for before the merge below so that they travel while
    // it runs: two rows of 512 bytes a load, as the outputs are stored (a token past the end: the last token's, unused).
    asm volatile("" : "+v"(at));
    float4 g[16];
    const uint32_t half_row = at >> 5, in_row = 4 * (at & 31);  // a lane's row of two; its dims of the half
    auto first_row = [&](int i) { return size_t(min(tok0 + i / 4, a.tokens - 1)) * a.heads + kv * SAETTA_GQA_GROUP + 2 * i % 8; };
    if constexpr (!SPLIT) {
#pragma unroll
        for (int i = 0; i < 16; i++) g[i] = *reinterpret_cast<const float4 *>(a.q_and_gate + first_row(i) * 2 * DIM + DIM + 128 * parity + (half_row * 2 * DIM + in_row));
    }
    // ---- the two waves of a row group merge their halves of the keys ----------------------
    // Each wave finishes half of the dims: parity 0 the accumulators 0..3 (dims 0..127), parity 1
    // the rest.  It hands the other half, m and l to its partner through LDS (the tiles are done
    // with: the loop ended on a barrier), four accumulator registers of a lane side by side.
    float4 *mine_out = reinterpret_cast<float4 *>(tiles + wave * MERGE_WAVE_BYTES) + at;
    unsigned char *theirs_base = tiles + (wave ^ 4) * MERGE_WAVE_BYTES;
    const float4 *theirs_in = reinterpret_cast<const float4 *>(theirs_base) + at;
    floatx16 fin[4];
    auto hand_over = [&](const floatx16 &x, int i) {
#pragma unroll
        for (int q4 = 0; q4 < 4; q4++) mine_out[(4 * i + q4) * 64] = float4{x[4 * q4], x[4 * q4 + 1], x[4 * q4 + 2], x[4 * q4 + 3]};
    };
    if (parity == 0) {
#pragma unroll
        for (int i = 0; i < 4; i++) fin[i] = acc[i], hand_over(acc[4 + i], i);
    } else {
#pragma unroll
        for (int i = 0; i < 4; i++) fin[i] = acc[4 + i], hand_over(acc[i], i);
    }
    float2 *ml_out = reinterpret_cast<float2 *>(tiles + wave * MERGE_WAVE_BYTES + 16 * 1024) + at;
    *ml_out = float2{m_ref, l_sum};
    lds_barrier();  // (the gate values stay on their way)
    const float2 ml_other = *(reinterpret_cast<const float2 *>(theirs_base + 16 * 1024) + at);
    const float m_other = ml_other.x, l_other = ml_other.y;
    const float m_new = fmaxf(m_ref, m_other);
    const float mine = __builtin_amdgcn_exp2f(m_ref - m_new), theirs = __builtin_amdgcn_exp2f(m_other - m_new);
    l_sum = l_sum * mine + l_other * theirs;
    auto joined = [&](int i) {
        const int mt = i >> 2, q4 = i & 3;
        const float4 x = theirs_in[i * 64];
        return float4{fin[mt][4 * q4] * mine + x.x * theirs, fin[mt][4 * q4 + 1] * mine + x.y * theirs,
                      fin[mt][4 * q4 + 2] * mine + x.z * theirs, fin[mt][4 * q4 + 3] * mine + x.w * theirs};
    };

    if constexpr (SPLIT) {
        // The part's O, m and l as they are, a contiguous kilobyte per store of a wave.  (Rows past the chunk's end leave
        // what their masked lanes hold; nothing reads it.)
        const float l = l_sum + __shfl_xor(l_sum, 32);
        const uint32_t ntiles = (a.tokens + TQ - 1) / TQ;
        const size_t item = (size_t(part_index) * ntiles + tile) * a.kv_heads + kv;
        float *po = a.part_o + ((item * WAVES + group * 2 + parity) * 16 * 64 + lane) * 4;
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const float4 w = joined(i);
            *reinterpret_cast<float4 *>(po + i * 64 * 4) = w;
        }
        if (parity == 0 && hf == 0) {
            float2 ml = {m_new, l};
            *reinterpret_cast<float2 *>(a.part_ml + ((item * 4 + group) * 32 + col) * 2) = ml;
        }
        if (tid == 0) *next_tile = got;
        return;
    }

    // ---- out = O / l * sigmoid(gate) ---------------------------------------------------
    // The lane's row sum is split over the two lane halves (each saw half the keys).
    const float l = l_sum + __shfl_xor(l_sum, 32);
    // Through LDS once more, so that a wave stores whole lines: 16 bytes of each of 32 rows are taken a row a cycle, gates
    // and outputs both (8 us of a tile's end, 1470 tokens from 0; now 4.2).  A lane's four dims of its row are a piece; the
    // pieces of the same dims lie side by side, 528 bytes from the next dims', in the place of what the partner handed over,
    // which nobody else reads (a wave's LDS accesses run in order).
    const float inv = 1.0f / l;
    float4 o[16];
#pragma unroll
    for (int i = 0; i < 16; i++) {
        o[i] = joined(i);
        o[i].x *= inv, o[i].y *= inv, o[i].z *= inv, o[i].w *= inv;
    }
    constexpr int PIECE = 32 * 16 + 16;
    static_assert(32 * PIECE <= MERGE_WAVE_BYTES, "the pieces of 32 rows");
    wave_sync();  // every lane has taken what the partner handed over
#pragma unroll
    for (int i = 0; i < 16; i++) *reinterpret_cast<float4 *>(theirs_base + (2 * i + (at >> 5)) * PIECE + (at & 31) * 16) = o[i];
    wave_sync();
#pragma unroll
    for (int i = 0; i < 16; i++) {
        const float4 x = *reinterpret_cast<const float4 *>(theirs_base + in_row / 4 * PIECE + (2 * i + half_row) * 16);
        float4 w;
        w.x = x.x * __builtin_amdgcn_rcpf(1.0f + __expf(-g[i].x));
        w.y = x.y * __builtin_amdgcn_rcpf(1.0f + __expf(-g[i].y));
        w.z = x.z * __builtin_amdgcn_rcpf(1.0f + __expf(-g[i].z));
        w.w = x.w * __builtin_amdgcn_rcpf(1.0f + __expf(-g[i].w));
        if (tok0 + i / 4 < a.tokens) *reinterpret_cast<float4 *>(a.out + first_row(i) * DIM + 128 * parity + (half_row * DIM + in_row)) = w;
    }
    if (tid == 0) *next_tile = got;
}

// The first tile that has a part `part` of part_blocks blocks (tiles see more keys the later they are), and how many
// (tile, part) pairs there are.
__device__ __host__ __forceinline__ uint32_t prefill_first_tile(uint32_t pos, uint32_t tokens, uint32_t part_blocks, uint32_t part, uint32_t tq = TQ) {
    const uint32_t ntiles = (tokens + tq - 1) / tq;
    const uint32_t keys = part * part_blocks * BK;  // a tile has the part if it sees more keys than these
    if (pos + tokens <= keys) return ntiles;
    if (pos + tq > keys) return 0;
    const uint32_t t = (keys - pos) / tq;  // tokens up to keys - pos see no key of it
    return t < ntiles ? t : ntiles - 1;
}
__device__ __host__ __forceinline__ uint32_t prefill_items(uint32_t pos, uint32_t tokens, uint32_t part_blocks, uint32_t tq = TQ) {
    const uint32_t ntiles = (tokens + tq - 1) / tq;
    // the parts that begin at a key the first tile sees are every tile's
    const uint32_t whole = (pos + (tokens < tq ? tokens : tq) - 1) / (part_blocks * BK) + 1;
    uint32_t n = whole * ntiles;
    for (uint32_t p = whole, first; (first = prefill_first_tile(pos, tokens, part_blocks, p, tq)) < ntiles; p++) n += ntiles - first;
    return n;
}

// A workgroup takes tiles until there are none left: with more tiles than workgroups (one per CU: the LDS ring
// fills a CU), the next tile starts without a new workgroup having to be dispatched.  Tiles are numbered from the
// one with the most keys down, the kv heads side by side.  Workgroup w starts with tile w; the others are handed
// out in that order to whoever asks next (one atomic add per tile on a counter behind the images, asked for
// before the tile's epilogue so that the answer is there when it ends): a workgroup that took a long tile, or runs
// on a slower CU, asks later and gets a shorter one, so that all of them end together (tiles dealt beforehand, the
// longest with the shortest, ended 40 us apart: the workgroups' rates differ by a tenth).
// SPLIT: an item is a part of a tile's keys, parts side by side in tiles and kv heads (workgroups that run together walk
// the same keys); the tiles that have a part p are the ones from prefill_first_tile(p) on.
template <bool SPLIT, bool EXACT, bool WIDE>
__global__ __launch_bounds__(THREADS, 2) void attention_prefill_kernel(PrefillArgs a) {
    constexpr uint32_t TILE = WIDE ? WIDE_TQ : TQ;
    extern __shared__ __attribute__((aligned(1024))) unsigned char tiles[];
    __shared__ uint32_t next_tile;
    const uint32_t ntiles = (a.tokens + TILE - 1) / TILE, G = gridDim.x;
    uint32_t total = ntiles * a.kv_heads;
    if constexpr (SPLIT) total = prefill_items(a.pos, a.tokens, a.part_blocks, TILE) * a.kv_heads;
    for (uint32_t idx = blockIdx.x; idx < total;) {
        // (the tiles from G on are handed out by one question each: the tiles before the last G ask one, when they end,
        // and the last G none: nothing is left by then, and the kernel's last epilogues do not wait for an answer)
        uint32_t at = idx / a.kv_heads, part = 0;
        if constexpr (SPLIT) {
            for (uint32_t n; at >= (n = ntiles - prefill_first_tile(a.pos, a.tokens, a.part_blocks, part, TILE)); part++) at -= n;
        }
        prefill_tile<SPLIT, EXACT, WIDE>(a, tiles, ntiles - 1 - at, idx % a.kv_heads, part, idx + G < total, &next_tile);
        lds_barrier();  // the next tile is known; this tile's merge has been read: the next tile's keys may land on it (its stores go on meanwhile)
        idx = next_tile;
    }
}

// Registers x[0..3] of four lanes, lane t holding piece t of row j in x[j]: then lane t holds piece j of its row t.
__device__ __forceinline__ void turn(u32x4 *x, int lane) {
    const bool odd = lane & 1, high = lane & 2;
#pragma unroll
    for (int j = 0; j < 4; j += 2)
#pragma unroll
        for (int w = 0; w < 4; w++) {
            const uint32_t u = x[j][w], v = x[j + 1][w];
            const uint32_t un = __builtin_amdgcn_mov_dpp(int(u), 0xb1, 0xf, 0xf, true), vn = __builtin_amdgcn_mov_dpp(int(v), 0xb1, 0xf, 0xf, true);
            x[j][w] = odd ? vn : u, x[j + 1][w] = odd ? v : un;
        }
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
        for (int w = 0; w < 4; w++) {
            const uint32_t u = x[j][w], v = x[j + 2][w];
            const uint32_t un = __builtin_amdgcn_mov_dpp(int(u), 0x4e, 0xf, 0xf, true), vn = __builtin_amdgcn_mov_dpp(int(v), 0x4e, 0xf, 0xf, true);
            x[j][w] = high ? vn : u, x[j + 2][w] = high ? v : un;
        }
}

// Joins the parts of every tile: out = sum_p 2^(m_p - m) O_p / sum_p 2^(m_p - m) l_p * sigmoid(gate).  A workgroup takes
// one token of one kv head: 8 rows x 256 dims, four float4 per thread.  The parts lie in accumulator order, where the 8
// rows' pieces of four dims are one line of 128 bytes: 8 neighbouring lanes take a line of a part (a lane per piece of ONE
// row made every lane of a load its own line: 22 us for 50 MB of parts).  Then four lanes turn their four pieces of four rows
// round, so that gates and outputs move 512 bytes of a row at a time and not 16 of each of eight, which are taken a row a
// cycle (the whole call: 1032 tokens at 38 41.1 -> 40.3 us, 150 at 9000 50.2 -> 49.0, 7 at 3000 19.0 -> 18.2).
// TEAMS: more than eight parts are dealt to four teams of 128 threads, joined through LDS: one team's batches come one after
// another, a trip through memory each (the whole call: 7 tokens at 3000 18.2 -> 17.4 us, 10 at 103706 63.5 -> 61.3; from 9 parts on
// four teams are ahead or even: 55 tokens at 17388 47.0 both).
constexpr int MERGE_THREADS = 128, MERGE_TEAMS = 4;
template <int TEAMS>
__global__ __launch_bounds__(MERGE_THREADS * TEAMS, 4) void prefill_merge_kernel(PrefillArgs a) {
    __shared__ floatx4 team_o[TEAMS > 1 ? TEAMS - 1 : 1][4][MERGE_THREADS];
    __shared__ float2 team_ml[TEAMS > 1 ? TEAMS - 1 : 1][8];
    const uint32_t tid = TEAMS > 1 ? threadIdx.x % MERGE_THREADS : threadIdx.x, team = TEAMS > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x / MERGE_THREADS) : 0;
    const uint32_t tok = blockIdx.x, kv = blockIdx.y, tile = tok / TQ, group = (tok % TQ) / 4;
    const uint32_t ntiles = (a.tokens + TQ - 1) / TQ;
    const uint32_t parts = (tile_blocks(a.pos, a.tokens, tile) + a.part_blocks - 1) / a.part_blocks;
    const size_t item_stride = size_t(ntiles) * a.kv_heads, item0 = size_t(tile) * a.kv_heads + kv;
    const uint32_t h = tid & 7, four = tid >> 3, col = (tok % 4) * 8 + h;  // pieces 4 four .. + 3 of row h
    // gates and outputs: piece 4 four + h % 4 of rows h / 4 * 4 .. + 3
    const size_t row = size_t(tok) * a.heads + kv * SAETTA_GQA_GROUP + (h & 4);
    const uint32_t dim = 16 * four + 4 * (h & 3);
    float4 g[4];
    if (team == 0) {
#pragma unroll
        for (int j = 0; j < 4; j++) g[j] = *reinterpret_cast<const float4 *>(a.q_and_gate + (row + j) * 2 * DIM + DIM + dim);
    }
    const float *ml = a.part_ml + ((item0 * 4 + group) * 32 + col) * 2;
    // (pieces 2i and 2i + 1 are accumulator registers 4i .. 4i + 3 of the lanes col and col + 32)
    const float *po = a.part_o + (((item0 * WAVES + group * 2 + (four >> 3)) * 16 + 2 * (four & 7)) * 64 + col) * 4;
    float m = 4.0f * NO_SCORE, l = 0.0f;
    floatx4 o[4] = {};
    // BATCH parts at a time, all of their loads requested before the first is used (past the last part: the last part
    // again, with no weight: in batches of 8 whatever the number, a tile of two parts asked for each of them four times;
    // 777 tokens from 0 12.1 -> 8.9 us, 2300 at 10000 36.4 -> 31.0, which is 4.8 TB/s of parts, gates and outputs)
    auto join = [&](auto batch) {
        constexpr int BATCH = decltype(batch)::value;
        for (uint32_t p0 = team * BATCH; p0 < parts; p0 += TEAMS * BATCH) {
            float2 x[BATCH];
            floatx4 y[BATCH][4];
#pragma unroll
            for (int j = 0; j < BATCH; j++) {
                const uint32_t p = min(p0 + j, parts - 1);
                x[j] = *reinterpret_cast<const float2 *>(ml + p * item_stride * (4 * 32 * 2));
#pragma unroll
                for (int k = 0; k < 4; k++) y[j][k] = *reinterpret_cast<const floatx4 *>(po + p * item_stride * (WAVES * 16 * 64 * 4) + ((k >> 1) * 64 + (k & 1) * 32) * 4);
            }
            float m_new = m;
#pragma unroll
            for (int j = 0; j < BATCH; j++) m_new = fmaxf(m_new, x[j].x);
            const float old = __builtin_amdgcn_exp2f(m - m_new);
            m = m_new;
            l *= old;
#pragma unroll
            for (int k = 0; k < 4; k++) o[k] *= old;
#pragma unroll
            for (int j = 0; j < BATCH; j++) {
                const float now = p0 + j < parts ? __builtin_amdgcn_exp2f(x[j].x - m_new) : 0.0f;
                l += x[j].y * now;
#pragma unroll
                for (int k = 0; k < 4; k++) o[k] += y[j][k] * now;
            }
        }
    };
    if constexpr (TEAMS > 1) {
        if (parts <= 4 * TEAMS) join(std::integral_constant<int, 4>{});
        else join(std::integral_constant<int, 8>{});
        if (team > 0) {
#pragma unroll
            for (int k = 0; k < 4; k++) team_o[team - 1][k][tid] = o[k];
            if (four == 0) team_ml[team - 1][h] = float2{m, l};
        }
        __syncthreads();
        if (team > 0) return;
        float top = m;
#pragma unroll
        for (int t = 0; t < TEAMS - 1; t++) top = fmaxf(top, team_ml[t][h].x);
        const float own = __builtin_amdgcn_exp2f(m - top);
        l *= own;
#pragma unroll
        for (int k = 0; k < 4; k++) o[k] *= own;
#pragma unroll
        for (int t = 0; t < TEAMS - 1; t++) {  // (a team without a part: l = 0, o = 0)
            const float now = __builtin_amdgcn_exp2f(team_ml[t][h].x - top);
            l += team_ml[t][h].y * now;
#pragma unroll
            for (int k = 0; k < 4; k++) o[k] += team_o[t][k][tid] * now;
        }
    } else if (parts <= 2) {
        join(std::integral_constant<int, 2>{});
    } else if (parts <= 4) {
        join(std::integral_constant<int, 4>{});
    } else {
        join(std::integral_constant<int, 8>{});
    }
    const float inv = 1.0f / l;
    u32x4 w[4];
#pragma unroll
    for (int k = 0; k < 4; k++) w[k] = __builtin_bit_cast(u32x4, o[k] * inv);
    turn(w, tid);
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const floatx4 x = __builtin_bit_cast(floatx4, w[j]);
        float4 r;
        r.x = x[0] * __builtin_amdgcn_rcpf(1.0f + __expf(-g[j].x));
        r.y = x[1] * __builtin_amdgcn_rcpf(1.0f + __expf(-g[j].y));
        r.z = x[2] * __builtin_amdgcn_rcpf(1.0f + __expf(-g[j].z));
        r.w = x[3] * __builtin_amdgcn_rcpf(1.0f + __expf(-g[j].w));
        *reinterpret_cast<float4 *>(a.out + (row + j) * DIM + dim) = r;
    }
}

// ---- short chunks over short contexts: one launch ------------------------------------------------
//
// A chunk of 166 tokens is 22 workgroups of the kernel above, which then walk their 166 keys in three steps behind a
// prologue and an epilogue of 7 us, and the prepare kernel is 3.8 us more before them: 22 us in all for 2 us of work.
// Here a workgroup takes ONE row group (4 tokens x 8 heads = 32 rows) of a kv head, eight times as many workgroups, and
// its 8 waves take alternate blocks of 32 keys, so that 256 keys are one round; each wave finishes 32 of the 256 dims.  The
// cache is read where it lies, once per row group: the keys go from memory to MFMA operands in registers, the values to a
// tile of the wave's own in LDS, row by row as in memory, and come back transposed (ds_read_b64_tr_b16).  Codes are
// dequantized on the way, with the arithmetic of the prepare kernel.
// The price is that every row group pulls (and dequantizes) the keys for itself: with many tokens the tiles of 16 and their
// images win, and with few over a long context a row group's keys go to several workgroups (SPLIT), whose parts the
// tiles' merge joins; the lines are in choose_small.
// What bounds a block of halves per wave, each with all dims of its own blocks (4 us for the eight of them): 256 KB through the CU's 64 bytes a cycle are 1.8 of
// them, the values' way through LDS and the query operands 1.4.  A key's operands straight from its row, 16 bytes a lane,
// took 5.3 us: such a load is taken a row a cycle, and so four lanes fetch 64 bytes of a row together and turn four rows
// round in registers.  Codes (4 us, once for every row group): vector instructions, of which a pair of codes is
// three (8-bit) or four, in packed halves; as f32, seven of them, the eight blocks took 5 us.  The values' reads are left to
// the compiler's counting: a wait for each four of them took 0.3 us of halves' four rounds.
// Measured, the whole call, tiles -> this: halves, 16 tokens at 16 18.3 -> 7.5 us, 166 from 0 21.7 -> 10.8; fetched row by
// row -> in turns: 16 at 500 20.5 -> 18.6, 300 from 0 19.1 -> 17.4, 500 from 0 23.1 -> 20.5, 500 at 500 32.2 -> 26.5; codes as f32 -> as halves: 8-bit
// 23.8 -> 20.2, 24.9 -> 21.8, 34.4 -> 28.8, 4-bit 23.3 -> 20.2, 23.4 -> 21.4, 33.3 -> 29.4, and no further from 64 bits.
// Halves fill the registers there: what depends on the lane alone is made anew where it is used (`at`), so that nothing spills; three
// spilled registers cost a launch 1 us (300 from 0 18.3), the instructions 0.1 to 0.5 (16 at 500 18.1).
// One maximum for the eight blocks of a round was faster with codes, but not with this precision: of each block the largest probability
// is now 1, without a rounding, and with the largest of eight blocks alone an output was up to 1.2 times as far from 64 bits.
constexpr int SMALL_WAVES = 8, SMALL_THREADS = 64 * SMALL_WAVES;
// How the waves divide the work on O.  OWN_BLOCKS: each all dims of its own blocks, joined at the end through LDS: 32 KB a wave
// written and read, in two rounds, 3000 of the 13900 cycles that a workgroup of 166 tokens took, and 128 registers of sums that
// the scores and the loads have to do without.  ONE_ROUND, SHARED_ROUNDS: the waves make the probabilities of a round's
// eight blocks, relative to each block's own maximum, and hand them round (2 KB a block); then each makes 32 dims of O over all of them, 16
// registers, with 2^(m_b - m) a factor of the block's product in 32 bits.  Nothing is joined, the values travel under the scores and
// the queries stay in registers, but a round's loads wait for the end of the round before, and its phases don't overlap.
// Whole call, us, OWN_BLOCKS -> ONE_ROUND (8 blocks at most): 166 from 0 13.4 -> 10.8 (halves), 14.7 -> 12.7 (8-bit), 14.8 -> 12.7 (4-bit); in parts of 8
// blocks, 10 at 3000, 17.7 -> 15.0, 19.5 -> 17.0, 19.2 -> 16.7.  -> SHARED_ROUNDS, halves: 300 from 0 16.8 -> 14.0, 700 25.4 -> 22.2, 900 32.2 -> 29.0,
// 30 at 500 17.8 -> 16.8, 500 at 300 23.4 -> 23.5, 500 at 800 29.7 -> 32.1; 4-bit: 300 from 0 17.6 -> 16.8, 520 21.8 -> 21.9, 766 28.7 -> 25.7, 30 at
// 500 20.2 -> 20.2, 500 at 300 25.5 -> 26.7; 8-bit spills 26 registers that way (300 from 0 17.8 -> 18.9) and has none.  So the line lies at the
// keys that a row group sees in the mean, and in parts, whose row groups all see the same, at the blocks of a part: of 16 blocks halves 12 at
// 20000 26.1 -> 23.6, 64 at 2000 22.5 -> 19.4, 4-bit 28.4 -> 26.7, 24.2 -> 22.7 (8-bit 28.2 -> 27.1, but 23.5 -> 24.8), of 24 7 at 40000 34.0 -> 31.5 and 32.9 ->
// 32.5, of 32 120 at 3000 29.2 -> 28.9 and 32.4 -> 32.8, of 40 30 at 16000 32.4 -> 33.7, of 72 55 at 17388 43.8 -> 50.6.  Distance from 64 bits: the same or less (halves, 500 at 300: 1.66e-4 -> 1.13e-4).
constexpr int OWN_BLOCKS = 0, ONE_ROUND = 1, SHARED_ROUNDS = 2;
constexpr uint32_t SHARED_KEYS_HALF = 544, SHARED_KEYS_4 = 464, SHARED_PART_HALF = 32, SHARED_PART_4 = 24;

struct SmallArgs {
    const uint16_t *q;  // f16 [tokens][heads][256]
    const unsigned char *kdata, *vdata;
    const uint16_t *kscales, *kbiases, *vscales, *vbiases;
    const float *q_and_gate;
    float *out;
    uint32_t heads, kv_heads, pos, tokens;
    float scale;
    // SPLIT: the keys in `nparts` parts of `part_blocks` blocks, a workgroup each; their O, m and l as PrefillArgs' parts
    uint32_t part_blocks, nparts;
    float *part_o, *part_ml;
};

template <int BITS, bool SHARED>
struct SmallLds {
    // the values of a wave's block: f16 rows as in memory.  Halves (copied in by 16-byte pieces in whole kilobytes), and codes where the
    // values are SHARED (rows of 576 would leave the maxima no room): rows of 512 bytes, row k rotated by 64 (k % 4); codes of a wave's own
    // blocks: rows of 576.  Either way the four rows of a transposing read, 32 bytes each, and those of its neighbours fall on different
    // banks.
    static constexpr int VROW = BITS == 16 || SHARED ? 512 : 576;
    static constexpr int VTILE = BK * VROW;
    static constexpr int Q_OFF = 0, V_OFF = 16 * 1024;
    // SHARED: the blocks' probabilities, two operands of 64 lanes x 16 bytes each, take the place of a tile or of the queries
    static_assert(SMALL_WAVES * 2 * 64 * 16 <= VTILE && SMALL_WAVES * 2 * 64 * 16 <= V_OFF, "the probabilities");
    // the merge, over both: four waves' O at a time, [wave][8 dim tiles][4][64 lanes][16 bytes], and [wave][row][m, l]
    static constexpr int ML_OFF = SHARED ? V_OFF + SMALL_WAVES * VTILE : 4 * 32 * 1024;
    static constexpr int MERGE_BYTES = ML_OFF + SMALL_WAVES * 32 * 8;
    static constexpr int TILES_BYTES = V_OFF + SMALL_WAVES * VTILE;
    static constexpr int BYTES = TILES_BYTES > MERGE_BYTES ? TILES_BYTES : MERGE_BYTES;
    static_assert(BYTES <= 160 * 1024, "LDS of a CU");
};

// Where dims 8 u .. + 7 of the 32 query rows lie in LDS, [k-step][half][row][16 bytes]: MFMA k-step and lane half are those in which a
// key's lane holds the same dims, which is what a 16-byte piece of its row gives, whatever a value's size.
template <int BITS>
__device__ __forceinline__ uint32_t small_place(uint32_t u) {
    constexpr uint32_t STEPS = 16 / BITS;
    const uint32_t st = BITS == 16 ? u / 8 * 4 + u % 4 : u / (2 * STEPS) * STEPS + u % STEPS, hf = BITS == 16 ? u / 4 % 2 : u / STEPS % 2;
    return st * 1024 + hf * 512;
}

template <int BITS, bool SPLIT, int ROUNDS>
__global__ __launch_bounds__(SMALL_THREADS, 2) void prefill_small_kernel(SmallArgs a) {
    constexpr bool ONE = ROUNDS == ONE_ROUND, SHARED = ROUNDS != OWN_BLOCKS;
    using L = SmallLds<BITS, SHARED>;
    constexpr int RB = row_bytes<BITS>(), PIECES = RB / 16, STEPS = 16 / BITS, VALUES = 128 / BITS;  // pieces of a row; values of one
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
    if constexpr (SHARED) {  // (every argument is asked for here, in one trip: the compiler asks for each where it is used)
        asm volatile("" ::"s"(a.q), "s"(a.kdata), "s"(a.vdata), "s"(a.q_and_gate), "s"(a.out), "s"(a.heads), "s"(a.kv_heads), "s"(a.pos), "s"(a.tokens), "s"(a.scale));
        if constexpr (BITS != 16) asm volatile("" ::"s"(a.kscales), "s"(a.kbiases), "s"(a.vscales), "s"(a.vbiases));
        if constexpr (SPLIT) asm volatile("" ::"s"(a.part_blocks), "s"(a.nparts), "s"(a.part_o), "s"(a.part_ml));
    }
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 31, hf = lane >> 5;
    const uint32_t kvh = a.kv_heads, groups = (a.tokens + 3) / 4;
    uint32_t kv = blockIdx.y, at_group = blockIdx.x, part = 0;
    if constexpr (SPLIT) {
        // Workgroups go to the 8 XCDs in turn, and each XCD has its own L2: an XCD takes an eighth of the (part, kv head, row
        // group) in a row, since the row groups of a part read the same keys.
        const uint32_t item = blockIdx.x % 8 * (gridDim.x / 8) + blockIdx.x / 8, pair = item / groups;
        if (pair >= a.nparts * kvh) return;
        at_group = item % groups, kv = pair % kvh, part = pair / kvh;
    }
    const uint32_t tok0 = (groups - 1 - at_group) * 4;  // (the row groups that see the most keys first)
    const uint32_t tok = tok0 + (col >> 3);
    const float c = a.scale * 1.4426950408889634f;
    const uint32_t keys = a.pos + min(tok0 + 4, a.tokens);  // what the last of its tokens sees
    const uint32_t first = SPLIT ? part * a.part_blocks : 0;         // blocks of keys: this workgroup's are first .. nblocks - 1
    uint32_t nblocks = (keys + BK - 1) / BK;
    if constexpr (SPLIT) {
        if (nblocks <= first) {
            // a part of its tile that this row group sees no key of: no weight in the merge (which multiplies what lies there)
            const size_t item = (size_t(part) * ((a.tokens + TQ - 1) / TQ) + tok0 / TQ) * kvh + kv;
            float4 *po = reinterpret_cast<float4 *>(a.part_o) + (item * WAVES + tok0 % TQ / 4 * 2) * 16 * 64;
            for (uint32_t i = tid; i < 2 * 16 * 64; i += SMALL_THREADS) po[i] = float4{0, 0, 0, 0};
            if (tid < 32) *reinterpret_cast<float2 *>(a.part_ml + ((item * 4 + tok0 % TQ / 4) * 32 + tid) * 2) = float2{4.0f * NO_SCORE, 0.0f};
            return;
        }
        nblocks = min(nblocks, first + a.part_blocks);
    }
    const uint32_t active = min(nblocks - first, uint32_t(SMALL_WAVES));  // waves that have a block
    const uint32_t lds0 = uint32_t(reinterpret_cast<uintptr_t>(lds));
    const uint32_t vtile = lds0 + L::V_OFF + wave * L::VTILE;

    // ---- what a block needs of memory ----
    // Keys: lane (key col, half hf) multiplies a piece of its row at a time.  Codes: the pieces 2i + hf, fetched as they are
    // multiplied.  Halves: the pieces 8i + 4 hf .. + 3; four lanes fetch 64 bytes of a row together, a row a register, and
    // turn them round, for a load of 16 bytes of each of many rows is taken a row a cycle (codes have half and a quarter of
    // the loads: turned, 0.3 us of 33 slower).
    u32x4 kreg[PIECES / 2];
    u32x2 kss = {0, 0}, kzs = {0, 0};  // scales and biases of the key's four groups
    constexpr int V_LOADS = BK * PIECES / 64, V_KEYS = 64 / PIECES;  // loads that bring the values; keys of one
    u32x4 vreg[BITS == 16 ? 1 : V_LOADS];
    uint32_t vss[BITS == 16 ? 1 : V_LOADS], vzs[BITS == 16 ? 1 : V_LOADS];
    const uint32_t vp = lane % PIECES, vk = lane / PIECES;  // codes: the lane's piece and key of a load
    auto row_of = [&](uint32_t key) { return min(key, keys - 1) * kvh + kv; };  // (past the end: the last row, masked; a cache is under 2 GB)
    auto fetch_keys = [&](uint32_t b) {
        if constexpr (BITS == 16) {
            uint32_t at = lane;  // (not kept in registers across the loop)
            asm volatile("" : "+v"(at));
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const u32x4 *src = reinterpret_cast<const u32x4 *>(a.kdata + (row_of(b * BK + (at & 28) + j) * RB + 64 * (at >> 5) + 16 * (at & 3)));
#pragma unroll
                for (int i = 0; i < PIECES / 8; i++) kreg[4 * i + j] = src[8 * i];
            }
        } else {
            const uint32_t row = row_of(b * BK + col);
            const u32x4 *src = reinterpret_cast<const u32x4 *>(a.kdata + (row * RB + 16 * hf));
#pragma unroll
            for (int i = 0; i < PIECES / 2; i++) kreg[i] = src[2 * i];
            kss = *reinterpret_cast<const u32x2 *>(a.kscales + row * 4);
            kzs = *reinterpret_cast<const u32x2 *>(a.kbiases + row * 4);
        }
    };
    // halves: load u of the block's values, straight to the tile: place p of row k holds piece p - 4 (k % 4)
    auto fetch_value = [&](uint32_t b, int u, uint32_t at) {
        const uint32_t k = 2 * u + (at >> 5);
        const uint64_t src = reinterpret_cast<uint64_t>(a.vdata) + row_of(b * BK + k) * RB + ((at - 4 * (k & 3)) & 31) * 16;
        asm volatile("s_mov_b32 m0, %0\n"
                     "s_nop 0\n"
                     "global_load_lds_dwordx4 %1, off\n"
                     :
                     : "s"(vtile + u * 1024), "v"(src)
                     : "memory", "m0");
    };
    auto fetch_values = [&](uint32_t b) {
        if constexpr (BITS == 16) {
            uint32_t at = lane;
            asm volatile("" : "+v"(at));
#pragma unroll
            for (int u = 0; u < V_LOADS; u++) fetch_value(b, u, at);
            // (loads into registers and into LDS do not come back in one order, and the compiler counts only the former:
            // all that is out is waited for here, in front of anything it may do with the keys)
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        } else {
#pragma unroll
            for (int u = 0; u < V_LOADS; u++) {
                const uint32_t row = row_of(b * BK + u * V_KEYS + vk);
                vreg[u] = *reinterpret_cast<const u32x4 *>(a.vdata + (row * RB + vp * 16));
                vss[u] = a.vscales[row * 4 + vp * 4 / PIECES], vzs[u] = a.vbiases[row * 4 + vp * 4 / PIECES];
            }
        }
    };
    // The 8 values of sub-step `sub` of a piece, as halves; s, z: scale and bias (f16 bits).  A code in the mantissa of 1024 is
    // 1024 + code; s * code + z is rounded once, as a half (the prepare kernel rounds it to f32 in between: they differ where
    // that f32 lies on the middle of two halves).
    auto eight = [&](const u32x4 &piece, int sub, uint32_t s, uint32_t z) {
        if constexpr (BITS == 16) {
            return __builtin_bit_cast(half8, piece);
        } else {
            const _Float16 sh = __builtin_bit_cast(_Float16, uint16_t(s)), zh = __builtin_bit_cast(_Float16, uint16_t(z));
            uint32_t o[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                constexpr int PER = 32 / BITS;
                const uint32_t word = piece[(8 * sub + 2 * i) / PER];
                const uint32_t at = (8 * sub + 2 * i) % PER * BITS / 8;  // the byte of the first code
                half2_ x;
                if constexpr (BITS == 8) {
                    x = __builtin_bit_cast(half2_, __builtin_amdgcn_perm(0x64646464u, word, at | 4u << 8 | (at + 1) << 16 | 4u << 24));
                    x = x + half2_{(_Float16)-1024.0f, (_Float16)-1024.0f};
                } else {  // (both nibbles of a byte, the second times 16)
                    x = __builtin_bit_cast(half2_, (__builtin_amdgcn_perm(word, word, at * 0x01010101u) & 0x00f0000fu) | 0x64006400u);
                    x = __builtin_elementwise_fma(x, half2_{(_Float16)1.0f, (_Float16)0.0625f}, half2_{(_Float16)-1024.0f, (_Float16)-64.0f});
                }
                o[i] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(x, half2_{sh, sh}, half2_{zh, zh}));
            }
            return __builtin_bit_cast(half8, u32x4{o[0], o[1], o[2], o[3]});
        }
    };

    typedef short short4 __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) short4 *LdsShort4;
    // ---- S^T = K Q^T of the block whose keys are in registers ----
    auto scores = [&](auto &&query) {
        floatx16 s;
#pragma unroll
        for (int r = 0; r < 16; r++) s[r] = 0.0f;
#pragma unroll
        for (int st = 0; st < 16; st++) {
            const int i = st / STEPS;
            uint32_t ks = 0, kz = 0;
            if constexpr (BITS != 16) {
                const int g = i * 2 * VALUES / SAETTA_QUANT_GROUP;
                ks = kss[g >> 1] >> (16 * (g & 1)), kz = kzs[g >> 1] >> (16 * (g & 1));
            }
            if (BITS == 16 && st % 4 == 0) turn(&kreg[i], lane);
            s = __builtin_amdgcn_mfma_f32_32x32x16_f16(eight(kreg[i], st % STEPS, ks, kz), query(st), s, 0, 0, 0);
        }
        return s;
    };
    // register r of a block's scores is key 4 hf + r % 4 + 8 (r / 4) of the block, the lane's row col
    auto mask = [&](floatx16 &s, uint32_t b) {
        const uint32_t key0 = b * BK;
        if (key0 + BK > a.pos + tok0 + 1) {
            const uint32_t len = a.pos + tok + 1, vis = len > key0 ? len - key0 : 0;
#pragma unroll
            for (int r = 0; r < 16; r++) s[r] = uint32_t(4 * hf + (r & 3) + 8 * (r >> 2)) < vis ? s[r] : NO_SCORE;
        }
    };
    // the operand of k-step sp, its sum added to l
    auto probabilities = [&](const floatx16 &s, int sp, float m, float &l) {
        uint32_t w[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float x = __builtin_amdgcn_exp2f(fmaf(s[8 * sp + 2 * i], c, -m)), y = __builtin_amdgcn_exp2f(fmaf(s[8 * sp + 2 * i + 1], c, -m));
            l += x + y;
            w[i] = pack_half2(x, y);
        }
        return __builtin_bit_cast(half8, u32x4{w[0], w[1], w[2], w[3]});
    };
    // codes: the block's values to the wave's tile
    auto store_values = [&]() {
        if constexpr (BITS != 16) {
#pragma unroll
            for (int u = 0; u < V_LOADS; u++) {
                const uint32_t in_row = SHARED ? (vp * VALUES * 2 + 64 * (vk & 3)) & 511 : vp * VALUES * 2;
                half8 *dst = reinterpret_cast<half8 *>(lds + L::V_OFF + wave * L::VTILE + (u * V_KEYS + vk) * L::VROW + in_row);
#pragma unroll
                for (int sub = 0; sub < STEPS; sub++) dst[sub] = eight(vreg[u], sub, vss[u], vzs[u]);
            }
        }
    };
    // What a wave finishes: O^T of dims 32 wave .. + 31, relative to `top`, with the sums l_all (the lane's row col)
    floatx16 fin;
#pragma unroll
    for (int r = 0; r < 16; r++) fin[r] = 0.0f;
    const float least = 0.25f * NO_SCORE * c;  // (above a masked score, as in the kernel above)
    float top = SHARED ? least : 4.0f * NO_SCORE, l_all = 0.0f;
    float2 *ml = reinterpret_cast<float2 *>(lds + L::ML_OFF);
    // Gates and outputs: lane l has dims 4 (l % 8) .. + 3 of those of rows 8 j + l / 8 (a row group's rows 8 j .. + 7 are a
    // token's), 128 bytes of a row a load or store.  16 bytes of each of 32 rows, as the accumulators lie, are taken a row a cycle.
    float4 g[4];
    const uint32_t in_token = (lane >> 3) * DIM + 32 * wave + 4 * (lane & 7);
    auto first_row = [&](int j) { return size_t(min(tok0 + j, a.tokens - 1)) * a.heads + kv * SAETTA_GQA_GROUP; };
    auto ask_gates = [&]() {
        if constexpr (!SPLIT) {
#pragma unroll
            for (int j = 0; j < 4; j++) g[j] = *reinterpret_cast<const float4 *>(a.q_and_gate + first_row(j) * 2 * DIM + DIM + ((lane >> 3) * DIM + in_token));
        }
    };

    if constexpr (SHARED) {
        // ---- the waves share the probabilities and the values of a round's blocks, and each makes 32 dims of O ----
        // Q^T operands: to registers by way of LDS.  Wave w fetches 64 bytes of each row, four lanes a row.
        half8 q[16];
        {
            half8 qv[2];
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const uint32_t r = 16 * i + (lane >> 2);
                qv[i] = *reinterpret_cast<const half8 *>(a.q + (size_t(min(tok0 + (r >> 3), a.tokens - 1)) * a.heads + kv * SAETTA_GQA_GROUP + (r & 7)) * DIM + 32 * wave + 8 * (lane & 3));
            }
            auto put = [&]() {
#pragma unroll
                for (int i = 0; i < 2; i++) *reinterpret_cast<half8 *>(lds + L::Q_OFF + small_place<BITS>(4 * wave + (lane & 3)) + (16 * i + (lane >> 2)) * 16) = qv[i];
            };
            if (uint32_t(wave) < active) {  // (each side with its own wait: behind a branch the compiler would wait for the keys too)
                fetch_keys(first + wave);
                put();
                if constexpr (BITS != 16) fetch_values(first + wave);
                asm volatile("; keys on their way" ::: "memory");
            } else {
                put();
                asm volatile("; no keys" ::: "memory");
            }
            lds_barrier();
            if constexpr (ONE) ask_gates();
            if (uint32_t(wave) < active) {
#pragma unroll
                for (int st = 0; st < 16; st++) q[st] = *reinterpret_cast<const half8 *>(lds + L::Q_OFF + st * 1024 + lane * 16);
            }
            if (!ONE || active == SMALL_WAVES) lds_barrier();  // the probabilities go over them
        }
        // the blocks' probabilities: in the place of the last wave's values, or, where it has some, of the queries
        const uint32_t p_at = !ONE || active == SMALL_WAVES ? L::Q_OFF : L::V_OFF + (SMALL_WAVES - 1) * L::VTILE;
        for (uint32_t b0 = first;;) {
            const uint32_t b = b0 + wave, here = ONE ? active : min(nblocks - b0, uint32_t(SMALL_WAVES));
            const bool mine = uint32_t(wave) < here, more = !ONE && b + SMALL_WAVES < nblocks;
            if (mine) {
                if constexpr (BITS == 16) {
                    // Loads into registers and into LDS do not come back in one order, and the compiler counts only the former: the
                    // keys are waited for here, in front of the values, which travel under the scores.
#pragma unroll
                    for (int i = 0; i < PIECES / 2; i++) asm volatile("" : "+v"(kreg[i]));
                }
                if constexpr (BITS != 16) asm volatile("" : "+v"(kss), "+v"(kzs));  // (nothing of them before the queries have left)
                floatx16 s = scores([&](int st) {
                    if constexpr (BITS == 16) fetch_value(b, st, lane);  // (a load beside each product)
                    return q[st];
                });
                if constexpr (BITS != 16) {
                    if (more) fetch_keys(b + SMALL_WAVES);
                }
                mask(s, b);
                // relative to the block's own maximum, so that a row's largest probability in it is 1, which f16 holds exactly
                float m = s[0];
#pragma unroll
                for (int r = 1; r < 16; r++) m = fmaxf(m, s[r]);
                m = fmaxf(max_across_halves(m) * c, least);
                float l = 0.0f;
#pragma unroll
                for (int sp = 0; sp < 2; sp++) *reinterpret_cast<half8 *>(lds + p_at + (2 * wave + sp) * 1024 + lane * 16) = probabilities(s, sp, m, l);
                l += __shfl_xor(l, 32);
                if (hf == 0) ml[wave * 32 + col] = float2{m, l};
                if constexpr (BITS != 16) {
                    store_values();
                    if (more) fetch_values(b + SMALL_WAVES);
                } else {
                    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                }
            }
            lds_barrier();  // the probabilities and the values are in LDS
            if constexpr (BITS == 16) {
                if (more) fetch_keys(b + SMALL_WAVES);
            }
            if (!ONE && b0 + SMALL_WAVES >= nblocks) ask_gates();
            // ---- O^T = sum over the blocks of 2^(m_b - top) V_b^T P_b^T ----
            float weight[SMALL_WAVES];
            {
                float2 x[SMALL_WAVES];
                const float before = top;
#pragma unroll
                for (int w = 0; w < SMALL_WAVES; w++) {
                    x[w] = ml[w * 32 + col];
                    if (uint32_t(w) >= here) x[w] = float2{4.0f * NO_SCORE, 0.0f};
                    top = fmaxf(top, x[w].x);
                }
                if constexpr (!ONE) {
                    const float alpha = __builtin_amdgcn_exp2f(before - top);
                    l_all *= alpha;
#pragma unroll
                    for (int r = 0; r < 16; r++) fin[r] *= alpha;
                }
#pragma unroll
                for (int w = 0; w < SMALL_WAVES; w++) weight[w] = __builtin_amdgcn_exp2f(x[w].x - top), l_all += x[w].y * weight[w];
            }
            // k-step sp, lane half hf: keys 16 sp + 4 hf .. + 3 and 8 further
            const uint32_t e = (lane >> 2) & 3, dim = ((lane >> 4) & 1) * 16 + (lane & 3) * 4;
            const uint32_t vrow = lds0 + L::V_OFF + (4 * hf + e) * L::VROW + (((32 * wave + dim) * 2 + 64 * e) & 511);
            auto block = [&](uint32_t w) {
                floatx16 t;
#pragma unroll
                for (int r = 0; r < 16; r++) t[r] = 0.0f;
                u32x2 r[4];
#pragma unroll
                for (int i = 0; i < 4; i++) r[i] = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<LdsShort4>(vrow + w * L::VTILE + 8 * i * L::VROW)));
#pragma unroll
                for (int sp = 0; sp < 2; sp++) {
                    const half8 p = *reinterpret_cast<const half8 *>(lds + p_at + (2 * w + sp) * 1024 + lane * 16);
                    const half8 v = __builtin_bit_cast(half8, u32x4{r[2 * sp].x, r[2 * sp].y, r[2 * sp + 1].x, r[2 * sp + 1].y});
                    t = __builtin_amdgcn_mfma_f32_32x32x16_f16(v, p, t, 0, 0, 0);
                }
                return t;
            };
#pragma unroll
            for (int w = 0; w < SMALL_WAVES; w += 2) {
                if (uint32_t(w) >= here) break;
                if constexpr (!ONE) __builtin_amdgcn_sched_barrier(0);  // (no reads of the next pair's before this one's are used)
                const floatx16 t0 = block(w);
                if (uint32_t(w + 1) < here) {
                    const floatx16 t1 = block(w + 1);
#pragma unroll
                    for (int r = 0; r < 16; r++) fin[r] += t0[r] * weight[w] + t1[r] * weight[w + 1];
                } else {
#pragma unroll
                    for (int r = 0; r < 16; r++) fin[r] += t0[r] * weight[w];
                }
            }
            if (ONE || (b0 += SMALL_WAVES) >= nblocks) break;
            lds_barrier();  // the round has been read
        }
    } else {
        if (uint32_t(wave) < active) fetch_keys(first + wave);
        // Q^T operands: through LDS, where all waves read them.  Wave w fetches 64 bytes of each row, four lanes a row.
        {
            half8 qv[2];
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const uint32_t r = 16 * i + (lane >> 2);
                qv[i] = *reinterpret_cast<const half8 *>(a.q + (size_t(min(tok0 + (r >> 3), a.tokens - 1)) * a.heads + kv * SAETTA_GQA_GROUP + (r & 7)) * DIM + 32 * wave + 8 * (lane & 3));
            }
            if (uint32_t(wave) < active) fetch_values(first + wave);
#pragma unroll
            for (int i = 0; i < 2; i++) *reinterpret_cast<half8 *>(lds + L::Q_OFF + small_place<BITS>(4 * wave + (lane & 3)) + (16 * i + (lane >> 2)) * 16) = qv[i];
        }
        lds_barrier();

        floatx16 acc[8];
#pragma unroll
        for (int mt = 0; mt < 8; mt++) {
#pragma unroll
            for (int r = 0; r < 16; r++) acc[mt][r] = 0.0f;
        }
        float m = least, l = 0.0f;
        for (uint32_t b = first + wave; b < nblocks; b += SMALL_WAVES) {
            floatx16 s = scores([&](int st) { return *reinterpret_cast<const half8 *>(lds + L::Q_OFF + st * 1024 + lane * 16); });
            if (b + SMALL_WAVES < nblocks) fetch_keys(b + SMALL_WAVES);
            mask(s, b);
            float bm = s[0];
#pragma unroll
            for (int r = 1; r < 16; r++) bm = fmaxf(bm, s[r]);
            bm = fmaxf(max_across_halves(bm) * c, NO_SCORE);
            if (__any(bm > m + TAU)) {
                const float m_new = bm > m + TAU ? bm : m, alpha = __builtin_amdgcn_exp2f(m - m_new);
                m = m_new, l *= alpha;
#pragma unroll
                for (int mt = 0; mt < 8; mt++) {
#pragma unroll
                    for (int r = 0; r < 16; r++) acc[mt][r] *= alpha;
                }
            }
            half8 p[2];
            float sum = 0.0f;
#pragma unroll
            for (int sp = 0; sp < 2; sp++) p[sp] = probabilities(s, sp, m, sum);
            l += sum;
            // ---- the values to the wave's tile (halves: they are there) ----
            if constexpr (BITS != 16) {
                store_values();
                if (b + SMALL_WAVES < nblocks) fetch_values(b + SMALL_WAVES);
            }
            // ---- O^T += V^T P^T: k-step sp, lane half hf: keys 16 sp + 4 hf .. + 3 and 8 further; a wave's LDS accesses run in order ----
            uint32_t at = lane;
            if (BITS == 16) asm volatile("" : "+v"(at));
            const uint32_t e = (at >> 2) & 3, dim = ((at >> 4) & 1) * 16 + (at & 3) * 4;
            const uint32_t vrow = vtile + (4 * (at >> 5) + e) * L::VROW;
#pragma unroll
            for (int mt = 0; mt < 8; mt++) {
                const uint32_t d = BITS == 16 ? ((32 * mt + dim) * 2 + 64 * e) & 511 : (32 * mt + dim) * 2;
                u32x2 r[4];
#pragma unroll
                for (int i = 0; i < 4; i++) r[i] = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<LdsShort4>(vrow + d + 8 * i * L::VROW)));
#pragma unroll
                for (int sp = 0; sp < 2; sp++) {
                    const half8 v = __builtin_bit_cast(half8, u32x4{r[2 * sp].x, r[2 * sp].y, r[2 * sp + 1].x, r[2 * sp + 1].y});
                    acc[mt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(v, p[sp], acc[mt], 0, 0, 0);
                }
            }
            if constexpr (BITS == 16) {
                // (what comes from memory into the tile is not in the order of the wave's LDS accesses: its reads have to be back)
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                if (b + SMALL_WAVES < nblocks) fetch_values(b + SMALL_WAVES);
            }
        }

        // ---- the waves' parts joined: wave w finishes dims 32 w .. 32 w + 31 ----
        ask_gates();
        lds_barrier();  // every wave is through with its tile and the query operands
        const float l_row = l + __shfl_xor(l, 32);
        if (hf == 0) ml[wave * 32 + col] = float2{m, l_row};
        auto tile_of = [&](int w, int mt) { return reinterpret_cast<float4 *>(lds + (w & 3) * 32768 + mt * 4096) + lane; };
        auto hand_out = [&]() {  // this wave's O, all dims
#pragma unroll
            for (int mt = 0; mt < 8; mt++) {
#pragma unroll
                for (int i = 0; i < 4; i++) tile_of(wave, mt)[i * 64] = float4{acc[mt][4 * i], acc[mt][4 * i + 1], acc[mt][4 * i + 2], acc[mt][4 * i + 3]};
            }
        };
        float weight[SMALL_WAVES];
        auto take_in = [&](int from) {  // the dims this wave finishes, from waves from .. from + 3
#pragma unroll
            for (int w = 0; w < 4; w++) {
                if (uint32_t(from + w) < active) {
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const float4 x = tile_of(w, wave)[i * 64];
                        fin[4 * i] += x.x * weight[from + w], fin[4 * i + 1] += x.y * weight[from + w];
                        fin[4 * i + 2] += x.z * weight[from + w], fin[4 * i + 3] += x.w * weight[from + w];
                    }
                }
            }
        };
        if (wave < 4 && uint32_t(wave) < active) hand_out();
        lds_barrier();
        {
            float2 x[SMALL_WAVES];
#pragma unroll
            for (int w = 0; w < SMALL_WAVES; w++) x[w] = ml[w * 32 + col];  // (a wave without a block: l = 0)
#pragma unroll
            for (int w = 0; w < SMALL_WAVES; w++) top = fmaxf(top, x[w].x);
#pragma unroll
            for (int w = 0; w < SMALL_WAVES; w++) weight[w] = __builtin_amdgcn_exp2f(x[w].x - top), l_all += x[w].y * weight[w];
        }
        take_in(0);
        if (active > 4) {
            lds_barrier();
            if (wave >= 4 && uint32_t(wave) < active) hand_out();
            lds_barrier();
            take_in(4);
        }
    }
    if constexpr (SPLIT) {
        // (rows past the chunk's end leave what their masked lanes hold; nothing reads it)
        const size_t item = (size_t(part) * ((a.tokens + TQ - 1) / TQ) + tok0 / TQ) * kvh + kv;
        const uint32_t group = tok0 % TQ / 4;
        float4 *po = reinterpret_cast<float4 *>(a.part_o) + ((item * WAVES + group * 2 + (wave >> 2)) * 16 + (wave & 3) * 4) * 64 + lane;
#pragma unroll
        for (int i = 0; i < 4; i++) po[i * 64] = float4{fin[4 * i], fin[4 * i + 1], fin[4 * i + 2], fin[4 * i + 3]};
        if (wave == 0 && hf == 0) *reinterpret_cast<float2 *>(a.part_ml + ((item * 4 + group) * 32 + col) * 2) = float2{top, l_all};
        return;
    }
    // Turned round (in the place of what the first wave handed to this one, which nobody else reads): piece p (dims 4 p .. + 3) of row
    // r at 16 ((r + 2 p) % 32) of the piece's 512 bytes, so that neither side meets in its banks.
    const float inv = 1.0f / l_all;
    unsigned char *turned = lds + wave * 4096;
    if constexpr (SHARED) lds_barrier();  // the values have been read
    else wave_sync();  // every lane has taken what was handed over
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const uint32_t piece = 2 * i + hf;
        *reinterpret_cast<float4 *>(turned + piece * 512 + (col + 2 * piece) % 32 * 16) = float4{fin[4 * i] * inv, fin[4 * i + 1] * inv, fin[4 * i + 2] * inv, fin[4 * i + 3] * inv};
    }
    wave_sync();
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const uint32_t piece = lane & 7;
        const float4 x = *reinterpret_cast<const float4 *>(turned + piece * 512 + (8 * j + (lane >> 3) + 2 * piece) % 32 * 16);
        float4 w;
        w.x = x.x * __builtin_amdgcn_rcpf(1.0f + __expf(-g[j].x));
        w.y = x.y * __builtin_amdgcn_rcpf(1.0f + __expf(-g[j].y));
        w.z = x.z * __builtin_amdgcn_rcpf(1.0f + __expf(-g[j].z));
        w.w = x.w * __builtin_amdgcn_rcpf(1.0f + __expf(-g[j].w));
        if (tok0 + j < a.tokens) *reinterpret_cast<float4 *>(a.out + first_row(j) * DIM + in_token) = w;
    }
}

// Workspaces the library owns when the caller passes none: one per (device, stream), grown on demand,
// so that calls on different streams never share one (work on one stream runs in order).  They are
// kept until the process ends: a caller with many short-lived streams passes its own.
constexpr int OWNED_DEVICES = 64;  // as many devices as the library's set-up admits
std::map<std::pair<int, hipStream_t>, OwnedWorkspace> g_owned;
std::mutex g_owned_mutex;

// The images, then a line for the attention kernel's count of tiles handed out.
size_t images_bytes(uint32_t pos, uint32_t tokens, uint32_t kv_heads) {
    const size_t blocks = (size_t(pos) + tokens + BK - 1) / BK;
    return blocks * kv_heads * IMG_BYTES;
}
size_t plain_workspace_bytes(uint32_t pos, uint32_t tokens, uint32_t kv_heads) { return images_bytes(pos, tokens, kv_heads) + 256; }

constexpr size_t PART_O_BYTES = size_t(TQ) * SAETTA_GQA_GROUP * DIM * 4, PART_ML_BYTES = size_t(TQ) * SAETTA_GQA_GROUP * 8;
constexpr uint32_t SMALL_MAX_PARTS = 64;
size_t parts_bytes(uint32_t tokens, uint32_t kv_heads, uint32_t nparts) {
    return size_t((tokens + TQ - 1) / TQ) * kv_heads * nparts * (PART_O_BYTES + PART_ML_BYTES);
}
uint32_t parts_of(uint32_t pos, uint32_t tokens, uint32_t part_blocks) {
    return (uint32_t((uint64_t(pos) + tokens + BK - 1) / BK) + part_blocks - 1) / part_blocks;
}

// The tiles' keys in parts of `blocks` blocks, n of them at most, which take `bytes` behind the images; not in parts where blocks is 0.
struct TileParts {
    uint32_t blocks, n;
    size_t bytes;
};
// How a chunk's launches are laid out: the row groups' own launch (small), with their keys in parts of `small_part_blocks`
// blocks where that is not 0 and there is room for them; or tiles, with their keys in the parts of tiles of WIDE_TQ tokens (wide) where
// those are ahead and there is room for them, else in those of tiles of TQ (narrow) where there is room for these, else whole.  Wide parts
// are often more than narrow ones, for a few per cent; whole keys are 1.2 to 5 times as slow (halves, wide | narrow | whole: 447 tokens at
// 86225 616 us in 229 MB | 632 in 207 | 1870, 288 at 129584 641 in 318 MB | 730 in 290 | 3130, 2210 at 5272 261 in 126 MB | 266 in 89 | 307).
struct FlashPlan {
    bool small;  // without parts, the row groups' launch is ahead of the tiles
    uint32_t small_part_blocks, cus;
    TileParts narrow, wide;
    size_t plain, small_parts;  // bytes of workspace: the images and the tile count; the row groups' parts, instead of the images and all
    size_t tiles() const { return plain + (wide.blocks ? wide.bytes : narrow.bytes); }
    size_t bytes() const { return tiles() > small_parts ? tiles() : small_parts; }
    bool takes_wide(size_t have) const { return wide.blocks && have >= plain + wide.bytes; }
    bool takes_narrow(size_t have) const { return narrow.blocks && have >= plain + narrow.bytes; }
};

// A tile is one workgroup's work, and 16 tokens of 2 kv heads are all a CU gets of it: chunks under 2048 tokens leave CUs
// idle, and between 2048 and 4096 a second round of tiles fills a part of them.  The rule takes the smallest of what the
// rounds of workgroups would take, in us, unsplit and with the keys in 2 to 32 parts, from figures measured on the MI355X:
// a workgroup's block of 32 keys takes 0.6 us while the chip has power to spare (up to ~170 workgroups) and the chip as a
// whole 284 blocks a us beyond that; the ends of an item (its first loads, the store of its part) 12 us, with the gate
// 14.5; the merge a launch and 128 KB read back per item; the images 4.5 us and 0.3 ns a key and kv head.
// (The ends have become 6 and 2.5 us shorter since, the merge 1; with these figures and narrow tiles alone the rule takes what is the fastest
// or within 2 % of it at 33 of 38 sizes from 20 to 3500 tokens, 0 to 10000 keys before them, both kinds of cache; the furthest off were
// 2300 tokens at 3000, 216 us instead of 201 in two parts, which wide tiles now take in 205, and 128 at 4000, 36 instead of 33, which
// row groups in parts now take.)
// Wide tiles (WIDE_TQ tokens, a row group a wave; always in parts, so that there are as many items): a copied part of keys or values serves eight
// row groups instead of four, half the global -> LDS copies, and the chip, which is bound by its power, does 5 % more blocks; a block
// alone takes 1.3 us for twice the rows and an item's ends 18.  Whole call, us, without -> with: 2048 tokens at 118784 (AttGemm) 3568 -> 3397, 1237 at
// 60007 (4-bit) 1142 -> 1082, 800 at 80000 1018 -> 978, 1024 at 30000 481 -> 465, 2300 at 3000 218 -> 205, 2100 at 1000 114 -> 106, 4096 at 20000 1307 ->
// 1254.  Not where the parts' merge costs more than that: 4096 at 4096 would take 467 instead of 387, 2048 at 10000 (355) is even.
// Measured, unsplit -> split by this rule, the whole call (8-bit cache): 100 tokens at 10000: 211 -> 47 us, at 100000
// (4-bit): 1886 -> 225; 500 at 40000: 770 -> 330; 2100 at 9000: 497 -> 405.  A full chunk (4096 tokens of 2 kv heads: two whole rounds) is
// split from some 19300 keys before it on, into two parts of wide tiles.
constexpr float MERGE_ITEM_US = 0.03f;
// n items in order of length, from `high` down to `low` blocks, handed out one by one to `cus` workgroups: us, if a block
// takes block_us alone and chip_us of the whole chip
float rounds_us(uint32_t cus, uint32_t n, float high, float low, float ends_us, float block_us, float chip_us) {
    float us = 0.0f, at = 0.0f;
    for (uint32_t left = n; left > 0;) {
        const uint32_t now = left < cus ? left : cus;
        const float mid = high - (high - low) * (at + 0.5f * float(now)) / float(n);  // mean length of the round's items
        const float alone = mid * block_us, shared = mid * float(now) * chip_us;
        us += (alone > shared ? alone : shared) + ends_us;
        at += float(now), left -= now;
    }
    const float one = high * block_us + ends_us;
    return us > one ? us : one;
}
// The tiles' part of the plan; tiles_us: what they would take, images and all.
FlashPlan tiles_plan(uint32_t pos, uint32_t tokens, uint32_t kv_heads, float &tiles_us) {
    constexpr float BLOCK_US = 0.6f, CHIP_BLOCKS_PER_US = 284.0f / 256.0f, PART_US = 12.0f, TILE_US = 14.5f, MERGE_US = 4.0f;
    constexpr float PREPARE_US = 4.5f, PREPARE_KEY_US = 0.0003f;
    constexpr float WIDE_PART_US = 18.0f, WIDE_BLOCK_US = 1.3f, WIDE_GAIN = 0.95f;
    FlashPlan f{};
    f.cus = cu_count();
    f.plain = plain_workspace_bytes(pos, tokens, kv_heads);
    tiles_us = 0.0f;
    if (tokens == 0 || kv_heads == 0) return f;
    const uint32_t ntiles = (tokens + TQ - 1) / TQ;
    const uint32_t longest = tile_blocks(pos, tokens, ntiles - 1), shortest = tile_blocks(pos, tokens, 0);
    const float chip_us = 1.0f / (CHIP_BLOCKS_PER_US * float(f.cus));
    const float unsplit = rounds_us(f.cus, ntiles * kv_heads, float(longest), float(shortest), TILE_US, BLOCK_US, chip_us);
    float best = 0.95f * unsplit;
    auto in_parts = [&](bool wide, TileParts &of) {
        const uint32_t tq = wide ? WIDE_TQ : TQ, n = (tokens + tq - 1) / tq, seen_by_all = pos + (tokens < tq ? tokens : tq) - 1;
        const float high = float(tile_blocks(pos, tokens, n - 1, tq)), low = float(tile_blocks(pos, tokens, 0, tq));
        const float blocks = 0.5f * (high + low) * float(n * kv_heads), chip = wide ? WIDE_GAIN * 2.0f * chip_us : chip_us;
        const float ends_us = wide ? WIDE_PART_US : PART_US, block_us = wide ? WIDE_BLOCK_US : BLOCK_US, item_us = (wide ? 2.0f : 1.0f) * MERGE_ITEM_US;
        // What `rounds` rounds of `items` items take is no less than this, and more with every further part: where it is no gain, nothing
        // further is.  (The rounds one by one are most of what the plan costs the host.)
        auto no_gain = [&](uint32_t rounds, uint32_t items) {
            return 0.999f * (blocks * chip + float(rounds) * ends_us + MERGE_US + item_us * float(items)) >= best;
        };
        if (no_gain(1, n * kv_heads)) return;
        uint32_t last = 0;
        for (uint32_t parts = 2; parts <= 32; parts++) {
            const uint32_t pb = ((longest + parts - 1) / parts + 1) / 2 * 2;  // (a step of the kernel is two blocks)
            if (pb < 4 || pb >= longest || pb == last) continue;
            last = pb;
            if (n * kv_heads * parts > f.cus) {  // (not a round, and short)
                const uint32_t least = (seen_by_all / (pb * BK) + 1) * n * kv_heads;
                if (no_gain((least + f.cus - 1) / f.cus, least)) break;
            }
            const uint32_t items = prefill_items(pos, tokens, pb, tq) * kv_heads;
            const float mid = blocks / float(items);
            const float us = rounds_us(f.cus, items, mid, mid, ends_us, block_us, chip) + MERGE_US + item_us * float(items);
            if (us < best) best = us, of.blocks = pb;
        }
        if (!of.blocks) return;
        of.n = parts_of(pos, tokens, of.blocks);
        of.bytes = parts_bytes(tokens, kv_heads, of.n);
    };
    in_parts(false, f.narrow);
    if (!f.narrow.blocks) best = unsplit;
    // (what the row groups are weighed against stays what it was before there were wide tiles: which chunks need no workspace is
    // decided there)
    const float narrow = best;
    best *= 0.985f;
    if (tokens > TQ) in_parts(true, f.wide);  // (of one tile a wide one takes twice a block's time for nothing)
    // (never less than 5 us, what short contexts' images were counted at when the row groups came in: a chunk that goes to them
    // without parts needs no workspace, and who calls it without one, recording or under capture, goes on to)
    const float prepare_us = PREPARE_US + PREPARE_KEY_US * float(pos + tokens) * float(kv_heads);
    tiles_us = narrow + (prepare_us > 5.0f ? prepare_us : 5.0f);
    return f;
}

// The row groups' part, for one kind of cache.  Without parts their workgroups take 0.5 us for a block (0.6 with codes), with a
// quarter of a tile's rows, and don't slow each other down; their ends take 5 us, and there are no images to prepare.  (Codes:
// 0.59, for at 0.6 a tie sends 64 tokens at 1000 to the tiles, 27.2 -> 31.4.)  Tiles -> row groups, halves | 8-bit | 4-bit: 16 tokens
// at 500 22.9 -> 18.3 | 24.0 -> 20.7 | 24.1 -> 20.6; 500 from 0 32.4 -> 20.3 | 33.4 -> 22.0 | 33.5 -> 21.9; 700 from 0 35.9 -> 25.7 | 37.0 -> 28.5 |
// 37.3 -> 26.6; 500 at 800 39.2 -> 31.0 | 40.9 -> 32.9 | 41.1 -> 33.8.  Past the line: 1250 from 0 46.5 -> 50.3 | 47.8 -> 55.1 | 47.8 -> 54.1.
// With their keys in parts, a multiple of 8 blocks (a round of a workgroup's waves) each, a workgroup has a part of a row
// group's keys: the few tokens of a short turn behind a long prefix then fill the chip, each CU reading a part of the cache where
// it lies, where the tiles would write and read the images of all of it for two or four of them.  0.36 us a block up to some
// 200 workgroups, the chip 590 blocks a us; parts are some 7 us of ends, the merge 4.2 and a little for each part.  Two rounds of
// workgroups at most (one, nearly always), and row groups for half of the CUs: 64 tokens of 2 kv heads may have up to 16 parts, 256
// tokens 2 to 4.
// The whole call, halves, what it was -> parts: 7 tokens at 3000 31.3 -> 19.5 us, at 20000 49.8 -> 29.9, at 100000 186 -> 54.6; 30 at 3000 34.1 ->
// 22.2, at 40000 79.0 -> 54.4; 64 at 1500 32.7 -> 20.9, at 20000 64.6 -> 52.8; 128 at 1000 25.0 -> 22.8, at 3000 35.6 -> 31.6; 250 at 1500
// 36.2 -> 31.9.  Left alone: 128 at 10000 54.1 and 53.5, 250 at 4000 46.8 and 52.1 (with codes 49.3 and 53.8).
// Against its keys in parts a workgroup that goes through all of them is counted a quarter dearer, over codes a third: the figure above
// is the lowest that sends a chunk away from the tiles, and 300 to 600 keys take longer (12 tokens over 8-bit codes at 400 take 18.4 us, by
// the figure 12.7).  Whole calls, unsplit -> in two or three parts, halves | 8-bit | 4-bit: 12 tokens at 330 12.8 (left whole) | 16.6 -> 14.9 | 15.4 ->
// 14.4; 12 at 540 17.6 -> 13.2 | 19.6 -> 15.2 | 20.1 -> 14.7; 60 at 470 17.0 -> 14.2 | 19.8 -> 16.3 | 20.7 -> 16.1; 100 at 400 15.2 -> 14.3 | 20.2 -> 16.6 |
// 18.1 -> 16.5; 150 at 470 19.9 -> 17.2 | 20.3 -> 19.1 | 21.0 -> 19.1.  That holds up to row groups for 0.3 of the CUs (so that two parts fill
// 0.6 of them): 200 tokens of 2 kv heads at 400 would go from 20.4 to 24.6 over 8-bit codes and 250 from 22.6 to 25.4.
void choose_small(FlashPlan &f, uint32_t pos, uint32_t tokens, uint32_t kv_heads, int bits, float tiles_us) {
    const bool codes = bits != 16;
    const float SMALL_US = 5.0f, BLOCK_US = codes ? 0.59f : 0.5f;
    const float PART_US = codes ? 7.5f : 6.5f, PART_BLOCK_US = codes ? 0.37f : 0.36f, CHIP_BLOCKS_PER_US = (codes ? 570.0f : 590.0f) / 256.0f;
    constexpr float MERGE_US = 4.2f, MERGE_PART_US = 0.1f;
    if (tokens == 0 || kv_heads == 0) return;
    const uint32_t longest = tile_blocks(pos, tokens, (tokens - 1) / TQ), shortest = tile_blocks(pos, tokens, 0);
    const uint32_t groups = (tokens + 3) / 4 * kv_heads;
    const float small_us = rounds_us(f.cus, groups, float(longest), float(shortest), SMALL_US, BLOCK_US, 0.0f);
    f.small = small_us < tiles_us;
    if (2 * uint64_t(groups) > f.cus) return;
    const bool few = 10 * uint64_t(groups) <= 3 * uint64_t(f.cus);
    float best = !f.small ? 0.95f * tiles_us : !few ? 0.95f * small_us : codes ? 1.35f * small_us : 1.25f * small_us;
    const uint32_t least = (longest + SMALL_MAX_PARTS - 1) / SMALL_MAX_PARTS;
    for (uint32_t pb = (least + SMALL_WAVES - 1) / SMALL_WAVES * SMALL_WAVES; pb < longest; pb += SMALL_WAVES) {
        const uint32_t nparts = (longest + pb - 1) / pb, items = groups * nparts;
        if (items > 2 * f.cus) continue;
        const float us = rounds_us(f.cus, items, float(pb), float(pb), PART_US, PART_BLOCK_US, 1.0f / (CHIP_BLOCKS_PER_US * float(f.cus))) +
                         MERGE_US + MERGE_PART_US * float(nparts) + 0.25f * MERGE_ITEM_US * float(items);
        if (us < best) best = us, f.small_part_blocks = pb;
        if (3 * items <= f.cus) break;  // (longer parts leave more of the chip idle)
    }
    if (f.small_part_blocks) f.small_parts = parts_bytes(tokens, kv_heads, parts_of(pos, tokens, f.small_part_blocks));
}

FlashPlan flash_plan(uint32_t pos, uint32_t tokens, uint32_t kv_heads, int bits) {
    float tiles_us;
    FlashPlan f = tiles_plan(pos, tokens, kv_heads, tiles_us);
    choose_small(f, pos, tokens, kv_heads, bits, tiles_us);
    return f;
}

// (for either kind of cache)
size_t workspace_bytes(uint32_t pos, uint32_t tokens, uint32_t kv_heads) {
    float tiles_us;
    FlashPlan halves = tiles_plan(pos, tokens, kv_heads, tiles_us), codes = halves;
    choose_small(halves, pos, tokens, kv_heads, 16, tiles_us), choose_small(codes, pos, tokens, kv_heads, 8, tiles_us);
    return halves.bytes() > codes.bytes() ? halves.bytes() : codes.bytes();
}

// The checks both prefill paths share.
int check_prefill(int bits, const uint16_t *q, const void *kdata, const void *vdata, const uint16_t *ks,
                  const uint16_t *kz, const uint16_t *vs, const uint16_t *vz, const float *q_and_gate, const float *out,
                  saetta_flash_params p, const void *workspace, const char *what) {
    SAETTA_REQUIRE(bits == 16 || bits == 8 || bits == 4, SAETTA_E_BITS, "%s: bits %d", what, bits);
    SAETTA_REQUIRE(p.kv_heads > 0 && p.heads == p.kv_heads * SAETTA_GQA_GROUP, SAETTA_E_SHAPE,
                   "%s needs 8 q heads per kv head (heads %u, kv heads %u)", what, p.heads, p.kv_heads);
    SAETTA_REQUIRE(q && kdata && vdata && q_and_gate && out, SAETTA_E_NULL, "%s: null buffer", what);
    SAETTA_REQUIRE(bits == 16 || (ks && kz && vs && vz), SAETTA_E_NULL, "%s: null scales or biases", what);
    SAETTA_REQUIRE(aligned(q, 16) && aligned(kdata, 16) && aligned(vdata, 16) && aligned(q_and_gate, 16) &&
                       aligned(out, 16) && aligned(workspace, 16),
                   SAETTA_E_ALIGN, "%s: buffers must be 16-byte aligned", what);
    const uint64_t rows = uint64_t(p.pos) + p.tokens;  // the cache holds the chunk's rows too
    SAETTA_REQUIRE(rows * p.kv_heads * 512 < (uint64_t(1) << 31), SAETTA_E_SHAPE, "%s: pos + tokens %llu out of range",
                   what, (unsigned long long)rows);
    return SAETTA_OK;
}

// The caller's workspace if it gave one of at least `need` bytes, else the library's own for this device
// and stream, grown to the first of `wants` bytes (in falling order) that can be had; `have`: the bytes of either.  The
// library's own is held under the lock until the launches that use it
// are queued (the caller keeps `owned_lock` until then): a second host thread on the same stream that has
// to grow it waits for them (hipStreamSynchronize) before it frees.
int acquire_workspace(hipStream_t stream, void *&workspace, size_t &have, size_t need, std::initializer_list<size_t> wants,
                      std::unique_lock<std::mutex> &owned_lock, const char *what, const char *sizer) {
    if (workspace) {
        SAETTA_REQUIRE(have >= need, SAETTA_E_SCRATCH, "%s: workspace of %zu bytes, %zu needed", what, have, need);
        return SAETTA_OK;
    }
    const size_t want = *wants.begin();
    // No workspace given: use (and grow) the library's own for this stream.  This may allocate, which a
    // stream under capture cannot do; and a plan outlives the buffer, which a later call may grow.
    SAETTA_REQUIRE(!recording(), SAETTA_E_SCRATCH, "%s: a recorded call needs a workspace of the caller's (%zu bytes, %s)", what, want, sizer);
    hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &capturing) != hipSuccess) (void)hipGetLastError();
    SAETTA_REQUIRE(capturing == hipStreamCaptureStatusNone, SAETTA_E_SCRATCH,
                   "%s: a stream under capture needs a workspace of the caller's (%zu bytes, %s)", what, want, sizer);
    int dev = 0;
    if (hipError_t e = hipGetDevice(&dev)) return fail(int(e), "%s: %s", what, hipGetErrorString(e));
    SAETTA_REQUIRE(dev >= 0 && dev < OWNED_DEVICES, SAETTA_E_DEVICE, "%s: device index %d (up to %d)", what, dev, OWNED_DEVICES - 1);
    owned_lock.lock();
    OwnedWorkspace &w = g_owned[std::make_pair(dev, stream)];
    hipError_t e = hipSuccess;
    auto alloc = [&](size_t bytes) -> void * {
        void *at = nullptr;
        if ((e = hipMalloc(&at, bytes)) == hipSuccess) return at;
        (void)hipGetLastError();  // (or the launches' status would be this)
        return nullptr;
    };
    auto release = [&](void *at) {
        (void)hipStreamSynchronize(stream);
        (void)hipFree(at);
    };
    if (!w.take(wants, alloc, release)) return fail(int(e), "%s: workspace of %zu bytes: %s", what, *(wants.end() - 1), hipGetErrorString(e));
    workspace = w.ptr, have = w.bytes;
    return SAETTA_OK;
}

// The images of rows 0 .. rows - 1 of the cache, at the start of the workspace.
uint32_t launch_prepare(hipStream_t stream, int bits, const void *kdata, const void *vdata, const uint16_t *ks,
                        const uint16_t *kz, const uint16_t *vs, const uint16_t *vz, void *workspace, uint32_t kv_heads,
                        uint64_t rows, uint32_t *tiles_taken = nullptr) {
    const uint32_t nblocks = uint32_t((rows + BK - 1) / BK);
    PrepareArgs pa{kdata, vdata, ks, kz, vs, vz, static_cast<unsigned char *>(workspace), kv_heads, nblocks,
                   uint32_t(rows), tiles_taken};
    const dim3 pgrid(nblocks, kv_heads);
    if (bits == 8) {
        launch(prefill_prepare_kernel<8>, pgrid, PREP_THREADS, 0, stream, pa);
    } else if (bits == 4) {
        launch(prefill_prepare_kernel<4>, pgrid, PREP_THREADS, 0, stream, pa);
    } else {
        launch(prefill_prepare_kernel<16>, pgrid, PREP_THREADS, 0, stream, pa);
    }
    return nblocks;
}

void launch_merge(hipStream_t stream, const PrefillArgs &a, uint32_t nparts) {
    const dim3 grid(a.tokens, a.kv_heads);
    if (nparts > 8) launch(prefill_merge_kernel<MERGE_TEAMS>, grid, MERGE_THREADS * MERGE_TEAMS, 0, stream, a);
    else launch(prefill_merge_kernel<1>, grid, MERGE_THREADS, 0, stream, a);
}

// The row groups' launch; with part_blocks, their keys in parts that lie at the start of the workspace, and the merge.
int launch_small(hipStream_t stream, int bits, const uint16_t *q, const void *kdata, const void *vdata, const uint16_t *ks,
                 const uint16_t *kz, const uint16_t *vs, const uint16_t *vz, const float *q_and_gate, float *out,
                 const saetta_flash_params &p, uint32_t part_blocks, void *workspace, const char *what) {
    SmallArgs a{q, static_cast<const unsigned char *>(kdata), static_cast<const unsigned char *>(vdata), ks, kz, vs, vz, q_and_gate, out, p.heads, p.kv_heads, p.pos, p.tokens, p.scale, 0, 0, nullptr, nullptr};
    auto kernels = [&](auto split, dim3 grid, uint32_t blocks) {  // blocks: the most of a workgroup
        constexpr bool SPLIT = decltype(split)::value;
        auto variant = [&](auto rounds) {
            constexpr int ROUNDS = decltype(rounds)::value;
            constexpr bool SHARED = ROUNDS != OWN_BLOCKS;
            if (bits == 8) {
                if constexpr (ROUNDS != SHARED_ROUNDS) launch(prefill_small_kernel<8, SPLIT, ROUNDS>, grid, SMALL_THREADS, SmallLds<8, SHARED>::BYTES, stream, a);
            } else if (bits == 4) {
                launch(prefill_small_kernel<4, SPLIT, ROUNDS>, grid, SMALL_THREADS, SmallLds<4, SHARED>::BYTES, stream, a);
            } else {
                launch(prefill_small_kernel<16, SPLIT, ROUNDS>, grid, SMALL_THREADS, SmallLds<16, SHARED>::BYTES, stream, a);
            }
        };
        if (blocks <= SMALL_WAVES) return variant(std::integral_constant<int, ONE_ROUND>{});
        const bool shared = SPLIT ? blocks <= (bits == 16 ? SHARED_PART_HALF : SHARED_PART_4) : p.pos + p.tokens / 2 <= (bits == 16 ? SHARED_KEYS_HALF : SHARED_KEYS_4);
        if (shared && bits != 8) return variant(std::integral_constant<int, SHARED_ROUNDS>{});
        variant(std::integral_constant<int, OWN_BLOCKS>{});
    };
    const uint32_t groups = (p.tokens + 3) / 4;
    if (!part_blocks) {
        kernels(std::false_type{}, dim3(groups, p.kv_heads), (p.pos + p.tokens + BK - 1) / BK);
        return launch_status(what);
    }
    a.part_blocks = part_blocks, a.nparts = parts_of(p.pos, p.tokens, part_blocks);
    a.part_o = static_cast<float *>(workspace);
    a.part_ml = a.part_o + size_t(a.nparts) * ((p.tokens + TQ - 1) / TQ) * p.kv_heads * (PART_O_BYTES / 4);
    kernels(std::true_type{}, dim3((a.nparts * p.kv_heads * groups + 7) / 8 * 8), part_blocks);
    PrefillArgs m{q, nullptr, q_and_gate, out, p.heads, p.kv_heads, p.pos, p.tokens, p.scale, 0, nullptr, part_blocks, a.part_o, a.part_ml};
    launch_merge(stream, m, a.nparts);
    return launch_status(what);
}

// The tiles' launches in a workspace of `have` bytes, plan.plain at least.
int launch_flash(hipStream_t stream, int bits, const uint16_t *q, const void *kdata, const void *vdata, const uint16_t *ks,
                 const uint16_t *kz, const uint16_t *vs, const uint16_t *vz, const float *q_and_gate, float *out,
                 const saetta_flash_params &p, void *workspace, size_t have, bool exact, const FlashPlan &plan, const char *what) {
    const uint64_t rows = uint64_t(p.pos) + p.tokens;
    unsigned char *ws = static_cast<unsigned char *>(workspace);
    uint32_t *tiles_taken = reinterpret_cast<uint32_t *>(ws + images_bytes(p.pos, p.tokens, p.kv_heads));
    const uint32_t nblocks = launch_prepare(stream, bits, kdata, vdata, ks, kz, vs, vz, workspace, p.kv_heads, rows, tiles_taken);
    const uint32_t ntiles = (p.tokens + TQ - 1) / TQ;
    PrefillArgs a{q, ws, q_and_gate, out, p.heads, p.kv_heads, p.pos, p.tokens, p.scale, nblocks, tiles_taken, 0, nullptr, nullptr};
    // one workgroup per CU at most: a workgroup's LDS ring fills a CU, and further tiles are taken in the kernel
    const bool wide = plan.takes_wide(have);
    if (wide || plan.takes_narrow(have)) {
        const TileParts &parts = wide ? plan.wide : plan.narrow;
        a.part_blocks = parts.blocks;
        a.part_o = reinterpret_cast<float *>(ws + plan.plain);
        a.part_ml = reinterpret_cast<float *>(ws + plan.plain + size_t(parts.n) * ntiles * p.kv_heads * PART_O_BYTES);
        const uint32_t total = prefill_items(p.pos, p.tokens, parts.blocks, wide ? WIDE_TQ : TQ) * p.kv_heads;
        auto *kernel = wide ? (exact ? attention_prefill_kernel<true, true, true> : attention_prefill_kernel<true, false, true>)
                            : (exact ? attention_prefill_kernel<true, true, false> : attention_prefill_kernel<true, false, false>);
        launch(kernel, dim3(total < plan.cus ? total : plan.cus), THREADS, LDS_BYTES, stream, a);
        launch_merge(stream, a, parts.n);
    } else {
        const uint32_t total = ntiles * p.kv_heads;
        launch(exact ? attention_prefill_kernel<false, true, false> : attention_prefill_kernel<false, false, false>, dim3(total < plan.cus ? total : plan.cus), THREADS, LDS_BYTES, stream, a);
    }
    return launch_status(what);
}

// The chunk in a workspace of `have` bytes (none: 0, for the row groups without parts only; else at least plan.plain): the plan's
// layout as far as there is room for its parts.
int launch_chunk(hipStream_t stream, int bits, const uint16_t *q, const void *kdata, const void *vdata, const uint16_t *ks,
                 const uint16_t *kz, const uint16_t *vs, const uint16_t *vz, const float *q_and_gate, float *out,
                 const saetta_flash_params &p, void *workspace, size_t have, bool exact, const FlashPlan &plan, const char *what) {
    const bool small_parts = plan.small_part_blocks && have >= plan.small_parts;
    if (small_parts || plan.small) {
        return launch_small(stream, bits, q, kdata, vdata, ks, kz, vs, vz, q_and_gate, out, p, small_parts ? plan.small_part_blocks : 0, workspace, what);
    }
    return launch_flash(stream, bits, q, kdata, vdata, ks, kz, vs, vz, q_and_gate, out, p, workspace, have, exact, plan, what);
}

int run_prefill(hipStream_t stream, int bits, const uint16_t *q, const void *kdata, const void *vdata,
                const uint16_t *ks, const uint16_t *kz, const uint16_t *vs, const uint16_t *vz,
                const float *q_and_gate, float *out, saetta_flash_params p, void *workspace, size_t workspace_size,
                const char *what) {
    if (int rc = check_prefill(bits, q, kdata, vdata, ks, kz, vs, vz, q_and_gate, out, p, workspace, what)) return rc;
    if (int rc = ensure_device()) return rc;
    if (p.tokens == 0) return SAETTA_OK;
    const FlashPlan plan = flash_plan(p.pos, p.tokens, p.kv_heads, bits);
    std::unique_lock<std::mutex> owned_lock(g_owned_mutex, std::defer_lock);
    // (a workspace that is given has to do for the images, whatever the chunk: which launches serve it is no caller's business.
    // One of the library's is taken where the chunk has a use for one, so that it runs as in one of the caller's; where there
    // is none to be had, it is one of fewer parts, or of the images alone, and a chunk that can do without does.)
    size_t have = workspace ? workspace_size : 0;
    auto acquire = [&](std::initializer_list<size_t> wants) {
        return acquire_workspace(stream, workspace, have, plan.plain, wants, owned_lock, what, "saetta_prefill_workspace_bytes");
    };
    if (workspace || !plan.small) {
        if (int rc = acquire({plan.bytes(), plan.plain + plan.narrow.bytes, plan.plain})) return rc;
    } else if (plan.small_parts > 0) {
        (void)acquire({plan.small_parts});
    }
    return launch_chunk(stream, bits, q, kdata, vdata, ks, kz, vs, vz, q_and_gate, out, p, workspace, have, false, plan, what);
}

// ---- the same chunk as matrix products over blocks of 1024 keys ---------------------------------
// (reference: AttGemm, src/attention_gemm.rs:95-364, its default variant: prefill_ag_scores_t,
// prefill_ag_pv_t and prefill_ag_final of kernels/attention_gemm.metal.)  The reference's other route to
// the same output: the keys are walked in blocks of 1024; for a block, one launch writes the
// probabilities of every query row against the block's keys to a scratch, relative to the maximum of
// each tile of keys, with the tile's maximum and sum beside them, and a second launch folds the block
// into the running (m, l, O) of every row: O = alpha O + sum over tiles of e^(t - m) (P_tile V_tile).
// The scratch is for one slice of the chunk's tokens; the slices run one after the other.
//
// A whole call (stages 0) does NOT take these passes: what they compute is what attention_prefill_kernel computes, and it
// needs no trip of the probabilities through memory (2048 tokens at 118784, half cache: 5.98 ms by the passes, scores 2.7
// + pv 3.2, against 3.6 ms; 64 to 4096 tokens at 0 to 130000: 1.6 to 4 times).  The passes run where a caller asks
// for them by number (stages 1 to 3), to see what the scores and the second product take by themselves, and to check the
// flash kernel by: with stages 3 the sums and their state are in the scratch (GemmArgs' o, m, l, in that order behind the
// tiles' sums), and AttGemm.passes_output of the Python mirror makes the outputs of them.
//
// Here the pair of launches takes a span of AG_SPAN blocks (the scratch holds that many blocks'
// probabilities: q and the output sums then go through memory once per span, and there are as many times
// fewer launches).  A tile is 32 keys (one key image), a row group is 4 tokens x 8 heads as above, and a
// workgroup is 4 waves: a row group each in pv (a 16-token tile), two each in scores.  Both kernels take the
// image parts through LDS (the parts of the tiles ahead are fetched into registers while the current one
// is used; one barrier a tile) and run
// the same transposed products as the flash kernel, so a lane owns a query row in both:
//   scores   S^T = K Q^T (Q^T in registers), mask, tile maximum and sum per row, P = 2^(s - t) as f16,
//            stored as the P^T operands of the second product (the accumulator's registers 8 sp .. 8 sp + 7
//            are the operand of k-step sp: 1 KB per wave and k-step, read back as it was written);
//   pv       m' = max(m, max_t t), O^T = alpha O^T + sum_t V^T_t (f_t P^T_t) with f_t = 2^(t - m') rounded
//            to f16 (the row sum takes the same rounded f_t).  O, m and l stay in the scratch.
constexpr int AG_KEYS = SAETTA_AG_KEYS;
constexpr int AG_TILES = AG_KEYS / BK;
constexpr int AG_SPAN = 8;                // blocks that one pair of launches takes
constexpr int AG_SPAN_TILES = AG_SPAN * AG_TILES;
constexpr int AG_WAVES = 4;
constexpr int AG_THREADS = 64 * AG_WAVES;
constexpr int AG_TOKENS = 4 * AG_WAVES;   // tokens of a workgroup
constexpr int AG_WGS = 512;               // scores: workgroups a launch should have at least (two to a CU)
constexpr int AG_RG = 2;                  // scores: row groups per wave, which share every fragment of keys it reads
constexpr int AG_P_TILE_BYTES = BK * 32 * 2;  // the P^T operands of one row group and tile of keys

struct GemmArgs {
    const uint16_t *q;
    const unsigned char *images;
    unsigned char *p;    // f16 [kv head][token tile][tile of keys][row group of the token tile][2 k-steps][64 lanes][8]
    float *tmax, *tsum;  // [kv head][token tile][tile of keys][row group of the token tile][32 rows], log2 domain
    float *o;            // [kv head][row group][8 dim tiles][4][64 lanes][4]: the accumulators as they are
    float *m, *l;        // [kv head][row group][32 rows]
    uint32_t heads, kv_heads, pos, tokens;  // of the slice
    float c;             // scale * log2(e)
    uint32_t nblocks;    // images per kv head
    uint32_t row_groups; // per kv head in the scratch
    uint32_t g0;         // the first key of the span of blocks the launch takes
    uint32_t split;      // scores: workgroups that share a span's tiles for one token tile (a power of two)
};

// Key of the last token of a token tile of `span` tokens at tok0, and how many of the tiles of the launch's span
// of blocks hold keys that some token of the tile can see.
__device__ __forceinline__ uint32_t ag_last_key(const GemmArgs &a, uint32_t tok0, uint32_t span = AG_TOKENS) {
    const uint32_t end = tok0 + span < a.tokens ? tok0 + span : a.tokens;
    return a.pos + end - 1;
}
__device__ __forceinline__ uint32_t ag_tiles(const GemmArgs &a, uint32_t tok0, uint32_t span = AG_TOKENS) {
    const uint32_t last_key = ag_last_key(a, tok0, span);
    if (last_key < a.g0) return 0;
    const uint32_t n = (last_key - a.g0) / BK + 1;
    return n < uint32_t(AG_SPAN_TILES) ? n : uint32_t(AG_SPAN_TILES);
}

__global__ __launch_bounds__(AG_THREADS, 2) void attention_gemm_scores_kernel(GemmArgs a) {
    __shared__ __attribute__((aligned(1024))) unsigned char k_lds[3][PART_BYTES];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, col = lane & 31, hf = lane >> 5;
    // a workgroup takes AG_RG token tiles of the pv kernel: a wave AG_RG row groups in a row (8 tokens)
    const uint32_t tok0 = blockIdx.y * (AG_TOKENS * AG_RG), kv = blockIdx.z;
    const uint32_t need = ag_tiles(a, tok0, AG_TOKENS * AG_RG);
    const uint32_t per = AG_SPAN_TILES / a.split;
    const uint32_t first = blockIdx.x * per;
    if (first >= need) return;  // (the whole workgroup)
    const uint32_t count = need - first < per ? need - first : per;
    const uint32_t rg0 = (blockIdx.y * AG_WAVES + wave) * AG_RG;                    // the wave's first row group
    const uint32_t wtok0 = tok0 + 4 * AG_RG * wave, head = kv * SAETTA_GQA_GROUP + (col & 7);  // and its first token

    // A tile's K part goes global -> registers (two register sets, four and three tiles ahead) -> LDS (three
    // buffers, two and one tile ahead) -> MFMA operands.  One barrier a tile.
    const unsigned char *img = a.images + (size_t(kv) * a.nblocks + a.g0 / BK + first) * IMG_BYTES;
    u32x4 pre[2][4];
    // (Fetches and LDS writes past the last tile are made all the same, of the last tile again and into a
    // buffer nobody reads any more: with no branch around a load or a store the compiler knows how many are in
    // flight at each wait, and waits for the oldest only.)
    auto fetch = [&](u32x4 *set, uint32_t t) {
        const u32x4 *src = reinterpret_cast<const u32x4 *>(img + size_t(t < count ? t : count - 1) * IMG_BYTES);
#pragma unroll
        for (int i = 0; i < 4; i++) set[i] = src[tid + AG_THREADS * i];
    };
    auto put = [&](const u32x4 *set, uint32_t t) {
        u32x4 *dst = reinterpret_cast<u32x4 *>(k_lds[t % 3]);
#pragma unroll
        for (int i = 0; i < 4; i++) dst[tid + AG_THREADS * i] = set[i];
    };
    fetch(pre[0], 0);
    fetch(pre[1], 1);

    // Q^T operands: lane (col, hf) holds dims 16 f + 8 hf .. + 7 of query row col
    half8 qf[AG_RG][16];
#pragma unroll
    for (int r = 0; r < AG_RG; r++) {
        const uint32_t tok = wtok0 + 4 * r + (col >> 3);
        if (tok < a.tokens) {
            const half8 *qp = reinterpret_cast<const half8 *>(a.q + (size_t(tok) * a.heads + head) * DIM) + hf;
#pragma unroll
            for (int f = 0; f < 16; f++) qf[r][f] = qp[2 * f];
        } else {
#pragma unroll
            for (int f = 0; f < 16; f++) qf[r][f] = half8{0, 0, 0, 0, 0, 0, 0, 0};
        }
    }

    typedef __attribute__((address_space(3))) half8 lds_half8;
    const uint32_t lds0 = uint32_t(reinterpret_cast<uintptr_t>(&k_lds[0][0]));
    auto products = [&](uint32_t t, floatx16 (&acc)[AG_RG]) {
        // One address per tile, the fragments by the instruction's offset field (the address is hidden from
        // the loop optimizer, which otherwise keeps sixteen running addresses and two additions a read).
        uint32_t frag = lds0 + (t % 3) * PART_BYTES + lane * 16;
        asm volatile("" : "+v"(frag));
#pragma unroll
        for (int r = 0; r < AG_RG; r++)
#pragma unroll
            for (int i = 0; i < 16; i++) acc[r][i] = 0.0f;
#pragma unroll
        for (int f = 0; f < 16; f++) {
            const half8 kf = *reinterpret_cast<const lds_half8 *>(uintptr_t(frag + f * 1024));
#pragma unroll
            for (int r = 0; r < AG_RG; r++) acc[r] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf, qf[r][f], acc[r], 0, 0, 0);
        }
    };

    auto softmax = [&](floatx16 acc, uint32_t t, int r) {
        const uint32_t rg = rg0 + r;
        const uint32_t limit = a.pos + wtok0 + 4 * r + (col >> 3);  // the last key the row sees
        // slot of (row group, tile) in the scratch: the four row groups of a token tile side by side, tile after
        // tile, so that what a workgroup writes at a step and over its tiles are long runs of memory
        const size_t slot0 = ((size_t(kv) * a.row_groups + rg) / AG_WAVES * AG_SPAN_TILES + first) * AG_WAVES + rg % AG_WAVES;
        // register i is key 8 (i / 4) + 4 hf + i % 4 of the tile.  Only a tile that reaches past the first
        // token of the row group has anything to mask (wave-uniform).
        const uint32_t key0 = a.g0 + (first + t) * BK;
        if (key0 + BK - 1 > a.pos + wtok0 + 4 * r) {
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const uint32_t key = key0 + 4 * hf + 8 * (i >> 2) + (i & 3);
                acc[i] = key <= limit ? acc[i] : NO_SCORE;
            }
        }
        // (v_max3 by hand: fmaxf first quiets each operand with a v_max of its own)
        float tmax;
        asm("v_max3_f32 %0, %1, %2, %3" : "=v"(tmax) : "v"(acc[0]), "v"(acc[1]), "v"(acc[2]));
#pragma unroll
        for (int i = 3; i < 15; i += 2) asm("v_max3_f32 %0, %1, %2, %3" : "=v"(tmax) : "v"(tmax), "v"(acc[i]), "v"(acc[i + 1]));
        asm("v_max_f32 %0, %1, %2" : "=v"(tmax) : "v"(tmax), "v"(acc[15]));
        tmax = across_rows<32, 64>(tmax, MaxOp{});
        // scores in the log2 domain: s = acc * c, the tile's maximum t = tmax * c (c > 0).  A masked score is
        // NO_SCORE * c - t: far below any exponent, 0.  With the whole tile masked t would be NO_SCORE * c itself
        // and the difference the product's rounding error: 0 is subtracted then, and every probability is 0.
        const float t_log2 = tmax * a.c;
        const bool none = tmax <= 0.5f * NO_SCORE;
        const float t_sub = none ? 0.0f : t_log2;
        half2_ ph[8];
        float sum = 0.0f;
#pragma unroll
        for (int i = 0; i < 16; i += 2) {
            const float2_ e = {__builtin_amdgcn_exp2f(fmaf(acc[i], a.c, -t_sub)), __builtin_amdgcn_exp2f(fmaf(acc[i + 1], a.c, -t_sub))};
            ph[i / 2] = __builtin_convertvector(e, half2_);
            // the sum of what the second product multiplies: the rounded halves, added in f32
            sum = __builtin_amdgcn_fdot2(ph[i / 2], half2_{(_Float16)1.0f, (_Float16)1.0f}, sum, false);
        }
        sum = across_rows<32, 64>(sum, SumOp{});
        const half8 p0 = {ph[0][0], ph[0][1], ph[1][0], ph[1][1], ph[2][0], ph[2][1], ph[3][0], ph[3][1]};
        const half8 p1 = {ph[4][0], ph[4][1], ph[5][0], ph[5][1], ph[6][0], ph[6][1], ph[7][0], ph[7][1]};
        const float tmax_out = none ? NO_SCORE : t_log2;
        const size_t slot = slot0 + size_t(t) * AG_WAVES;
        unsigned char *pt = a.p + slot * AG_P_TILE_BYTES + lane * 16;
        *reinterpret_cast<half8 *>(pt) = p0;
        *reinterpret_cast<half8 *>(pt + 1024) = p1;
        // (both lanes of a row hold the same two values: one stores the maximum, the other the sum)
        float *stat = (hf ? a.tsum : a.tmax) + slot * 32 + col;
        *stat = hf ? sum : tmax_out;
    };

    put(pre[0], 0);
    fetch(pre[0], 2);
    put(pre[1], 1);
    fetch(pre[1], 3);
    __syncthreads();
    // iteration t: behind its barrier tile t is in LDS (written two iterations ago) and every wave is done with
    // tile t - 1, whose buffer takes tile t + 2 from the register set, which is then sent for tile t + 4.
    auto step = [&](u32x4 *set, uint32_t t) {
        if (t) __syncthreads();
        put(set, t + 2);
        fetch(set, t + 4);
        floatx16 acc[AG_RG];
        products(t, acc);
#pragma unroll
        for (int r = 0; r < AG_RG; r++) softmax(acc[r], t, r);
    };
    // (The first pair stands in front of the loop: the loads and stores in flight where the loop is entered
    // are then the ones in flight where it repeats, and the waits inside it are exact.)
    uint32_t t = 0;
    if (count >= 2) {
        step(pre[0], 0);
        step(pre[1], 1);
        for (t = 2; t + 1 < count; t += 2) {
            step(pre[0], t);
            step(pre[1], t + 1);
        }
    }
    if (t < count) step(pre[0], t);
}

__global__ __launch_bounds__(AG_THREADS, 2) void attention_gemm_pv_kernel(GemmArgs a) {
    __shared__ __attribute__((aligned(1024))) unsigned char v_lds[2][PART_BYTES];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, col = lane & 31, hf = lane >> 5;
    const uint32_t tok0 = blockIdx.y * AG_TOKENS, kv = blockIdx.z;
    const uint32_t need = ag_tiles(a, tok0);
    if (need == 0) return;  // nothing of this span (the sums stand as an earlier one left them)
    const uint32_t rg = blockIdx.y * AG_WAVES + wave;
    const size_t rows = size_t(kv) * a.row_groups + rg;
    const size_t state = rows * 32 + col;
    const bool first_block = a.g0 == 0;

    // slot of (row group, tile): as the scores kernel wrote them
    const size_t slot0 = rows / AG_WAVES * AG_SPAN_TILES * AG_WAVES + wave;
    const float *tm = a.tmax + slot0 * 32 + col, *ts = a.tsum + slot0 * 32 + col;
    // (all of the block's tile maxima requested at once: a loop over `need` waits for each load in turn)
    float mb = NO_SCORE;
    for (uint32_t c = 0; c < need; c += 64) {  // (64 at a time: so many registers are free here)
        float tmaxes[64];
#pragma unroll
        for (int t = 0; t < 64; t++) tmaxes[t] = tm[(c + t < need ? c + t : need - 1) * AG_WAVES * 32];
#pragma unroll
        for (int t = 0; t < 64; t++) mb = fmaxf(mb, tmaxes[t]);
    }
    // (every row sees key 0, so m is a score from the first block on)
    const float m_old = first_block ? NO_SCORE : a.m[state], l_old = first_block ? 0.0f : a.l[state];
    const float m_new = fmaxf(m_old, mb);
    const float alpha = first_block ? 0.0f : __builtin_amdgcn_exp2f(m_old - m_new);

    floatx16 acc[8];
    float *op = a.o + rows * 8 * 1024 + lane * 4;
    if (first_block) {
#pragma unroll
        for (int mt = 0; mt < 8; mt++)
#pragma unroll
            for (int i = 0; i < 16; i++) acc[mt][i] = 0.0f;
    } else {
#pragma unroll
        for (int mt = 0; mt < 8; mt++)
#pragma unroll
            for (int q4 = 0; q4 < 4; q4++) {
                const floatx4 x = *reinterpret_cast<const floatx4 *>(op + (mt * 4 + q4) * 256);
#pragma unroll
                for (int e = 0; e < 4; e++) acc[mt][4 * q4 + e] = x[e] * alpha;
            }
    }

    // the V^T part of an image
    const unsigned char *img = a.images + (size_t(kv) * a.nblocks + a.g0 / BK) * IMG_BYTES + PART_BYTES;
    // a tile's operands are fetched into registers two tiles ahead (two register sets, the loop in pairs)
    struct Ahead {
        u32x4 v[4];
        half8 p0, p1;
        float tm, ts;
    } pre[2];
    const unsigned char *pp = a.p + slot0 * AG_P_TILE_BYTES + lane * 16;
    auto fetch = [&](Ahead &set, uint32_t t) {  // (past the last tile: the last tile again, never used)
        t = t < need ? t : need - 1;
        const u32x4 *src = reinterpret_cast<const u32x4 *>(img + size_t(t) * IMG_BYTES);
#pragma unroll
        for (int i = 0; i < 4; i++) set.v[i] = src[tid + AG_THREADS * i];
        set.p0 = *reinterpret_cast<const half8 *>(pp + size_t(t) * AG_WAVES * AG_P_TILE_BYTES);
        set.p1 = *reinterpret_cast<const half8 *>(pp + size_t(t) * AG_WAVES * AG_P_TILE_BYTES + 1024);
        set.tm = tm[t * AG_WAVES * 32], set.ts = ts[t * AG_WAVES * 32];
    };
    fetch(pre[0], 0);
    fetch(pre[1], 1);
    float lsum = 0.0f;
    auto tile = [&](Ahead &set, uint32_t t) {
        unsigned char *buf = v_lds[t & 1];
#pragma unroll
        for (int i = 0; i < 4; i++) reinterpret_cast<u32x4 *>(buf)[tid + AG_THREADS * i] = set.v[i];
        __syncthreads();
        half8 pc0 = set.p0, pc1 = set.p1;
        const float tmc = set.tm, tsc = set.ts;
        fetch(set, t + 2);
        // a tile the row sees nothing of has t = NO_SCORE: its factor is 0, like its probabilities
        const _Float16 fh = (_Float16)__builtin_amdgcn_exp2f(tmc - m_new);
        lsum += (float)fh * tsc;
        pc0 *= fh, pc1 *= fh;
#pragma unroll
        for (int mt = 0; mt < 8; mt++) {
            const half8 v0 = *reinterpret_cast<const half8 *>(buf + (2 * mt) * 1024 + lane * 16);
            const half8 v1 = *reinterpret_cast<const half8 *>(buf + (2 * mt + 1) * 1024 + lane * 16);
            acc[mt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(v0, pc0, acc[mt], 0, 0, 0);
            acc[mt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(v1, pc1, acc[mt], 0, 0, 0);
        }
    };
    uint32_t t = 0;
    if (need >= 2) {  // (the first pair in front of the loop, as in the scores kernel)
        tile(pre[0], 0);
        tile(pre[1], 1);
        for (t = 2; t + 1 < need; t += 2) {
            tile(pre[0], t);
            tile(pre[1], t + 1);
        }
    }
    if (t < need) tile(pre[0], t);
    const float l_new = alpha * l_old + lsum;

    if (hf == 0) a.m[state] = m_new, a.l[state] = l_new;
#pragma unroll
    for (int mt = 0; mt < 8; mt++)
#pragma unroll
        for (int q4 = 0; q4 < 4; q4++) {
            floatx4 x;
#pragma unroll
            for (int e = 0; e < 4; e++) x[e] = acc[mt][4 * q4 + e];
            *reinterpret_cast<floatx4 *>(op + (mt * 4 + q4) * 256) = x;
        }
}

size_t align_up(size_t n, size_t a) { return (n + a - 1) / a * a; }

// Row groups of the scratch per kv head for slices of up to `slice` tokens: whole workgroups.
size_t gemm_row_groups(uint32_t slice) {
    constexpr uint32_t SPAN = AG_TOKENS * AG_RG;  // what a scores workgroup covers
    return size_t((slice + SPAN - 1) / SPAN) * AG_WAVES * AG_RG;
}

size_t gemm_scratch_bytes(uint32_t slice, uint32_t kv_heads) {
    const size_t groups = gemm_row_groups(slice) * kv_heads;
    return groups * (size_t(AG_SPAN_TILES) * AG_P_TILE_BYTES + 2 * size_t(AG_SPAN_TILES) * 32 * 4 + 32 * size_t(DIM) * 4 + 2 * 32 * 4);
}

uint32_t gemm_slice(uint32_t tokens, uint32_t slice_tokens) {
    return slice_tokens == 0 || slice_tokens > tokens ? tokens : slice_tokens;
}

// The images and the passes' scratch for slices of `slice` tokens: what a call cannot do with less of.  It grows with the
// key a chunk ends at and with the slice, so a workspace for a chunk does for every shorter one up to the same key.
size_t passes_workspace_bytes(uint32_t pos, uint32_t tokens, uint32_t slice, uint32_t kv_heads) {
    return align_up(plain_workspace_bytes(pos, tokens, kv_heads), 256) + gemm_scratch_bytes(slice, kv_heads);
}

// That, or the images and the parts of the flash kernel's keys: what is more.
size_t gemm_workspace_bytes(uint32_t pos, uint32_t tokens, uint32_t slice_tokens, uint32_t kv_heads) {
    const size_t passes = passes_workspace_bytes(pos, tokens, gemm_slice(tokens, slice_tokens), kv_heads);
    const size_t flash = workspace_bytes(pos, tokens, kv_heads);
    return passes > flash ? passes : flash;
}

int run_gemm(hipStream_t stream, int bits, const uint16_t *q, const void *kdata, const void *vdata, const uint16_t *ks,
             const uint16_t *kz, const uint16_t *vs, const uint16_t *vz, const float *q_and_gate, float *out,
             saetta_flash_params p, uint32_t slice_tokens, uint32_t stages, void *workspace, size_t workspace_size) {
    const char *what = "attn_gemm";
    if (int rc = check_prefill(bits, q, kdata, vdata, ks, kz, vs, vz, q_and_gate, out, p, workspace, what)) return rc;
    SAETTA_REQUIRE(stages <= 3, SAETTA_E_SHAPE, "%s: stages %u (0: all passes; 1, 2: scores only; 3: no outputs)", what, stages);
    const uint64_t rows = uint64_t(p.pos) + p.tokens;
    if (int rc = ensure_device()) return rc;
    if (p.tokens == 0) return SAETTA_OK;
    const uint32_t slice = gemm_slice(p.tokens, slice_tokens);
    // (a whole call runs in no slices: it asks for the passes' scratch of the smallest)
    const size_t need = passes_workspace_bytes(p.pos, p.tokens, stages == 0 ? 1 : slice, p.kv_heads);
    size_t have = workspace ? workspace_size : 0;
    std::unique_lock<std::mutex> owned_lock(g_owned_mutex, std::defer_lock);
    // All of the call: the flash kernel's result is the same and it is there in 0.5 to 0.6 of the time (see above).  Where
    // the workspace has no room for parts of the keys they are not split.
    if (stages == 0) {
        const FlashPlan plan = flash_plan(p.pos, p.tokens, p.kv_heads, bits);
        if (int rc = acquire_workspace(stream, workspace, have, need, {std::max(plan.bytes(), need), std::max(plan.plain + plan.narrow.bytes, need), need}, owned_lock, what, "saetta_attn_gemm_workspace_bytes")) return rc;
        return launch_chunk(stream, bits, q, kdata, vdata, ks, kz, vs, vz, q_and_gate, out, p, workspace, have, true, plan, what);
    }
    if (int rc = acquire_workspace(stream, workspace, have, need, {need}, owned_lock, what, "saetta_attn_gemm_workspace_bytes")) return rc;
    const uint32_t nblocks = launch_prepare(stream, bits, kdata, vdata, ks, kz, vs, vz, workspace, p.kv_heads, rows);

    const size_t groups = gemm_row_groups(slice) * p.kv_heads;
    unsigned char *at = static_cast<unsigned char *>(workspace) + align_up(plain_workspace_bytes(p.pos, p.tokens, p.kv_heads), 256);
    GemmArgs a{};
    a.images = static_cast<const unsigned char *>(workspace);
    a.p = at, at += groups * AG_SPAN_TILES * AG_P_TILE_BYTES;
    a.tmax = reinterpret_cast<float *>(at), at += groups * AG_SPAN_TILES * 32 * 4;
    a.tsum = reinterpret_cast<float *>(at), at += groups * AG_SPAN_TILES * 32 * 4;
    a.o = reinterpret_cast<float *>(at), at += groups * 32 * DIM * 4;
    a.m = reinterpret_cast<float *>(at), at += groups * 32 * 4;
    a.l = reinterpret_cast<float *>(at);
    a.heads = p.heads, a.kv_heads = p.kv_heads;
    a.c = p.scale * 1.4426950408889634f;
    a.nblocks = nblocks;
    a.row_groups = uint32_t(gemm_row_groups(slice));
    const size_t width = size_t(p.heads) * DIM;
    // A slice of tokens is a chunk of its own at pos + t0: its rows of q, q_and_gate and out, the whole
    // cache (src/attention_gemm.rs:162-188).
    for (uint32_t t0 = 0; t0 < p.tokens; t0 += slice) {
        a.tokens = p.tokens - t0 < slice ? p.tokens - t0 : slice;
        a.pos = p.pos + t0;
        a.q = q + t0 * width;
        const uint32_t tiles = (a.tokens + AG_TOKENS - 1) / AG_TOKENS;
        const uint64_t end = uint64_t(a.pos) + a.tokens;
        // scores: as many workgroups per token tile as make AG_WGS in all (2 for chunks of 4096 tokens, 4 for 2048)
        const uint32_t wide = (tiles + AG_RG - 1) / AG_RG;
        a.split = 2;
        while (a.split < 16 && a.split * wide * p.kv_heads < uint32_t(AG_WGS)) a.split *= 2;
        // a span of AG_SPAN blocks of AG_KEYS keys at a time: its scores, then its pv
        for (uint64_t g0 = 0; g0 < end; g0 += uint64_t(AG_SPAN) * AG_KEYS) {
            a.g0 = uint32_t(g0);
            launch(attention_gemm_scores_kernel, dim3(a.split, wide, p.kv_heads), AG_THREADS, 0, stream, a);
            if (stages == 1 || stages == 2) continue;
            launch(attention_gemm_pv_kernel, dim3(1, tiles, p.kv_heads), AG_THREADS, 0, stream, a);
        }
    }
    return launch_status(what);
}

}  // namespace

int setup_prefill() {
    if (int rc = load_kernel(reinterpret_cast<const void *>(prefill_merge_kernel<1>))) return rc;
    auto raise_small = [](auto bits_c) {
        constexpr int BITS = decltype(bits_c)::value;
        std::vector<std::pair<const void *, int>> kernels = {
            {reinterpret_cast<const void *>(prefill_small_kernel<BITS, false, OWN_BLOCKS>), SmallLds<BITS, false>::BYTES},
            {reinterpret_cast<const void *>(prefill_small_kernel<BITS, true, OWN_BLOCKS>), SmallLds<BITS, false>::BYTES},
            {reinterpret_cast<const void *>(prefill_small_kernel<BITS, false, ONE_ROUND>), SmallLds<BITS, true>::BYTES},
            {reinterpret_cast<const void *>(prefill_small_kernel<BITS, true, ONE_ROUND>), SmallLds<BITS, true>::BYTES}};
        if constexpr (BITS != 8) {
            kernels.push_back({reinterpret_cast<const void *>(prefill_small_kernel<BITS, false, SHARED_ROUNDS>), SmallLds<BITS, true>::BYTES});
            kernels.push_back({reinterpret_cast<const void *>(prefill_small_kernel<BITS, true, SHARED_ROUNDS>), SmallLds<BITS, true>::BYTES});
        }
        for (const auto &[kernel, bytes] : kernels) {
            if (int rc = int(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes))) return rc;
        }
        return 0;
    };
    if (int rc = raise_small(std::integral_constant<int, 16>{})) return rc;
    if (int rc = raise_small(std::integral_constant<int, 8>{})) return rc;
    if (int rc = raise_small(std::integral_constant<int, 4>{})) return rc;
    if (int rc = load_kernel(reinterpret_cast<const void *>(attention_gemm_scores_kernel))) return rc;
    if (int rc = load_kernel(reinterpret_cast<const void *>(attention_gemm_pv_kernel))) return rc;
    for (const void *kernel : {reinterpret_cast<const void *>(attention_prefill_kernel<true, false, false>), reinterpret_cast<const void *>(attention_prefill_kernel<true, true, false>),
                               reinterpret_cast<const void *>(attention_prefill_kernel<true, false, true>), reinterpret_cast<const void *>(attention_prefill_kernel<true, true, true>),
                               reinterpret_cast<const void *>(attention_prefill_kernel<false, false, false>), reinterpret_cast<const void *>(attention_prefill_kernel<false, true, false>)}) {
        if (int rc = int(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, LDS_BYTES))) return rc;
    }
    return 0;
}
}  // namespace saetta

using namespace saetta;

extern "C" size_t saetta_prefill_workspace_bytes(uint32_t pos, uint32_t tokens, uint32_t kv_heads) {
    return workspace_bytes(pos, tokens, kv_heads);
}

extern "C" int saetta_attn_prefill(saetta_stream_t stream, const uint16_t *q_f16, const uint16_t *keys,
                                   const uint16_t *values, const float *q_and_gate, float *out,
                                   saetta_flash_params p, void *workspace, size_t workspace_bytes) {
    return run_prefill(as_stream(stream), 16, q_f16, keys, values, nullptr, nullptr, nullptr, nullptr, q_and_gate,
                       out, p, workspace, workspace_bytes, "attn_prefill");
}

extern "C" int saetta_attn_prefill_quant(saetta_stream_t stream, int bits, const uint16_t *q_f16,
                                         saetta_quant_rows keys, saetta_quant_rows values,
                                         const float *q_and_gate, float *out, saetta_flash_params p,
                                         void *workspace, size_t workspace_bytes) {
    SAETTA_REQUIRE(bits == 8 || bits == 4, SAETTA_E_BITS, "attn_prefill_quant: bits %d (8 or 4)", bits);
    return run_prefill(as_stream(stream), bits, q_f16, keys.data, values.data, keys.scales, keys.biases,
                       values.scales, values.biases, q_and_gate, out, p, workspace, workspace_bytes,
                       "attn_prefill_quant");
}

extern "C" size_t saetta_attn_gemm_workspace_bytes(uint32_t pos, uint32_t tokens, uint32_t slice_tokens, uint32_t kv_heads) {
    return gemm_workspace_bytes(pos, tokens, slice_tokens, kv_heads);
}

extern "C" int saetta_attn_gemm(saetta_stream_t stream, int bits, const uint16_t *q_f16, saetta_quant_rows keys,
                                saetta_quant_rows values, const float *q_and_gate, float *out, saetta_flash_params p,
                                uint32_t slice_tokens, uint32_t stages, void *workspace, size_t workspace_bytes) {
    return run_gemm(as_stream(stream), bits, q_f16, keys.data, values.data, keys.scales, keys.biases, values.scales,
                    values.biases, q_and_gate, out, p, slice_tokens, stages, workspace, workspace_bytes);
}
