// Split-K decode / verify attention over the KV cache for gfx950 (MI355X).
//
// What it computes (reference: DecodeAttention::record{,_quant}
// src/attention.rs:73-135, AttentionRows::record{,_quant} src/rows.rs:369-493;
// CPU definition src/cpu/attention.rs:141-181): for each of m query rows and
// each of the 16 q heads,
//     out = softmax(q K^T * scale) V * sigmoid(gate)
// over the first len_r cached tokens, 8 q heads sharing one kv head, head dim
// 256.  The cache is f16 or 8/4-bit group-affine codes (groups of 64 dims,
// f16 scale and bias, x = s*q + z; layout in kv_quant.hip).
//
// Shape of the work: 2 kv heads only, so all parallelism comes from splitting
// the context.  The context actually in use (read from TokenParams in device
// memory when the kernel runs) is cut into 16-token blocks and the blocks are
// dealt evenly to the `nsplits` workgroups of each kv head, so every
// workgroup streams the same number of bytes whatever the position is.  A
// workgroup walks its range in iterations of 64 to 192 tokens, keeps an
// online softmax per query row, and writes one unnormalised partial (o, m, l)
// per (row, q head); a second kernel merges the partials and applies the gate.
//
// Inside an iteration the two contractions run on the matrix cores
// (v_mfma_f32_16x16x32_f16), because at 15-28 FLOP per cache byte a vector-ALU
// dot product cannot keep up with HBM:
//   phase A  S^T = K Q^T   wave w takes the 16-token blocks w, w+4, w+8;
//            A operand = key codes of 16 tokens, B operand = the query rows.
//   phase B  online softmax per row over the iteration's scores (in LDS).
//   phase C  O += P V      wave w takes dims 64w..64w+63, which is exactly
//            one quantization group, for all tokens of the iteration.
// Codes are never dequantized element by element.  A code byte c is placed in
// the low mantissa bits of an f16 with a zero exponent, i.e. the subnormal
// c * 2^-24, with one v_perm_b32 per two codes; the matrix cores take
// subnormal inputs.  Scale and bias of a group are applied to the 64-dim
// partial dot product (keys) or folded into the probability operand (values):
//   q.k   = sum_g  s_g * (q_g . c_g)  +  sum_g z_g * sum(q_g)
//   P V_g = (P * s_g) C_g + (P . z_g)
// and the key bias term sum_g z_g * sum(q_g) is itself one small MFMA.
// The value operand needs (token, token+1) pairs per dim while memory holds
// (dim, dim+1) pairs per token; the same v_perm_b32 that widens the bytes
// picks them from two tokens' words, so the transposition costs nothing.
// q and P are split into f16 hi + lo parts (two MFMAs into one accumulator,
// or for a single row the hi and lo parts share one 16-row tile), which keeps
// the result within ~1e-6 of an f32 evaluation.
//
// All cache reads of the register kernels are buffer loads with the cache's
// size as the bound: rows past the capacity read as 0 instead of faulting, and
// the per-lane address is one 32-bit offset plus scalar and immediate parts.
//
// Kernels (one body, attention_partial_body, behind template switches):
//   attention_partial_kernel_p   one query row, one workgroup per CU (all registers)
//   attention_partial_kernel_1   one query row over codes, two workgroups per CU (long 4-bit caches)
//   attention_partial_kernel_n   2 rows (1 tile), 3-4 rows (2 tiles), 5-6 (3 tiles), 7-8 (4 tiles)
//   attention_partial_kernel_s   one to four query rows over codes in large caches: four more waves
//                                move the codes into LDS (global_load_lds), a whole share at once
//                                with the keys requested first (longer shares: rounds in alternate
//                                halves of LDS), the waves meeting through counters in LDS
//   attention_partial_kernel_h   three to eight query rows over a half cache: loader waves, a wave per tile
//                                (decode_half_rows.hpp)
//   attention_partial_kernel_c   the same over codes: two rows and more in the caches that code_rows names
//                                (decode_code_rows.hpp)
//   attention_reduce_kernel      the merge of the splits and the gate
//   attention_token_alone_kernel a recorded token step over a small cache: store, attention and gate
// Which one runs is decided in run_attention from the launch arguments alone, so that the partial
// and the reduce stage of a step agree on the number of splits.
#include "common.hpp"
#include "kv_quant_device.hpp"
#include "lanes.hpp"
#include "prep_device.hpp"

namespace saetta {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr int DIM = SAETTA_HEAD_DIM;
constexpr int THREADS = 256;
constexpr int BLOCK = 16;                     // tokens per MFMA block
// A buffer offset past any cache (their sizes stay below 2^31): the load returns 0 and touches no
// memory.  With UNCOND, loads that an iteration does not need are issued with it instead of being
// branched around, so that the number of loads in flight at every wait is known when the kernel is
// compiled: loads return in order, and a wait whose count is not known has to wait for all of them.
// (Measured per kernel: it pays for up to four query rows, not for the larger tiles.)
constexpr int OOB = int(0x80000000u);
// s_waitcnt operand that waits for the vector memory counter only (gfx9 encoding: vmcnt in bits
// 3:0 and 15:14, the other counters at their maxima).
constexpr int vmcnt_only(int n) {
    return (n & 15) | 0x70 | 0xf00 | ((n >> 4) << 14);
}
constexpr float NO_SCORE = -1e30f;            // finite "minus infinity" of the running max

// q is multiplied by scale * log2(e) * Q_UP before the hi/lo split so that
// the lo part stays a normal f16; probabilities by P_UP for the same reason.
constexpr float Q_UP = 16.0f;
constexpr float P_UP = 256.0f;
// A code byte b is fed to the matrix cores as the f16 subnormal b * 2^-24.
// 4-bit codes sit in the HIGH nibble of that byte (16c * 2^-24): the adders
// align products by exponent field, so leading zero bits of a subnormal
// mantissa are lost precision, and the high nibble loses four fewer.
template <int BITS>
constexpr float code_up() {
    return BITS == 8 ? 16777216.0f : BITS == 4 ? 1048576.0f : 1.0f;
}
// Bytes of one (token, kv head) of keys or values.
template <int BITS>
constexpr int row_bytes() {
    return BITS == 16 ? 512 : BITS * 32;
}

struct PartialArgs {
    const float *q;
    const void *kdata;
    const void *vdata;
    const uint16_t *kscales, *kbiases, *vscales, *vbiases;
    float *part_o;
    float *part_ml;
    uint32_t heads, kv_heads, capacity;
    float scale;
    uint32_t rows, nsplits;
    const saetta_token_params *tp;
    uint32_t decode_len;  // 1: every row sees min(kv_len, capacity); 0: row r sees position + r + 1
    uint32_t *status;     // the device's sticky status word (pinned host memory)
};
// The same with the step before the scores taken in.
struct TokenArgs {
    PartialArgs a;        // nsplits: the context's workgroups and one
    PrepArgs prep;
    uint32_t new_heads;   // q heads of a row that a workgroup of the new rows takes (register kernels)
};

__device__ __forceinline__ uint32_t perm(uint32_t hi, uint32_t lo, uint32_t sel) {
    return __builtin_amdgcn_perm(hi, lo, sel);
}

__device__ __forceinline__ half8 as_half8(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
    u32x4 v = {a, b, c, d};
    return __builtin_bit_cast(half8, v);
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void *p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, int(bytes), 0x00020000);
}

// ---- key codes: 16 dims of one token per lane and group ----------------------
template <int BITS>
struct KeyRegs {
    uint32_t w[BITS == 16 ? 8 : BITS / 2];  // 32 B (f16), 16 B (8-bit), 8 B (4-bit)
};

// Lane (t, j) reads dims 64g + 16j .. +15 of its token: `voff` is the lane's
// byte offset of (token, kv head, j), `soff` the scalar part (block), g is an immediate.
template <int BITS>
__device__ __forceinline__ KeyRegs<BITS> load_key(__amdgpu_buffer_rsrc_t rsrc, int voff, int soff, int g) {
    KeyRegs<BITS> r;
    if constexpr (BITS == 8) {
        u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(rsrc, voff + g * 64, soff, 0);
        r.w[0] = v.x, r.w[1] = v.y, r.w[2] = v.z, r.w[3] = v.w;
    } else if constexpr (BITS == 4) {
        u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(rsrc, voff + g * 32, soff, 0);
        r.w[0] = v.x, r.w[1] = v.y;
    } else {
        u32x4 v0 = __builtin_amdgcn_raw_buffer_load_b128(rsrc, voff + g * 128, soff, 0);
        u32x4 v1 = __builtin_amdgcn_raw_buffer_load_b128(rsrc, voff + g * 128 + 16, soff, 0);
        r.w[0] = v0.x, r.w[1] = v0.y, r.w[2] = v0.z, r.w[3] = v0.w;
        r.w[4] = v1.x, r.w[5] = v1.y, r.w[6] = v1.z, r.w[7] = v1.w;
    }
    return r;
}

// Bytes of the lane's 16 dims inside a group.
template <int BITS>
constexpr int key_piece() {
    return BITS == 16 ? 32 : BITS * 2;
}

// The A operand of k-step `ab` (0: the lane's first 8 dims, 1: the next 8).
template <int BITS>
__device__ __forceinline__ half8 key_operand(const KeyRegs<BITS> &r, int ab) {
    if constexpr (BITS == 8) {
        const uint32_t w0 = r.w[2 * ab], w1 = r.w[2 * ab + 1];
        return as_half8(perm(0, w0, 0x0c010c00u), perm(0, w0, 0x0c030c02u), perm(0, w1, 0x0c010c00u),
                        perm(0, w1, 0x0c030c02u));
    } else if constexpr (BITS == 4) {
        const uint32_t w = r.w[ab];
        const uint32_t x = (w << 4) & 0xf0f0f0f0u, y = w & 0xf0f0f0f0u;
        // slots: dims 0,2 | 4,6 | 1,3 | 5,7
        return as_half8(perm(0, x, 0x0c010c00u), perm(0, x, 0x0c030c02u), perm(0, y, 0x0c010c00u),
                        perm(0, y, 0x0c030c02u));
    } else {
        return as_half8(r.w[4 * ab], r.w[4 * ab + 1], r.w[4 * ab + 2], r.w[4 * ab + 3]);
    }
}

// Which of the lane's 8 dims of a k-step sits in MFMA slot e.
template <int BITS>
__device__ __forceinline__ constexpr int key_slot_dim(int e) {
    if (BITS == 4) {
        constexpr int order[8] = {0, 2, 4, 6, 1, 3, 5, 7};
        return order[e];
    }
    return e;
}

// ---- value codes: one dword per token, 8 tokens per lane and k-step -----------
// 8-bit: the dword holds dims 4n..4n+3 of the wave's group; 4-bit: lanes 2i and
// 2i+1 load the same dword (8 dims) and use its low / high 16 bits; f16: two
// dwords, dims 2n, 2n+1 and 32+2n, 32+2n+1 of the wave's 64.
template <int BITS>
struct ValRegs {
    uint32_t w[BITS == 16 ? 16 : 8];
};

// Byte offset of the lane's dword inside a (token, kv head) row.
template <int BITS>
__device__ __forceinline__ int val_lane_offset(int wave, int n) {
    if constexpr (BITS == 8) return wave * 64 + n * 4;
    if constexpr (BITS == 4) return wave * 32 + (n >> 1) * 4;
    return wave * 128 + n * 4;
}

// B operand of output tile `tile` (0..3) from the 8 tokens' words of a k-step.
// Tile e covers dims 4n + e (8/4-bit) or 32*(e/2) + 2n + e%2 (f16) of the wave's 64.
template <int BITS>
__device__ __forceinline__ half8 val_operand(const ValRegs<BITS> &r, int tile, int n) {
    uint32_t o[4];
    if constexpr (BITS == 8) {
        const uint32_t sel = 0x0c000c00u | (uint32_t(4 + tile) << 16) | uint32_t(tile);
#pragma unroll
        for (int i = 0; i < 4; i++) o[i] = perm(r.w[2 * i + 1], r.w[2 * i], sel);
    } else if constexpr (BITS == 4) {
        // the byte first, by a selector of the lane's own that every word shares, then its nibble: two tiles take the same
        // byte, so four instructions make two words of operands (nine with the nibbles cut out of each token's word)
        const uint32_t byte = uint32_t(n & 1) * 2 + uint32_t(tile >> 1);
        const uint32_t sel = 0x0c040c00u + byte * 0x00010001u;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t w = perm(r.w[2 * i + 1], r.w[2 * i], sel);
            o[i] = (tile & 1 ? w : w << 4) & 0x00f000f0u;
        }
    } else {
        const int set = tile >> 1;
        const uint32_t sel = (tile & 1) ? 0x07060302u : 0x05040100u;
#pragma unroll
        for (int i = 0; i < 4; i++) o[i] = perm(r.w[set * 8 + 2 * i + 1], r.w[set * 8 + 2 * i], sel);
    }
    return as_half8(o[0], o[1], o[2], o[3]);
}

// f32 -> f16 hi part and f16 lo part with hi + lo = x to ~2^-22.  hi is x with
// the low 13 mantissa bits cleared, which an f16 holds exactly whatever way
// the conversion rounds; a conversion-based split breaks at ties when the
// compiler fuses one of the two conversions with the multiply that made x.
__device__ __forceinline__ void split_hi_lo(float x, _Float16 &hi, _Float16 &lo) {
    const float h = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, x) & 0xffffe000u);
    hi = (_Float16)h;
    lo = (_Float16)(x - h);
}

__device__ __forceinline__ float half_bits_to_float(uint32_t bits16) {
    return (float)__builtin_bit_cast(_Float16, uint16_t(bits16));
}

// The largest of four lane groups' values.  (By the instruction: fmaxf of a value that comes out of an exchange takes two more, which
// quiet what might be a signalling NaN.)
struct RawMaxOp {
    __device__ __forceinline__ float operator()(float a, float b) const {
        float r;
        asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
        return r;
    }
};

// The f16 of one group of a pair in the scales' planes, of two tokens: sel, of group_sel, names the group.
typedef _Float16 half2_ __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t group_sel(int group) { return group & 1 ? 0x07060302u : 0x05040100u; }
__device__ __forceinline__ half2_ group_halves(uint32_t w0, uint32_t w1, uint32_t sel) { return __builtin_bit_cast(half2_, perm(w1, w0, sel)); }

// One query row's probability operand of a k-step, times the value scales of a group (sv, zv: the tokens' dwords of scales and biases,
// sel: the group's).  The two lanes of a head (n and n + 8) make four of the lane group's eight tokens each (p4), both parts, and hand
// over what the other one feeds: the hi lane (n < 8) feeds hi parts and wants the other lane's of tokens 4-7, the lo lane lo parts
// and the other lane's of tokens 0-3.  A product with a scale and its lo part are fused operations that take the f16 as it is, two
// tokens' from one permute, and the exchange writes half of a row's lanes (bank masks): 40 vector instructions where shifts, conversions
// and selects made 54.
__device__ __forceinline__ half8 one_row_operand(const floatx4 &p4, float f, const u32x4 &sv, const u32x4 &zv, uint32_t sel, float &zacc) {
    const half2_ s[2] = {group_halves(sv.x, sv.y, sel), group_halves(sv.z, sv.w, sel)}, z[2] = {group_halves(zv.x, zv.y, sel), group_halves(zv.z, zv.w, sel)};
    float x[4], lo[4];
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const float p = p4[e] * f;
        zacc = fmaf(p, float(z[e >> 1][e & 1]), zacc);
        x[e] = fmaf(p, float(s[e >> 1][e & 1]), 0.0f);
        lo[e] = fmaf(p, float(s[e >> 1][e & 1]), -__builtin_bit_cast(float, __builtin_bit_cast(uint32_t, x[e]) & 0xffffe000u));
    }
    // round toward zero: exact truncation to the hi part
    int hi0 = __builtin_bit_cast(int, __builtin_amdgcn_cvt_pkrtz(x[0], x[1])), hi1 = __builtin_bit_cast(int, __builtin_amdgcn_cvt_pkrtz(x[2], x[3]));
    int lo0 = __builtin_bit_cast(int, __builtin_amdgcn_cvt_pkrtz(lo[0], lo[1])), lo1 = __builtin_bit_cast(int, __builtin_amdgcn_cvt_pkrtz(lo[2], lo[3]));
    constexpr int ROR_8 = 0x128, UPPER = 0xc, LOWER = 0x3;  // lanes 8-15 | 0-7 of a row of 16
    uint32_t o[4] = {uint32_t(__builtin_amdgcn_update_dpp(hi0, lo0, ROR_8, 0xf, UPPER, false)), uint32_t(__builtin_amdgcn_update_dpp(hi1, lo1, ROR_8, 0xf, UPPER, false)),
                     uint32_t(__builtin_amdgcn_update_dpp(lo0, hi0, ROR_8, 0xf, LOWER, false)), uint32_t(__builtin_amdgcn_update_dpp(lo1, hi1, ROR_8, 0xf, LOWER, false))};
    // (pinned: left alone, the compiler moves an operand's arithmetic down to its use, behind the wait for the values)
    asm volatile("" : "+v"(o[0]), "+v"(o[1]), "+v"(o[2]), "+v"(o[3]));
    return as_half8(o[0], o[1], o[2], o[3]);
}

// ---- the step before the scores, taken in -------------------------------------------------------
//
// A token step of a plan records attention_prep_store, the partial and the reduce stage of a layer one after the other.
// The first is a launch of 2.7 us (20 workgroups and row; 1.6 us is what any launch costs in a graph) for 20 KB of work, so
// where the three stand next to each other on the same buffers (run_attention looks while they are recorded) the partial
// stage does it:
//  * every workgroup of the context norms and rotates the query rows it needs itself, under the first loads of the cache;
//    its context are the tokens BEFORE the new ones;
//  * workgroups of their own (behind the context's) make the new keys and values, store them and the query rows, and
//    write the new tokens' own partial result (the last split), from the values just as the cache holds them.  Nobody in
//    the launch reads what another workgroup of it writes, as long as the step's buffers lie apart (token_step looks).
// The keys', values' and codes' bits are those of attention_prep_store_kernel (the same operations in the same order).
// A workgroup of the new rows takes some rows and some heads of them, and makes the keys and values of all rows up to
// those for itself.  The loader kernels have 12 waves: one workgroup does it all.  The register kernels have 4, so that a
// row's heads are dealt out two to a workgroup where CUs are free, and a row has one workgroup where the context would
// fill them all.  The total stays at one workgroup per CU: where it was 128 per kv head the context gives some up.
// Measured per layer, ten layers in a graph, against the store as a launch of its own: one row 9.9 against 11.9 us (codes,
// 300 tokens of 8192), 12.6 against 15.2 (f16, 7000 of 8192), 16.6 against 18.1 (8-bit, 32768), 33 against 35 (4-bit,
// 150000); two rows 11.7 against 13.7 (f16, 3000), 18 against 20.4 (8-bit, 32768); three 24.1 against 26; four 15.8
// against 17.2 (8-bit, 3000), 36.2 against 37.7 (60000).

// The other half wavefront's value.
__device__ __forceinline__ float half_swap(float x, bool lower) {
    uint32_t u = __builtin_bit_cast(uint32_t, x), v = u;
    swap_rows32(u, v);  // u = (lower, lower), v = (upper, upper)
    return __builtin_bit_cast(float, lower ? v : u);
}

constexpr int NEW_ROWS = 4;  // rows of a token step that takes the store in, at most
// Tokens of the context before the new ones; new tokens that row `row` sees.
__device__ __forceinline__ uint32_t tokens_before(const PartialArgs &a, uint32_t position, uint32_t kv_len) {
    return min(a.decode_len ? min(position, kv_len) : position, a.capacity);
}
__device__ __forceinline__ uint32_t tokens_new(const PartialArgs &a, uint32_t position, uint32_t kv_len, uint32_t row) {
    const uint32_t seen = min(a.decode_len ? min(kv_len, position + 1) : position + row + 1, a.capacity);
    return seen > position ? seen - position : 0;
}

// Dims 64 i + lane of a kv head's row of the cache.
template <int BITS>
__device__ __forceinline__ void cached_row(const void *data, const uint16_t *scales, const uint16_t *biases, size_t slot, uint32_t lane, float (&x)[4]) {
#pragma unroll
    for (uint32_t i = 0; i < 4; i++) {
        const uint32_t d = 64 * i + lane;
        if constexpr (BITS == 16) {
            x[i] = half_bits_to_float(static_cast<const uint16_t *>(data)[slot * DIM + d]);
        } else {
            constexpr uint32_t VPL = 32 / BITS;
            const uint32_t word = static_cast<const uint32_t *>(data)[slot * (DIM / VPL) + d / VPL];
            x[i] = fmaf(half_bits_to_float(scales[slot * 4 + i]), float((word >> (d % VPL * BITS)) & ((1u << BITS) - 1)), half_bits_to_float(biases[slot * 4 + i]));
        }
    }
}

// What a workgroup makes of the new rows: the keys and values of all rows up to its last, q heads head0 .. head0 + heads - 1 of rows
// row0 .. row0 + nrows - 1 (of up to R), in LDS and, those that are its own, in memory.  A wave takes whole heads: lane l holds dims l,
// 64 + l, 128 + l, 192 + l.
struct NewRows {
    float *keys, *values, *queries;  // [row][256] as the cache gives them; [row][head][256]
};
template <int BITS, int R>
__device__ __forceinline__ NewRows make_rows(const PartialArgs &a, const PrepArgs &p, unsigned char *lds, uint32_t waves, uint32_t row0, uint32_t nrows,
                                             uint32_t head0, uint32_t heads, uint32_t position) {
    const uint32_t tid = threadIdx.x, lane = tid & 63, kv = blockIdx.y, kvh = a.kv_heads, rows = row0 + nrows;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    float2 *rope = reinterpret_cast<float2 *>(lds);                                          // [row][32] sine, cosine
    float *keys = reinterpret_cast<float *>(lds + R * 32 * 8), *values = keys + rows * DIM;
    float *queries = values + rows * DIM;
    // items: the rows' keys, their values, then the q heads
    const uint32_t items = 2 * rows + nrows * heads;
    float next[4];
    auto request = [&](uint32_t item) {
        item = item < items ? item : items - 1;
        const uint32_t q = item - 2 * rows;
        const float *src = item < rows       ? p.k + (size_t(item) * kvh + kv) * DIM
                           : item < 2 * rows ? p.v + (size_t(item - rows) * kvh + kv) * DIM
                                             : p.q_and_gate + (size_t(row0 + q / heads) * a.heads + kv * 8 + head0 + q % heads) * 2 * DIM;
#pragma unroll
        for (int i = 0; i < 4; i++) next[i] = src[64 * i + lane];
    };
    request(wave);
    float qn[4], kn[4];
#pragma unroll
    for (int i = 0; i < 4; i++) qn[i] = p.q_norm[64 * i + lane], kn[i] = p.k_norm[64 * i + lane];
    if (tid < 32 * rows) {
        float s, c;
        rope_angle(position + (tid >> 5), rope_frequency(tid & 31, 32, p.p.log2_theta), s, c);
        rope[tid] = float2{s, c};
    }
    __syncthreads();
    for (uint32_t item = wave; item < items; item += waves) {
        const bool is_q = item >= 2 * rows, is_k = item < rows;
        const uint32_t q = item - 2 * rows, row = is_q ? row0 + q / heads : is_k ? item : item - rows;
        float x[4];
#pragma unroll
        for (int i = 0; i < 4; i++) x[i] = next[i];
        if (item + waves < items) request(item + waves);
        if (is_q || is_k) {
            float sq[4];
#pragma unroll
            for (int i = 0; i < 4; i++) sq[i] = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, square_sum(x[i]))));
            const float scale = norm_scale((sq[0] + sq[1]) + (sq[2] + sq[3]), p.p.eps);
#pragma unroll
            for (int i = 0; i < 4; i++) x[i] = __fmul_rn(x[i], __fmul_rn(scale, is_q ? qn[i] : kn[i]));
            const float2 sc = rope[row * 32 + (lane & 31)];
            const float other = half_swap(x[0], lane < 32);
            x[0] = lane < 32 ? rope_first(x[0], other, sc.x, sc.y) : rope_second(other, x[0], sc.x, sc.y);
        }
        if (is_q) {
            float *dst = p.q_out + (size_t(row) * a.heads + kv * 8 + head0 + q % heads) * DIM, *keep = queries + q * DIM;
#pragma unroll
            for (int i = 0; i < 4; i++) dst[64 * i + lane] = x[i], keep[64 * i + lane] = x[i];
            continue;
        }
        const bool mine = row >= row0 && head0 == 0;  // of the workgroups that make it, the one that stores it
        if (is_k && mine && p.k_back) {
#pragma unroll
            for (int i = 0; i < 4; i++) p.k_back[(size_t(row) * kvh + kv) * DIM + 64 * i + lane] = x[i];
        }
        const size_t slot = size_t(position + row) * kvh + kv;  // (head row of the cache)
        const bool stored = mine && position + row < a.capacity;
        float *keep = (is_k ? keys : values) + row * DIM;
        if constexpr (BITS == 16) {
            uint16_t *dst = (is_k ? p.keys_half : p.values_half) + slot * DIM;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const __half h = __float2half_rn(x[i]);
                if (stored) dst[64 * i + lane] = __half_as_ushort(h);
                keep[64 * i + lane] = __half2float(h);
            }
        } else {
            // the quantizer wants 32 / BITS neighbouring values per lane: through LDS, where the cache's values then go
            constexpr uint32_t VPL = 32 / BITS, LANES = SAETTA_QUANT_GROUP / VPL;
#pragma unroll
            for (int i = 0; i < 4; i++) keep[64 * i + lane] = x[i];
            wave_sync();
            if (lane < DIM / VPL) {
                float v[VPL];
#pragma unroll
                for (uint32_t e = 0; e < VPL; e++) v[e] = keep[lane * VPL + e];
                __half s, z;
                const uint32_t word = quantize_lane<BITS>(v, s, z);
                if (stored) {
                    const saetta_quant_rows c = is_k ? p.kq : p.vq;
                    c.data[slot * (DIM / VPL) + lane] = word;
                    if (lane % LANES == 0) c.scales[slot * 4 + lane / LANES] = __half_as_ushort(s), c.biases[slot * 4 + lane / LANES] = __half_as_ushort(z);
                }
                const float sf = __half2float(s), zf = __half2float(z);
#pragma unroll
                for (uint32_t e = 0; e < VPL; e++) keep[lane * VPL + e] = fmaf(sf, float((word >> (e * BITS)) & ((1u << BITS) - 1)), zf);
            }
        }
    }
    __syncthreads();
    return {keys, values, queries};
}

// A workgroup of the new rows (see make_rows).
template <int BITS, int R>
__device__ __forceinline__ void new_rows(const PartialArgs &a, const PrepArgs &p, unsigned char *lds, uint32_t waves, uint32_t row0, uint32_t nrows,
                                         uint32_t head0, uint32_t heads) {
    const uint32_t lane = threadIdx.x & 63, kv = blockIdx.y, kvh = a.kv_heads;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t position = a.tp->position, kv_len = a.tp->kv_len;
    const auto [keys, values, queries] = make_rows<BITS, R>(a, p, lds, waves, row0, nrows, head0, heads, position);
    // the new tokens' partial result of every (row, head): scores in units of log2(e), as the other splits'
    for (uint32_t pair = wave; pair < nrows * heads; pair += waves) {
        const uint32_t row = row0 + pair / heads, seen = tokens_new(a, position, kv_len, row);
        float q[4], score[R], m = NO_SCORE, l = 0.0f, o[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int i = 0; i < 4; i++) q[i] = queries[pair * DIM + 64 * i + lane] * (a.scale * 1.4426950408889634f);
#pragma unroll
        for (uint32_t t = 0; t < uint32_t(R); t++) {
            score[t] = NO_SCORE;
            if (t < seen) {
                float dot = 0.0f;
#pragma unroll
                for (int i = 0; i < 4; i++) dot += q[i] * keys[t * DIM + 64 * i + lane];
                score[t] = group_reduce<64>(dot, SumOp());
                m = fmaxf(m, score[t]);
            }
        }
#pragma unroll
        for (uint32_t t = 0; t < uint32_t(R); t++) {
            if (t < seen) {
                const float prob = __builtin_amdgcn_exp2f(score[t] - m);
                l += prob;
#pragma unroll
                for (int i = 0; i < 4; i++) o[i] += prob * values[t * DIM + 64 * i + lane];
            }
        }
        if constexpr (R == 1) {
            // a decode sees min(kv_len, capacity) tokens: where the record's kv_len is not position + 1 but more, rows
            // of the cache past the new one too.  No step of a model has any, so one after the other will do.
            const uint32_t end = a.decode_len ? min(kv_len, a.capacity) : 0;
            for (uint32_t t = position + 1; t < end && position < end; t++) {
                float x[4], dot = 0.0f;
                cached_row<BITS>(a.kdata, a.kscales, a.kbiases, size_t(t) * kvh + kv, lane, x);
#pragma unroll
                for (int i = 0; i < 4; i++) dot += q[i] * x[i];
                const float s = group_reduce<64>(dot, SumOp()), top = fmaxf(m, s);
                const float keep = __builtin_amdgcn_exp2f(m - top), prob = __builtin_amdgcn_exp2f(s - top);
                cached_row<BITS>(a.vdata, a.vscales, a.vbiases, size_t(t) * kvh + kv, lane, x);
                m = top, l = l * keep + prob;
#pragma unroll
                for (int i = 0; i < 4; i++) o[i] = o[i] * keep + prob * x[i];
            }
        }
        const size_t slot = (size_t(row) * a.nsplits + (a.nsplits - 1)) * a.heads + kv * 8 + head0 + pair % heads;
#pragma unroll
        for (int i = 0; i < 4; i++) a.part_o[slot * DIM + 64 * i + lane] = o[i];
        if (lane == 0) *reinterpret_cast<floatx2 *>(a.part_ml + 2 * slot) = floatx2{m, l};
    }
}

// TILES: 16-row tiles of query rows (rows * 8 heads, rounded up).  PACKED: one
// verify row; its 8 heads' hi parts are operand rows 0-7 and lo parts rows 8-15
// of a single tile.  Otherwise hi and lo are two MFMAs into one accumulator.
// ITB: blocks per iteration of a workgroup (a multiple of 4: one block per wave and round), at most (walk).
template <int BITS, int TILES, bool PACKED, int ITB>
struct Shape {
    static constexpr int IT_BLOCKS = ITB;
    static constexpr int IT_TOKENS = BLOCK * ITB;
    static constexpr int SC_STRIDE = IT_TOKENS + 4;  // floats; keeps rows on different LDS banks
    static constexpr bool QUANT = BITS != 16;
    static constexpr int S_ROWS = 16 * TILES;                  // rows of the score buffer
    static constexpr int SOFT_ROWS = PACKED ? 8 : TILES == 3 ? 64 : 16 * TILES;  // rows phase B's threads are dealt to (three tiles: a wave has none)
    static constexpr int TPR = THREADS / SOFT_ROWS;            // threads per row in phase B
    static constexpr int TPT = IT_TOKENS / TPR;                // tokens per thread in phase B
    static constexpr int PARTS = PACKED ? 1 : 2;
    // LDS map, in bytes
    static constexpr int Q_OFF = 0;
    static constexpr int Q_BYTES = TILES * PARTS * 8 * 64 * 16;  // [tile][part][step][lane] half8
    static constexpr int S_OFF = Q_OFF + Q_BYTES;
    static constexpr int S_BYTES = S_ROWS * SC_STRIDE * 4;  // [row][token] f32
    static constexpr int KS_OFF = S_OFF + S_BYTES;          // [token][4] f16
    static constexpr int KZ_OFF = KS_OFF + (QUANT ? IT_TOKENS * 8 : 0);
    static constexpr int VS_OFF = KZ_OFF + (QUANT ? IT_TOKENS * 8 : 0);  // [4][token] f16
    static constexpr int VZ_OFF = VS_OFF + (QUANT ? IT_TOKENS * 8 : 0);
    static constexpr int ALPHA_OFF = VZ_OFF + (QUANT ? IT_TOKENS * 8 : 0);  // [S_ROWS] f32
    static constexpr int QZ_OFF = ALPHA_OFF + S_ROWS * 4;                   // [tile][hi, lo][lane] half8
    static constexpr int ZSUM_OFF = QZ_OFF + TILES * 2 * 64 * 16;           // [wave][S_ROWS] f32
    static constexpr int LDS_BYTES = ZSUM_OFF + 4 * S_ROWS * 4;
    // the new rows' workgroup of attention_token_kernel_*: the angles, then keys, values and 8 query rows per row
    static constexpr int ROWS = PACKED ? 1 : 2 * TILES;
    static_assert(2 * 1024 + ROWS * 10 * 256 * 4 <= LDS_BYTES, "the new rows' workgroup fits");
};

template <int BITS, int TILES, bool PACKED, int ITB, bool UNCOND, bool PREP = false>
__device__ __forceinline__ void attention_partial_body(const PartialArgs &a, const PrepArgs *prep = nullptr, uint32_t new_heads = 8) {
    constexpr bool QUANT = BITS != 16;
    constexpr int PARTS = PACKED ? 1 : 2;
    constexpr int RB = row_bytes<BITS>();
    extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
    const int tid = int(threadIdx.x), lane = tid & 63, wave = tid >> 6;
    const int n = lane & 15, j = lane >> 4;
    const uint32_t split = blockIdx.x, kv = blockIdx.y;
    const uint32_t kvh = a.kv_heads;
    const uint32_t real_rows = a.rows * 8;  // (row, head) pairs of this kv head
    const uint32_t context_splits = PREP ? a.nsplits - 1 : a.nsplits;
    if constexpr (PREP) {
        if (split >= context_splits) {
            const uint32_t per_row = SAETTA_GQA_GROUP / new_heads, at = split - context_splits;
            new_rows<BITS, PACKED ? 1 : TILES == 1 ? 2 : NEW_ROWS>(a, *prep, lds_raw, THREADS / 64, at / per_row, 1, at % per_row * new_heads, new_heads);
            return;
        }
    }

    // ---- query values: requested first, so that nothing they wait for is behind the cache (loads return in order: with
    // two and four tiles, asked for when they are used, they came behind the whole first iteration, 1.5 to 2.4 us) ----
    // Item (tile t, k-step, lane l) is the 8 values that lane l feeds to the MFMA k-step;
    // operand row `on` of tile t: PACKED -> head on & 7, part on >> 3; else (row, head)
    // pair 16t + on, both parts.
    auto load_q_item = [&](int item, float (&v)[8]) {
        const int t = item / 512, step = (item / 64) & 7, l = item & 63;
        const int on = l & 15, oj = l >> 4;
        const int g = step >> 1, ab = step & 1;
        const int pair = PACKED ? (on & 7) : 16 * t + on;
        if (PACKED || pair < int(real_rows)) {  // (a single row always has its 8 heads)
            const int row = pair >> 3, head = pair & 7;
            const size_t of_head = size_t(row) * a.heads + kv * 8 + head;
            const float *src = (PREP ? prep->q_and_gate + of_head * 2 * DIM : a.q + of_head * DIM) + 64 * g + 16 * oj + 8 * ab;
            const float4 f0 = *reinterpret_cast<const float4 *>(src);
            const float4 f1 = *reinterpret_cast<const float4 *>(src + 4);
            v[0] = f0.x, v[1] = f0.y, v[2] = f0.z, v[3] = f0.w;
            v[4] = f1.x, v[5] = f1.y, v[6] = f1.z, v[7] = f1.w;
        } else {
#pragma unroll
            for (int e = 0; e < 8; e++) v[e] = 0.0f;
        }
    };
    const uint32_t position = a.tp->position, kv_len = a.tp->kv_len;
    float q_early[TILES * 2][8];
#pragma unroll
    for (int k = 0; k < TILES * 2; k++) load_q_item(tid + k * THREADS, q_early[k]);
    float norm_w[PREP ? 2 : 1][8];  // the norm's weights of the thread's dims (k-steps wave and wave + 4)
    if constexpr (PREP) {
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const float4 *src = reinterpret_cast<const float4 *>(prep->q_norm + 64 * ((wave + 4 * k) >> 1) + 16 * j + 8 * (wave & 1));
            const float4 f0 = src[0], f1 = src[1];
            norm_w[k][0] = f0.x, norm_w[k][1] = f0.y, norm_w[k][2] = f0.z, norm_w[k][3] = f0.w;
            norm_w[k][4] = f1.x, norm_w[k][5] = f1.y, norm_w[k][6] = f1.z, norm_w[k][7] = f1.w;
        }
    }

    double frequency = 0.0;
    if constexpr (PREP) {  // (while the position is on its way)
        frequency = rope_frequency(tid & 31, 32, prep->p.log2_theta);
        asm volatile("" : "+v"(frequency));
    }

    // ---- the context and this workgroup's share of it -----------------------------
    // Tokens the last row sees; the longest context of the launch.  (PREP: the tokens before the new ones.)
    const uint32_t max_len = PREP ? tokens_before(a, position, kv_len) : min(a.decode_len ? kv_len : position + a.rows, a.capacity);
    const uint32_t nblocks = (max_len + BLOCK - 1) / BLOCK;
    uint32_t blk_begin, blk_end;
    if (nblocks <= context_splits) {
        blk_begin = split;
        blk_end = split + 1;
        if (split >= nblocks) return;
    } else {
        // (split + 1) * nblocks < 2^32: at most 256 splits and 2^27 blocks (32-bit cache offsets)
        blk_begin = split * nblocks / context_splits;
        blk_end = (split + 1) * nblocks / context_splits;
    }
    const uint32_t range = blk_end - blk_begin;

    // ---- the share in iterations of at most `blocks` blocks, of whose values `value_steps` k-steps are asked for ----
    // Up to four rows ask for all an iteration may need, what it does not need out of range (see load_keys): the compiler then
    // knows how many loads are in flight at each wait, but each such load still costs its turn, eight of them 0.2 to 0.5 us.  So
    // the shares of up to 4 and up to 6 blocks have code of their own.  Us a layer, ten layers in a graph, 8192 tokens of capacity
    // (halves, 8-bit, 4-bit): 1000 tokens (2 blocks) one row 8.9 -> 7.9, 8.5 -> 8.1, 8.6 -> 8.1, two rows 10.1 -> 9.3, 9.6 -> 9.2, 9.7 -> 9.3;
    // 6000 tokens (6) one row 10.1 -> 9.6, 9.7 -> 9.3, 9.5 -> 9.1, two rows of halves 11.7 -> 11.3 (of codes 11.1 -> 11.3, so they go on
    // with all four k-steps); from 7 blocks on as before within 1 % (two rows 1.5 %).  Twelve blocks in one iteration, for shares
    // of 9 to 12, were ahead of two by 0.3 us and took as much from the shares of 7 and 8.  Three and four rows, whose iterations are of 12
    // blocks, have code for up to 4 and up to 8 (3 rows, 8-bit and 4-bit: 1000 tokens 12.9 -> 12.4 and 12.9 -> 12.3, 8000, of 8 blocks, 15.9 ->
    // 15.1 and 16.0 -> 14.7); from 9 blocks on within 1 %, 2656 tokens of 2688 1.7 %.
    auto walk = [&](auto blocks, auto value_steps) __attribute__((always_inline)) {
        using Sh = Shape<BITS, TILES, PACKED, decltype(blocks)::value>;
        constexpr int IT_BLOCKS = Sh::IT_BLOCKS, IT_TOKENS = Sh::IT_TOKENS, SC_STRIDE = Sh::SC_STRIDE;
        constexpr int KROUNDS = IT_BLOCKS / 4, KSTEPS = decltype(value_steps)::value;
        half8 *q_lds = reinterpret_cast<half8 *>(lds_raw + Sh::Q_OFF);
        float *s_lds = reinterpret_cast<float *>(lds_raw + Sh::S_OFF);
        uint16_t *ks_lds = reinterpret_cast<uint16_t *>(lds_raw + Sh::KS_OFF);
        uint16_t *kz_lds = reinterpret_cast<uint16_t *>(lds_raw + Sh::KZ_OFF);
        uint16_t *vs_lds = reinterpret_cast<uint16_t *>(lds_raw + Sh::VS_OFF);
        uint16_t *vz_lds = reinterpret_cast<uint16_t *>(lds_raw + Sh::VZ_OFF);
        float *alpha_lds = reinterpret_cast<float *>(lds_raw + Sh::ALPHA_OFF);
        _Float16 *qz_lds = reinterpret_cast<_Float16 *>(lds_raw + Sh::QZ_OFF);
        float *zsum_lds = reinterpret_cast<float *>(lds_raw + Sh::ZSUM_OFF);
        const uint32_t n_it = (range + IT_BLOCKS - 1) / IT_BLOCKS;
        const uint32_t per_it = (range + n_it - 1) / n_it;
        const uint32_t n_rounds = n_it;
        // Four splits in a row start a quarter of their share apart, so that shares of nearly a power of two do not meet in the
        // same memory channels at every moment (see attention_partial_s_body; f16, one row: 68 against 58 us per layer at 131000
        // tokens, 39 against 33 at 65500, the same in between).  3 and 4 rows are bound by their matrix instructions.
        constexpr bool STAGGER = TILES != 2;
        const uint32_t first_round = STAGGER ? (split & 3) * n_it / 4 : 0;
        auto place = [&](uint32_t it) { return it + first_round < n_it ? it + first_round : it + first_round - n_it; };

        const uint32_t cap_rows = a.capacity * kvh;
        const __amdgpu_buffer_rsrc_t k_rsrc = make_rsrc(a.kdata, cap_rows * RB);
        const __amdgpu_buffer_rsrc_t v_rsrc = make_rsrc(a.vdata, cap_rows * RB);
        const __amdgpu_buffer_rsrc_t ks_rsrc = make_rsrc(a.kscales, QUANT ? cap_rows * 8 : 0);
        const __amdgpu_buffer_rsrc_t kz_rsrc = make_rsrc(a.kbiases, QUANT ? cap_rows * 8 : 0);
        const __amdgpu_buffer_rsrc_t vs_rsrc = make_rsrc(a.vscales, QUANT ? cap_rows * 8 : 0);
        const __amdgpu_buffer_rsrc_t vz_rsrc = make_rsrc(a.vbiases, QUANT ? cap_rows * 8 : 0);
        const int tok_stride = int(kvh) * RB;  // bytes between tokens of one kv head

        // ---- the loads of one iteration ------------------------------------------------
        // Everything an iteration reads is requested before anything is computed: keys first
        // (phase A needs them first), then the small scale/bias rows, then the values.
        KeyRegs<BITS> kreg[KROUNDS][4];
        ValRegs<BITS> vreg[KSTEPS];
        u32x2 ksr = {0, 0}, kzr = {0, 0}, vsr = {0, 0}, vzr = {0, 0};
        auto blocks_of = [&](uint32_t it) { return it < n_it ? min(per_it, blk_end - (blk_begin + place(it) * per_it)) : 0u; };
        auto load_keys = [&](uint32_t it) {
            const uint32_t base = (blk_begin + place(it) * per_it) * BLOCK, nb = blocks_of(it);
            const int voff = int((base + BLOCK * wave + n) * kvh + kv) * RB + j * key_piece<BITS>();
#pragma unroll
            for (int i = 0; i < KROUNDS; i++) {
                const bool need = uint32_t(wave + 4 * i) < nb;
                if (UNCOND || need) {
                    const int off = need ? voff : OOB;
#pragma unroll
                    for (int g = 0; g < 4; g++) kreg[i][g] = load_key<BITS>(k_rsrc, off, i * 64 * tok_stride, g);
                }
            }
        };
        auto load_scales = [&](uint32_t it) {
            if constexpr (QUANT) {
                const uint32_t base = (blk_begin + place(it) * per_it) * BLOCK;
                const bool need = uint32_t(tid) < blocks_of(it) * BLOCK;
                if (UNCOND || need) {
                    const int voff = need ? int((base + tid) * kvh + kv) * 8 : OOB;
                    ksr = __builtin_amdgcn_raw_buffer_load_b64(ks_rsrc, voff, 0, 0);
                    kzr = __builtin_amdgcn_raw_buffer_load_b64(kz_rsrc, voff, 0, 0);
                    vsr = __builtin_amdgcn_raw_buffer_load_b64(vs_rsrc, voff, 0, 0);
                    vzr = __builtin_amdgcn_raw_buffer_load_b64(vz_rsrc, voff, 0, 0);
                }
            }
        };
        auto load_values = [&](uint32_t it) {
            const uint32_t base = (blk_begin + place(it) * per_it) * BLOCK, ksteps = (blocks_of(it) + 1) / 2;
            const int voff = int((base + 8 * j) * kvh + kv) * RB + val_lane_offset<BITS>(wave, n);
#pragma unroll
            for (int ks = 0; ks < KSTEPS; ks++) {
                const bool need = uint32_t(ks) < ksteps;
                if (UNCOND || need) {
                    const int off = need ? voff : OOB;
#pragma unroll
                    for (int e = 0; e < 8; e++) {
                        const int soff = (32 * ks + e) * tok_stride;
                        vreg[ks].w[e] = __builtin_amdgcn_raw_buffer_load_b32(v_rsrc, off, soff, 0);
                        if constexpr (BITS == 16) {
                            vreg[ks].w[8 + e] = __builtin_amdgcn_raw_buffer_load_b32(v_rsrc, off + 64, soff, 0);
                        }
                    }
                }
            }
        };
        // Loads return in order: the scales first, since the barrier that publishes them must not wait for the keys, the values
        // last.  (One row: left to itself the compiler asked for the values before the keys; with the epilogue's exchanges 8-bit 300
        // tokens of 8192 8.4 -> 8.0 us a layer, halves 4096 10.0 -> 9.8.  Two rows in this order 8.9 -> 9.0, so they keep the compiler's.)
        auto in_order = [] {
            if constexpr (PACKED) __builtin_amdgcn_sched_barrier(0);
        };
        load_scales(0), in_order();
        load_keys(0), in_order();
        load_values(0), in_order();

        // ---- prologue: query rows to f16 hi/lo operands in LDS ------------------------
        // (while the first iteration's keys are in flight; the values are requested after it)
        if constexpr (PREP) {
            // the norm (each wave has two of the eight k-steps of a row's dims) and the rotation (dims 0-63: k-steps 0 and 1, the
            // waves 0 and 1; a pair's values are half a wavefront apart), where the scores will be
            float *squares = s_lds;                                       // [tile][wave][column]
            float2 *rope = reinterpret_cast<float2 *>(s_lds + 4 * 4 * 16);  // [row][32]
#pragma unroll
            for (int t = 0; t < TILES; t++) {
                float sum = 0.0f;
#pragma unroll
                for (int k = 2 * t; k < 2 * t + 2; k++) {
#pragma unroll
                    for (int e = 0; e < 8; e++) sum += q_early[k][e] * q_early[k][e];
                }
                sum = across_rows<16, 64>(sum, SumOp());
                if (j == 0) squares[(t * 4 + wave) * 16 + n] = sum;
            }
            if (tid < int(32 * a.rows)) {
                float s, c;
                rope_angle(position + (tid >> 5), frequency, s, c);
                rope[tid] = float2{s, c};
            }
            __syncthreads();
#pragma unroll
            for (int t = 0; t < TILES; t++) {
                const float *sq = squares + t * 64 + n;
                const float scale = query_scale((sq[0] + sq[16]) + (sq[32] + sq[48]), prep->p.eps);
#pragma unroll
                for (int k = 0; k < 2; k++) {
#pragma unroll
                    for (int e = 0; e < 8; e++) q_early[2 * t + k][e] *= scale * norm_w[k][e];
                }
                if (wave < 2) {
                    const int row = PACKED ? 0 : min(2 * t + (n >> 3), int(a.rows) - 1);
#pragma unroll
                    for (int e = 0; e < 8; e++) {
                        const float2 sc = rope[row * 32 + 16 * (j & 1) + 8 * wave + e];
                        const float x = q_early[2 * t][e], other = half_swap(x, j < 2);
                        q_early[2 * t][e] = j < 2 ? rope_first(x, other, sc.x, sc.y) : rope_second(other, x, sc.x, sc.y);
                    }
                }
            }
        }
        {
            const float qmul = a.scale * 1.4426950408889634f * Q_UP;
#pragma unroll
            for (int k = 0; k < TILES * 2; k++) {
                const int item = tid + k * THREADS;
                const int t = item / 512, step = (item / 64) & 7, l = item & 63;
                const int on = l & 15;
                const float (&v)[8] = q_early[k];
                half8 hi, lo;
                float sum_hi = 0.0f, sum_lo = 0.0f;
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    _Float16 h, lw;
                    split_hi_lo(v[key_slot_dim<BITS>(e)] * qmul, h, lw);
                    hi[e] = h;
                    lo[e] = lw;
                    sum_hi += (float)h;
                    sum_lo += (float)lw;
                }
                float sum;
                if constexpr (PACKED) {
                    q_lds[step * 64 + l] = (on < 8) ? hi : lo;
                    sum = (on < 8) ? sum_hi : sum_lo;
                } else {
                    q_lds[((t * 2 + 0) * 8 + step) * 64 + l] = hi;
                    q_lds[((t * 2 + 1) * 8 + step) * 64 + l] = lo;
                    sum = sum_hi + sum_lo;
                }
                // The key bias term sum_g z_g * sum_{d in g} q_d is one more MFMA over the same 32
                // (lane group, slot) pairs: its B operand holds, in lane l and slot `step`, the sum of
                // the 8 operand values this item made (divided by Q_UP, as hi and lo halves), and its
                // A operand holds z_g of the step's group.
                if constexpr (QUANT) {
                    _Float16 h, lw;
                    split_hi_lo(sum * (1.0f / Q_UP), h, lw);
                    qz_lds[((t * 2 + 0) * 64 + l) * 8 + step] = h;
                    qz_lds[((t * 2 + 1) * 64 + l) * 8 + step] = lw;
                }
            }
        }
        __syncthreads();

        // Query operands of a single tile live in registers for the whole kernel.
        half8 q_reg[TILES == 1 ? PARTS * 8 : 1];
        half8 qz_reg[2] = {{0, 0, 0, 0, 0, 0, 0, 0}, {0, 0, 0, 0, 0, 0, 0, 0}};
        if constexpr (TILES == 1) {
#pragma unroll
            for (int i = 0; i < PARTS * 8; i++) q_reg[i] = q_lds[i * 64 + lane];
            if constexpr (QUANT) {
                qz_reg[0] = *reinterpret_cast<const half8 *>(qz_lds + lane * 8);
                qz_reg[1] = *reinterpret_cast<const half8 *>(qz_lds + (64 + lane) * 8);
            }
        }

        // ---- running state -------------------------------------------------------------
        // Phase B: thread (row, part) of SOFT_ROWS x TPR.
        const int b_row = tid / Sh::TPR, b_part = tid % Sh::TPR;
        uint32_t b_len;  // tokens row b_row sees
        {
            const int vrow = PACKED ? 0 : b_row >> 3;
            const bool real = PACKED || b_row < int(real_rows);
            const uint32_t len = PREP ? max_len : a.decode_len ? kv_len : position + vrow + 1;
            b_len = real ? min(len, a.capacity) : 0;
        }
        float m_run = NO_SCORE, l_part = 0.0f;
        // Phase C: accumulators of this wave's 64 dims, per tile 4 output tiles of 16 dims.
        floatx4 acc[TILES][4];
        float zacc[TILES];
#pragma unroll
        for (int t = 0; t < TILES; t++) {
            zacc[t] = 0.0f;
#pragma unroll
            for (int e = 0; e < 4; e++) acc[t][e] = floatx4{0, 0, 0, 0};
        }

        // What phase B leaves for phase C: P * P_UP; over halves, where no scale goes into it, its hi and lo parts side by side
        // (every wave takes all rows' P: split here, once, it is two permutes for two values there).
        constexpr bool P_SPLIT = BITS == 16 && !PACKED;
        auto p_word = [&](float x) {
            if constexpr (!P_SPLIT) return x;
            _Float16 h, lw;
            split_hi_lo(x, h, lw);
            return __builtin_bit_cast(float, uint32_t(__builtin_bit_cast(uint16_t, h)) | uint32_t(__builtin_bit_cast(uint16_t, lw)) << 16);
        };
        for (uint32_t round = 0; round < n_rounds; round++) {
            const uint32_t it = round;
            const uint32_t blk0 = blk_begin + place(it) * per_it;
            const uint32_t nb = blocks_of(it);  // blocks of this iteration, 0..ITB
            const uint32_t base = blk0 * BLOCK;
            const uint32_t it_tokens = nb * BLOCK;
            const uint32_t ksteps = (nb + 1) / 2;

            // Scales and biases of the iteration's tokens to LDS: thread = token, 4 groups each.  The key
            // ones before the barrier (phase A reads them); the value ones after it: a wave may still be
            // reading the previous iteration's in its phase C until every wave has arrived here.
            if constexpr (QUANT) {
                if (tid < IT_TOKENS) {
                    *reinterpret_cast<u32x2 *>(ks_lds + 4 * tid) = ksr;
                    *reinterpret_cast<u32x2 *>(kz_lds + 4 * tid) = kzr;
                }
            }
            __syncthreads();  // key scales visible; the previous iteration's phase C is over
            if constexpr (QUANT) {
                if (tid < IT_TOKENS) {
                    // Tokens past the context or the iteration get value scale 0 and bias 0, so that
                    // whatever their rows hold stays out of O (their probabilities are 0 as well).
                    if (uint32_t(tid) >= it_tokens || base + tid >= max_len) vsr = u32x2{0, 0}, vzr = u32x2{0, 0};
                    vs_lds[0 * IT_TOKENS + tid] = uint16_t(vsr.x), vs_lds[1 * IT_TOKENS + tid] = uint16_t(vsr.x >> 16);
                    vs_lds[2 * IT_TOKENS + tid] = uint16_t(vsr.y), vs_lds[3 * IT_TOKENS + tid] = uint16_t(vsr.y >> 16);
                    vz_lds[0 * IT_TOKENS + tid] = uint16_t(vzr.x), vz_lds[1 * IT_TOKENS + tid] = uint16_t(vzr.x >> 16);
                    vz_lds[2 * IT_TOKENS + tid] = uint16_t(vzr.y), vz_lds[3 * IT_TOKENS + tid] = uint16_t(vzr.y >> 16);
                }
            }
            // ---- phase A: scores -------------------------------------------------------
#pragma unroll
            for (int t = 0; t < TILES; t++) {
                half8 qt[PARTS * 8];
                half8 qz[2] = {qz_reg[0], qz_reg[1]};
                if constexpr (TILES == 1) {
#pragma unroll
                    for (int i = 0; i < PARTS * 8; i++) qt[i] = q_reg[i];
                } else {
#pragma unroll
                    for (int i = 0; i < PARTS * 8; i++) qt[i] = q_lds[(t * PARTS * 8 + i) * 64 + lane];
                    if constexpr (QUANT) {
                        qz[0] = *reinterpret_cast<const half8 *>(qz_lds + ((t * 2 + 0) * 64 + lane) * 8);
                        qz[1] = *reinterpret_cast<const half8 *>(qz_lds + ((t * 2 + 1) * 64 + lane) * 8);
                    }
                }
#pragma unroll
                for (int i = 0; i < KROUNDS; i++) {
                    const int blk = wave + 4 * i;
                    if (uint32_t(blk) >= nb) break;
                    const int tok0 = BLOCK * blk + 4 * j;  // this lane's 4 tokens in C layout
                    floatx4 s = {0, 0, 0, 0};
                    if constexpr (QUANT) {
                        // bias term: slot e of every lane group belongs to group e / 2 of token n
                        const u32x2 zr = *reinterpret_cast<const u32x2 *>(kz_lds + 4 * (BLOCK * blk + n));
                        const half8 zop = as_half8(perm(0, zr.x, 0x01000100u), perm(0, zr.x, 0x03020302u),
                                                   perm(0, zr.y, 0x01000100u), perm(0, zr.y, 0x03020302u));
                        s = __builtin_amdgcn_mfma_f32_16x16x32_f16(zop, qz[0], s, 0, 0, 0);
                        s = __builtin_amdgcn_mfma_f32_16x16x32_f16(zop, qz[1], s, 0, 0, 0);
                    }
                    floatx4 r[4];
#pragma unroll
                    for (int g = 0; g < 4; g++) {
                        r[g] = floatx4{0, 0, 0, 0};
#pragma unroll
                        for (int ab = 0; ab < 2; ab++) {
                            const half8 kop = key_operand<BITS>(kreg[i][g], ab);
#pragma unroll
                            for (int part = 0; part < PARTS; part++) {
                                r[g] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kop, qt[part * 8 + g * 2 + ab], r[g], 0,
                                                                              0, 0);
                            }
                        }
                    }
                    if constexpr (QUANT) {
                        // scales of tokens tok0..tok0+3, 4 groups each: 32 contiguous bytes
                        const u32x4 s01 = *reinterpret_cast<const u32x4 *>(ks_lds + 4 * tok0);
                        const u32x4 s23 = *reinterpret_cast<const u32x4 *>(ks_lds + 4 * tok0 + 8);
                        const uint32_t sw[8] = {s01.x, s01.y, s01.z, s01.w, s23.x, s23.y, s23.z, s23.w};
                        constexpr float C1 = code_up<BITS>() / Q_UP;
#pragma unroll
                        for (int tk = 0; tk < 4; tk++) {
                            float d = 0.0f;
#pragma unroll
                            for (int g = 0; g < 4; g++) {
                                d += half_bits_to_float(sw[2 * tk + (g >> 1)] >> (16 * (g & 1))) * r[g][tk];
                            }
                            s[tk] += d * C1;
                        }
                    } else {
#pragma unroll
                        for (int tk = 0; tk < 4; tk++) s[tk] = (r[0][tk] + r[1][tk] + r[2][tk] + r[3][tk]) * (1.0f / Q_UP);
                    }
                    *reinterpret_cast<floatx4 *>(s_lds + (16 * t + n) * SC_STRIDE + tok0) = s;
                }
            }
            // The key registers and the scale registers are free: request the next iteration's.
            if (it + 1 < n_it) {
                load_scales(it + 1);
                load_keys(it + 1);
            }
            __syncthreads();

            // ---- phase B: online softmax per row ---------------------------------------
            // Writes P * P_UP over the scores; l sums the plain P.
            {
                // A thread's tokens: TPT in a row, or (three and four tiles, 48 of them) CH in a row of every 32, so that a k-step
                // without tokens is no work for anyone (8 rows at 300 tokens, 8-bit 23.7 -> 23.1 us a layer; two rows 12.0 -> 12.3).
                constexpr bool BY_STEP = TILES >= 3;
                constexpr int CH = BY_STEP ? 32 / Sh::TPR : Sh::TPT, STEP = CH % 4 == 0 ? 4 : 2;
                static_assert(CH % STEP == 0, "whole pieces");
                typedef float piece __attribute__((ext_vector_type(STEP)));
                float sv[Sh::TPT];
                const bool scores = Sh::SOFT_ROWS == Sh::S_ROWS || PACKED || b_row < Sh::S_ROWS;  // (three tiles: the last wave has no rows)
                float *row = s_lds + (scores ? b_row : 0) * SC_STRIDE + b_part * CH;
                const uint32_t tok0 = b_part * CH;
                // tokens of this row in this iteration: inside the iteration and inside the row's context
                const uint32_t lim = b_len > base ? min(b_len - base, it_tokens) : 0;
                auto steps = [&](bool all, auto f) {  // f(index of the thread's value, the token's place in the iteration)
#pragma unroll
                    for (int i = 0; i < Sh::TPT; i += CH) {
                        const int at = i / CH * 32;
                        if (BY_STEP && !all && uint32_t(i / CH) >= ksteps) break;
#pragma unroll
                        for (int k = 0; k < CH; k += STEP) f(i + k, at + k);
                    }
                };
                float cm = NO_SCORE;
                steps(true, [&](int i, int at) {
                    piece v = *reinterpret_cast<const piece *>(row + at);
                    if constexpr (PACKED) v += *reinterpret_cast<const piece *>(row + 8 * SC_STRIDE + at);
#pragma unroll
                    for (int e = 0; e < STEP; e++) {
                        sv[i + e] = v[e];
                        cm = (tok0 + at + e < lim) ? fmaxf(cm, v[e]) : cm;
                    }
                });
                cm = group_reduce<Sh::TPR>(cm, MaxOp());
                const float nm = fmaxf(m_run, cm);
                const float al = __builtin_amdgcn_exp2f(m_run - nm);
                float sum = 0.0f;
                steps(false, [&](int i, int at) {
                    piece v;
#pragma unroll
                    for (int e = 0; e < STEP; e++) {
                        const float x = (tok0 + at + e < lim) ? __builtin_amdgcn_exp2f(sv[i + e] - nm) : 0.0f;
                        sum += x;
                        v[e] = p_word(x * P_UP);
                    }
                    if (scores) *reinterpret_cast<piece *>(row + at) = v;
                });
                l_part = l_part * al + sum;
                m_run = nm;
                if (scores) {
                    if (b_part == 0) alpha_lds[b_row] = al;
                }
            }
            __syncthreads();

            // ---- phase C: O += P V for this wave's group -------------------------------
            // The probability operands need only P and the value scales, so they are all built
            // before the first value code is touched: what is left to do once the (large,
            // last-requested) value loads land is the byte permutes and the MFMAs.
            auto build_p = [&](int t, int ks, half8 &phi, half8 &plo) {
                const float *prow = s_lds + (PACKED ? (n & 7) : 16 * t + n) * SC_STRIDE;
                const int tk = 32 * ks + 8 * j;
                const floatx4 p0 = *reinterpret_cast<const floatx4 *>(prow + tk);
                const floatx4 p1 = *reinterpret_cast<const floatx4 *>(prow + tk + 4);
                float pv[8] = {p0[0], p0[1], p0[2], p0[3], p1[0], p1[1], p1[2], p1[3]};
                if constexpr (QUANT) {
                    const u32x4 sr = *reinterpret_cast<const u32x4 *>(vs_lds + wave * IT_TOKENS + tk);
                    const u32x4 zr = *reinterpret_cast<const u32x4 *>(vz_lds + wave * IT_TOKENS + tk);
                    const uint32_t sw[4] = {sr.x, sr.y, sr.z, sr.w}, zw[4] = {zr.x, zr.y, zr.z, zr.w};
#pragma unroll
                    for (int e = 0; e < 8; e++) {
                        zacc[t] += pv[e] * half_bits_to_float(zw[e >> 1] >> (16 * (e & 1)));
                        pv[e] *= half_bits_to_float(sw[e >> 1] >> (16 * (e & 1)));
                    }
                }
                if constexpr (PACKED) {
                    // hi lanes (n < 8) keep x and let the conversion truncate it to its hi part;
                    // lo lanes subtract the hi part first.
                    const uint32_t lo_mask = (n >= 8) ? 0xffffe000u : 0u;
                    uint32_t o[4];
#pragma unroll
                    for (int e = 0; e < 8; e += 2) {
                        const float x0 = pv[e] - __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, pv[e]) & lo_mask);
                        const float x1 =
                            pv[e + 1] - __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, pv[e + 1]) & lo_mask);
                        // round toward zero: exact truncation to the hi part in hi lanes
                        o[e / 2] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(x0, x1));
                    }
                    phi = as_half8(o[0], o[1], o[2], o[3]);
                } else if constexpr (P_SPLIT) {
                    uint32_t h[4], lw[4];
#pragma unroll
                    for (int e = 0; e < 8; e += 2) {
                        const uint32_t w0 = __builtin_bit_cast(uint32_t, pv[e]), w1 = __builtin_bit_cast(uint32_t, pv[e + 1]);
                        h[e / 2] = perm(w1, w0, 0x05040100u), lw[e / 2] = perm(w1, w0, 0x07060302u);
                    }
                    phi = as_half8(h[0], h[1], h[2], h[3]), plo = as_half8(lw[0], lw[1], lw[2], lw[3]);
                } else {
#pragma unroll
                    for (int e = 0; e < 8; e++) {
                        _Float16 h, lw;
                        split_hi_lo(pv[e], h, lw);
                        phi[e] = h;
                        plo[e] = lw;
                    }
                }
            };
#pragma unroll
            for (int t = 0; t < TILES; t++) {
                // Rescale what was summed so far.  Accumulator rows (C layout) are 4j..4j+3.
                if (round > 0) {
                    const int arow = PACKED ? ((4 * j) & 7) : 16 * t + 4 * j;
                    const floatx4 al = *reinterpret_cast<const floatx4 *>(alpha_lds + arow);
#pragma unroll
                    for (int e = 0; e < 4; e++) acc[t][e] *= al;
                    zacc[t] *= alpha_lds[PACKED ? (n & 7) : 16 * t + n];
                }
                if constexpr (PACKED) {
                    half8 phi[KSTEPS], plo[KSTEPS];
#pragma unroll
                    for (int ks = 0; ks < KSTEPS; ks++) {
                        if (uint32_t(ks) < ksteps) build_p(t, ks, phi[ks], plo[ks]);
                    }
#pragma unroll
                    for (int ks = 0; ks < KSTEPS; ks++) {
                        if (uint32_t(ks) >= ksteps) break;
                        if constexpr (BITS == 16) {
                            // Rows past the context may hold anything, NaN included: 0 * NaN must not reach O.
#pragma unroll
                            for (int e = 0; e < 8; e++) {
                                if (base + 32 * ks + 8 * j + e >= max_len) vreg[ks].w[e] = 0, vreg[ks].w[8 + e] = 0;
                            }
                        }
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            const half8 vop = val_operand<BITS>(vreg[ks], e, n);
                            acc[t][e] = __builtin_amdgcn_mfma_f32_16x16x32_f16(phi[ks], vop, acc[t][e], 0, 0, 0);
                            if constexpr (!PACKED) {
                                acc[t][e] = __builtin_amdgcn_mfma_f32_16x16x32_f16(plo[ks], vop, acc[t][e], 0, 0, 0);
                            }
                        }
                    }
                }
            }
            if constexpr (!PACKED) {
                // (the k-steps outside: a step's value operands are permuted once for all tiles)
#pragma unroll
                for (int ks = 0; ks < KSTEPS; ks++) {
                    if (uint32_t(ks) >= ksteps) break;
                    if constexpr (BITS == 16) {
#pragma unroll
                        for (int e = 0; e < 8; e++) {
                            if (base + 32 * ks + 8 * j + e >= max_len) vreg[ks].w[e] = 0, vreg[ks].w[8 + e] = 0;
                        }
                    }
                    half8 vop[4];
#pragma unroll
                    for (int e = 0; e < 4; e++) vop[e] = val_operand<BITS>(vreg[ks], e, n);
#pragma unroll
                    for (int t = 0; t < TILES; t++) {
                        half8 phi, plo;
                        build_p(t, ks, phi, plo);
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            acc[t][e] = __builtin_amdgcn_mfma_f32_16x16x32_f16(phi, vop[e], acc[t][e], 0, 0, 0);
                            acc[t][e] = __builtin_amdgcn_mfma_f32_16x16x32_f16(plo, vop[e], acc[t][e], 0, 0, 0);
                        }
                    }
                }
            }
            if (it + 1 < n_it) load_values(it + 1);
        }

        // ---- epilogue: one partial per (row, head) ------------------------------------
        // m and l from the phase B threads.
        l_part = group_reduce<Sh::TPR>(l_part, SumOp());
        if (b_part == 0 && (PACKED || b_row < int(real_rows))) {
            const int vrow = PACKED ? 0 : b_row >> 3, head = b_row & 7;
            const size_t slot = (size_t(vrow) * a.nsplits + split) * a.heads + kv * 8 + head;
            *reinterpret_cast<floatx2 *>(a.part_ml + 2 * slot) = floatx2{m_run, l_part};
        }
        // Bias sums: reduce over the 4 lane groups, hand to the C-layout lanes through LDS.
        if constexpr (QUANT) {
#pragma unroll
            for (int t = 0; t < TILES; t++) {
                float z = zacc[t];
                z = across_rows<16, 64>(z, SumOp());
                // One copy per wave: the sum of wave w's group lives at [w][row].
                if (j == 0 && (!PACKED || n < 8)) zsum_lds[wave * Sh::S_ROWS + 16 * t + n] = z;
            }
            // written and read by lanes of the same wave: no workgroup barrier
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
        constexpr float unscale = code_up<BITS>() / P_UP;
#pragma unroll
        for (int t = 0; t < TILES; t++) {
            // PACKED: rows 8-15 hold the lo part of rows 0-7, lanes j + 2 those of lanes j: the sums of register i end up in the lanes
            // j = 0, 1 and those of register i + 2 in the lanes 2, 3 (one exchange and one addition for both, and every lane stores).
            floatx4 o[4];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                o[e] = acc[t][e];
                if constexpr (PACKED) {
#pragma unroll
                    for (int i = 0; i < 2; i++) {
                        // (the builtin: what reads a matrix instruction's result has to be an instruction that the compiler knows)
                        const float first = o[e][i], third = o[e][i + 2];
                        const auto both = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, first), __builtin_bit_cast(uint32_t, third), false, false);
                        o[e][i] = __builtin_bit_cast(float, uint32_t(both[0])) + __builtin_bit_cast(float, uint32_t(both[1]));
                    }
                }
            }
#pragma unroll
            for (int i = 0; i < (PACKED ? 2 : 4); i++) {
                const int pair = PACKED ? 4 * (j & 1) + 2 * (j >> 1) + i : 16 * t + 4 * j + i;  // (row, head) pair of this accumulator row
                if (!PACKED && pair >= int(real_rows)) continue;
                const int vrow = PACKED ? 0 : pair >> 3, head = pair & 7;
                const float zb = QUANT ? zsum_lds[wave * Sh::S_ROWS + pair] * (1.0f / P_UP) : 0.0f;
                const size_t slot = (size_t(vrow) * a.nsplits + split) * a.heads + kv * 8 + head;
                float *dst = a.part_o + slot * DIM + 64 * wave;
                // (Five to eight rows past the caches: up to 17 MB that the L2s would hold dirty until the kernel's end, 27.0 against
                // 27.7 us a layer for 8 rows at 7000 tokens.  Fewer rows are read back sooner than they are written out: plain.)
                auto put = [&](float *to, auto value) {
                    if constexpr (TILES >= 3) __builtin_nontemporal_store(value, reinterpret_cast<decltype(value) *>(to));
                    else *reinterpret_cast<decltype(value) *>(to) = value;
                };
                if constexpr (BITS == 16) {
                    // tile e: dims 32*(e/2) + 2n + e%2
                    put(dst + 2 * n, floatx2{o[0][i] * unscale, o[1][i] * unscale});
                    put(dst + 32 + 2 * n, floatx2{o[2][i] * unscale, o[3][i] * unscale});
                } else {
                    put(dst + 4 * n, floatx4{o[0][i] * unscale + zb, o[1][i] * unscale + zb, o[2][i] * unscale + zb, o[3][i] * unscale + zb});
                }
            }
        }
    };
    using std::integral_constant;
    if constexpr (UNCOND && TILES == 2) {
        if (range <= 4) walk(integral_constant<int, 4>(), integral_constant<int, 2>());
        else if (range <= 8) walk(integral_constant<int, 8>(), integral_constant<int, 4>());
        else walk(integral_constant<int, ITB>(), integral_constant<int, ITB / 2>());
    } else if constexpr (UNCOND) {
        constexpr bool HAS_3 = PACKED || BITS == 16;
        if (__builtin_expect(range > (HAS_3 ? 6 : 4), 1)) walk(integral_constant<int, ITB>(), integral_constant<int, ITB / 2>());
        else if (HAS_3 && range > 4) walk(integral_constant<int, ITB>(), integral_constant<int, HAS_3 ? 3 : ITB / 2>());
        else walk(integral_constant<int, 4>(), integral_constant<int, 2>());
    } else {
        walk(integral_constant<int, ITB>(), integral_constant<int, ITB / 2>());
    }
}

// One query row over codes (a single packed tile) fits two waves per SIMD, i.e. two workgroups
// per CU (attention_partial_kernel_1, for long contexts); the others take the whole register file
// and run one workgroup per CU.  Which one runs is decided in run_attention.
// Blocks per iteration of each kernel.
constexpr int ITB_TWO_PER_CU = 12, ITB_ONE_PER_CU = 8;
template <int TILES>
constexpr int itb_rows() {
    return TILES == 1 ? 8 : 12;
}
// UNCOND of each kernel (three and four rows over halves come to theirs with SAETTA_STAGE_NO_LOADERS only, and stay as they were)
template <int BITS, int TILES>
constexpr bool all_asked() {
    return TILES == 1 || (TILES == 2 && BITS != 16);
}

template <int BITS>
__global__ __launch_bounds__(THREADS, 2) void attention_partial_kernel_1(PartialArgs a) {
    attention_partial_body<BITS, 1, true, ITB_TWO_PER_CU, false>(a);
}

template <int BITS, int TILES>
__global__ __launch_bounds__(THREADS) void attention_partial_kernel_n(PartialArgs a) {
    attention_partial_body<BITS, TILES, false, itb_rows<TILES>(), all_asked<BITS, TILES>()>(a);
}

template <int BITS>
__global__ __launch_bounds__(THREADS) void attention_partial_kernel_p(PartialArgs a) {
    attention_partial_body<BITS, 1, true, ITB_ONE_PER_CU, true>(a);
}

// The same with the step before the scores taken in.
template <int BITS, int TILES>
__global__ __launch_bounds__(THREADS) void attention_token_kernel_n(TokenArgs t) {
    attention_partial_body<BITS, TILES, false, itb_rows<TILES>(), all_asked<BITS, TILES>(), true>(t.a, &t.prep, t.new_heads);
}
template <int BITS>
__global__ __launch_bounds__(THREADS) void attention_token_kernel_p(TokenArgs t) {
    attention_partial_body<BITS, 1, true, ITB_ONE_PER_CU, true, true>(t.a, &t.prep, t.new_heads);
}

// What a wave of attention_partial_kernel_s does when a bounded wait on an LDS counter has run out (it never
// should): one lane stores a code in the device's sticky status word, which the host reads at its next call
// (a plain vector store to pinned host memory), and the workgroup's partials get l = NaN, so that the
// reduce stage gives NaN for these (row, head) pairs and never a plausible number.  (If the wave that stores
// the maxima and sums is still to come and has not given up itself, its store wins; the status word stands.)
__device__ __noinline__ void wait_gave_up(uint32_t *status, float *part_ml, uint32_t code, uint32_t rows, uint32_t nsplits,
                                          uint32_t split, uint32_t heads, uint32_t kv) {
    const uint32_t lane = threadIdx.x & 63;
    if (lane == 0) __hip_atomic_store(status, code, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    if (lane < 8 * rows) {
        const size_t slot = (size_t(lane >> 3) * nsplits + split) * heads + kv * 8 + (lane & 7);
        part_ml[2 * slot + 1] = __builtin_nanf("");
    }
}

// ---- one to four query rows over codes, keys first ------------------------------------------------
// attention_partial_kernel_s: the workgroup's share is taken in rounds of up to 17 blocks of 16
// tokens whose codes all lie in LDS at once (17: a context of 128 x 256 tokens and a few more still
// is one round).  The KEYS of a round are requested before its values, so they are there when half
// of the round's bytes are, and everything that does not need a value code runs while the values
// are still on their way: the scores of all the tokens, their softmax (every block relative to its
// own maximum, by the wave that computed its scores; the blocks are joined by one factor per block
// and head), and the probability operands P * value scale.  When the last values land, what is left
// is one k-step of O += P V per wave (8 LDS reads, 16 byte permutes, 4 MFMAs), the merge of two
// waves and the store.
// Eight computing waves and four loader waves that move codes from global memory straight into LDS
// (global_load_lds, no registers): two request the round's scales, biases and keys, and two, once
// those requests are out, the values.  A loader waits for its own loads in order and raises a
// counter in LDS when a part of the keys, or a 64-token slot of the values, has landed.  In phase A
// computing wave w takes the blocks w and w + 8 (wave 0 also block 16); in phase C waves 2g and
// 2g + 1 share quantization group g (dims 64g .. 64g + 63) and take alternate k-steps of 32 tokens,
// so that each of the round's value slots gives every wave one k-step.
// A wave that requests more than the memory pipeline takes stands still until it is accepted, so a
// wave that requests values cannot tell anybody that earlier data is there: that is why the keys and
// the values have different requesters, and why the waves meet through counters in LDS and not
// through s_barrier (which would wait for the loaders to finish requesting).  LDS executes a wave's
// instructions in order, so data written before a counter is raised is there when the counter is
// seen.  Every wait on a counter is bounded (SPIN_LIMIT polls), so every wave ends whatever happens.
// Longer shares take further rounds with an online softmax between the rounds.
// M query rows (a verify step, 2..4) take one round over codes that serve every row; two rows share a
// tile (see the rows' part of the kernel).
template <int BITS, int M>
struct KeysFirst {
    static constexpr int PAIRS = (M + 1) / 2;               // tiles of two query rows (one row: its own tile)
    static constexpr int LOADERS = 4, WAVES = 8;            // loader waves (keys: 0, 1; values: 2, 3), then the computing waves
    static constexpr int K_LOADERS = 2, V_LOADERS = 2;
    static constexpr int RB_ = BITS * 32;                   // bytes of a (token, kv head) row of codes
    static constexpr int ROUND_BLOCKS = 17, ROUND_TOKENS = ROUND_BLOCKS * BLOCK;
    // One row, a share of more than one round: rounds of ALT_BLOCKS blocks that ALTERNATE between two halves of the
    // keys' and the values' places (and of the scales and the block table), so that the loaders are a round ahead of
    // the computing waves and the stream from memory never waits for them.  The halves are the blocks 0-7 and 8-15 of
    // the single round's places.  (Rounds of 16 blocks for 4-bit codes, which are half the bytes, in places of 32
    // blocks: measured slower, 30.0 against 28.3 us at 150k tokens; the code below takes either.)
    static constexpr bool ALTERNATE = M == 1;
    static constexpr int ALT_BLOCKS = 8;
    static constexpr int AREA_BLOCKS = (ALTERNATE && 2 * ALT_BLOCKS > ROUND_BLOCKS) ? 2 * ALT_BLOCKS : ROUND_BLOCKS;  // blocks of codes LDS has room for, keys and values each
    static constexpr int SB_TOKENS = AREA_BLOCKS * BLOCK;
    static constexpr int KSTEPS = (ROUND_BLOCKS + 1) / 2;   // of 32 tokens; the last one is half there
    static constexpr int SLOTS = (KSTEPS + 1) / 2;          // value slots of 64 tokens: 5, the last one block 16 alone
    static constexpr int PIECES = RB_ / 16;
    static constexpr int PER_BLOCK = PIECES / 4;            // load instructions per block of keys, and of values: 4 | 2
    static constexpr int V_GROUP_TOKENS = 64 / PIECES;      // token rows one load instruction brings: 4 | 8
    static constexpr int K_BLOCK_BYTES = BLOCK * RB_;       // [64-byte piece][token]: what one load instruction brings
    // Values: whole token rows, each rotated by a quarter row per 8 tokens ((token / 8) % 4 quarters),
    // so that the four lane groups of a value read, which are 8 tokens apart, fall on different banks.
    static constexpr int V_ROT = RB_ / 4;
    static constexpr int K_LOADS = 8 * PER_BLOCK;           // per key-loader wave: blocks 0-15, half of them before the other
    static constexpr int V_LOADS = 8 * PER_BLOCK;           // per value-loader wave: slots 0-3
    static constexpr int SC_LOADS = 16;                     // scales and biases of a key loader's 128 tokens: 4 arrays x 2 planes x 2
    static constexpr int X_LOADS = 8 + PER_BLOCK;           // block 16: its scales and biases (4 arrays x 2 planes) and its keys
    static_assert(SC_LOADS + K_LOADS + X_LOADS < 64, "vmcnt is 6 bits");
    // LDS map, in bytes.  The scores of a block (its probabilities relative to the block's maximum,
    // [row][head][token] f32, 512 bytes a row) lie over the block's own keys, which only the wave that
    // writes them has read.
    static constexpr int Q_OFF = 0;                                // [k-step][lane] half8: one row's operands at a time
    static constexpr int QZ_OFF = Q_OFF + 8 * 64 * 16;             // [hi, lo][lane][k-step] f16
    // scales and biases: per array two planes of one dword per token, the f16 of groups (0, 1) and of (2, 3)
    static constexpr int SB_OFF = QZ_OFF + 2 * 64 * 16;            // [ks | kz | vs | vz][plane][token] u32
    static constexpr int SB_ARRAY = 2 * SB_TOKENS * 4;
    // the blocks' maxima and sums, [row][head][block]: one row has room for a stride of 20 (16-byte reads; blocks 17-19
    // never exist: maximum "none", sum 0), several rows have not
    static constexpr int BSTRIDE = M == 1 ? (AREA_BLOCKS + 3) / 4 * 4 : ROUND_BLOCKS;
    static constexpr int BSINGLE = (ROUND_BLOCKS + 3) / 4 * 4;      // entries of a row that a single round looks at (one row)
    static constexpr int BROW = 8 * BSTRIDE;                       // floats of a row's table
    static constexpr int BMAX_OFF = SB_OFF + 4 * SB_ARRAY;         // [row][head][block] f32: the block's maximum score
    static constexpr int BSUM_OFF = BMAX_OFF + M * BROW * 4;       // [row][head][block] f32: sum of 2^(score - maximum)
    static constexpr int ZS_OFF = BSUM_OFF + M * BROW * 4;         // [wave][pair][column] f32 (one row: [wave][head])
    static constexpr int SYNC_OFF = ZS_OFF + WAVES * PAIRS * 16 * 4;  // 32 counters, u32
    static constexpr int K_OFF = (SYNC_OFF + 32 * 4 + 255) / 256 * 256;
    static constexpr int V_OFF = K_OFF + AREA_BLOCKS * K_BLOCK_BYTES;
    // Several rows over a share of more than one round: rounds of SHORT_BLOCKS blocks, which leave room in
    // LDS for every pair's query operands to stay ([pair][hi, lo][k-step][lane] half8, then [pair][hi, lo][lane][k-step]
    // f16 of the key bias term), so that they need no registers between one round's scores and the next's.
    // 8-bit codes: over the keys' blocks that short rounds never fill; 4-bit: behind the values.
    // (Two pairs: rounds of 12, for which there is room.  A round costs 2.6 us beside its bytes, and with the new
    // tokens' split taken out of the context's 128 a share of 32 blocks is one of 33, a fifth round of 8: four rows at 65500
    // tokens, 4-bit, 42.3 -> 38.5 us a layer, 120000 60.7 -> 56.0, 262000 114.6 -> 105.5; 8-bit 42.0 -> 37.7, 57.6 -> 54.5,
    // 109.3 -> 99.4; behind at some lengths between: 80000 43.9 -> 44.9; and behind without the new tokens' split, where
    // shares of 32 and 64 blocks are whole rounds of 8: four rows, 8-bit, at 65000 tokens 37.8 -> 38.2, 131000 62.5 -> 64.2.)
    static constexpr int SHORT_BLOCKS = PAIRS == 2 ? 12 : 8;
    static constexpr int QP_PAIR_BYTES = 2 * 8 * 64 * 16, QPZ_PAIR_BYTES = 2 * 64 * 16;
    static constexpr int QP_BYTES = M > 1 ? PAIRS * (QP_PAIR_BYTES + QPZ_PAIR_BYTES) : 0;
    static constexpr int QP_OFF = BITS == 8 ? K_OFF + SHORT_BLOCKS * K_BLOCK_BYTES : V_OFF + AREA_BLOCKS * K_BLOCK_BYTES;
    static constexpr int QPZ_OFF = QP_OFF + PAIRS * QP_PAIR_BYTES;
    // (8-bit, two pairs: they reach into the values' places, whose last SHORT_BLOCKS blocks the short rounds fill then)
    static constexpr int V_SHORT = BITS == 8 && PAIRS == 2 ? (AREA_BLOCKS - SHORT_BLOCKS) * K_BLOCK_BYTES : 0;
    static_assert(BITS != 8 || M == 1 || QP_OFF + QP_BYTES <= V_OFF + V_SHORT, "the query operands fit between the short rounds' keys and values");
    static constexpr int LDS_BYTES = (BITS == 8 || M == 1) ? V_OFF + AREA_BLOCKS * K_BLOCK_BYTES : QP_OFF + QP_BYTES;
    // one row: the merge of two waves, [group][lane < 32][4 rows] of 16 bytes, lies over the query operands,
    // which nobody reads after the last scores
    static constexpr int X_OFF = Q_OFF;
    static_assert(LDS_BYTES <= 160 * 1024, "LDS of a CU");
    static_assert(M * 512 <= K_BLOCK_BYTES, "the scores fit over the keys");
    static_assert(4 * 32 * 64 <= QZ_OFF - Q_OFF, "the merge fits over the query operands");
    // the counters
    static constexpr int C_KEYS = 0;    // key loaders that have requested the first round's keys
    static constexpr int C_QUERY = 1;   // computing waves that have written a row's query operands (8 per row)
    static constexpr int C_SCORES = 2;  // ... written their scores (8 per round)
    static constexpr int C_BUILT = 3;   // ... built their probability operands (8 per round)
    static constexpr int C_DONE = 4;    // ... are through with the round's values (8 per round)
    static constexpr int C_LENGTH = 5;  // (not a counter: the context length or the position, for every wave)
    static constexpr int C_VREQ = 6;    // alternating rounds: value loaders that have requested a round's values (2 per round)
    static constexpr int C_QREAD = 7;   // computing waves that have a row's query operands in registers (several rows)
    static constexpr int C_KPART = 8;   // [3]: key loaders whose blocks 0-7 and scales | blocks 8-15 | block 16 have landed (2 per round)
    static constexpr int C_SLOT = 12;   // [5]: value loaders whose values of slot s have landed (2 per round)
    // (alternating rounds: C_KPART, C_SLOT [2]: rounds of key | value loader L that have landed.  A counter for both loaders would not
    // say which of two rounds on their way it was.)
    static constexpr int C_MERGE = 20;  // [4]: one row: wave 2g + 1 has written its sums for wave 2g | two pairs of rows: blocks
                                        // whose keys the two waves of scores w % 4 have in registers; then [4] as with one row
    static constexpr int C_NORM = 28;       // the step before the scores: computing waves that have written their sums of squares
    static constexpr int C_POSITION = 29;   // (not a counter: the first new token's position)
    static constexpr uint32_t SPIN_LIMIT = 1u << 20;
    static constexpr int THREADS_ = (LOADERS + WAVES) * 64;
    static_assert(2 * 1024 + M * 10 * DIM * 4 <= LDS_BYTES, "the new rows' workgroup fits");
};

template <int BITS, int M, bool PREP>
__device__ __forceinline__ void attention_partial_s_body(const PartialArgs &a, const PrepArgs *prep) {
    using W = KeysFirst<BITS, M>;
    constexpr int RB = W::RB_, RT = W::SB_TOKENS, RBK = W::ROUND_BLOCKS;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
    const int lane = threadIdx.x & 63;
    const int wave_all = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
    const int n = lane & 15, j = lane >> 4;
    const uint32_t split = blockIdx.x, kv = blockIdx.y, kvh = a.kv_heads;
    const bool loader = wave_all < W::LOADERS;
    const int wave = wave_all - W::LOADERS;          // computing waves: 0..7
    uint32_t *sync_lds = reinterpret_cast<uint32_t *>(lds_raw + W::SYNC_OFF);
    const uint32_t lds0 = uint32_t(reinterpret_cast<uintptr_t>(lds_raw));
    const uint32_t context_splits = PREP ? a.nsplits - 1 : a.nsplits;
    if constexpr (PREP) {
        if (split == context_splits) {
            new_rows<BITS, M>(a, *prep, lds_raw, W::LOADERS + W::WAVES, 0, M, 0, SAETTA_GQA_GROUP);
            return;
        }
    }

    // ---- query values: requested first (computing waves: thread = (k-step, lane) item of every row) ----
    auto load_query = [&](int r, float (&v)[8]) {
        const int step = wave, g = step >> 1, ab = step & 1;
        const size_t of_head = size_t(r) * a.heads + kv * 8 + (n & 7);
        const float *src = (PREP ? prep->q_and_gate + of_head * 2 * DIM : a.q + of_head * DIM) + 64 * g + 16 * j + 8 * ab;
        const float4 f0 = *reinterpret_cast<const float4 *>(src);
        const float4 f1 = *reinterpret_cast<const float4 *>(src + 4);
        v[0] = f0.x, v[1] = f0.y, v[2] = f0.z, v[3] = f0.w, v[4] = f1.x, v[5] = f1.y, v[6] = f1.z, v[7] = f1.w;
    };
    // (several rows: per pair of rows, the row that the lane's column of the pair's tile belongs to.  The
    // loader waves leave the registers as they are: a value set for them would have to be merged with the
    // loaded one, and that copy would wait for the load in front of the barrier, where the loader waves
    // stand until every wave has arrived.)
    float qv[W::PAIRS][8];
    if (!loader) {
#pragma unroll
        for (int p = 0; p < W::PAIRS; p++) load_query(M == 1 ? 0 : min(2 * p + (n >> 3), M - 1), qv[p]);
    }
    float norm_w[8];
    if constexpr (PREP) {
        if (!loader) {
            const float4 *src = reinterpret_cast<const float4 *>(prep->q_norm + 64 * (wave >> 1) + 16 * j + 8 * (wave & 1));
            const float4 f0 = src[0], f1 = src[1];
            norm_w[0] = f0.x, norm_w[1] = f0.y, norm_w[2] = f0.z, norm_w[3] = f0.w, norm_w[4] = f1.x, norm_w[5] = f1.y, norm_w[6] = f1.z, norm_w[7] = f1.w;
        }
    }

    // ---- the context and this workgroup's share of it -----------------------------
    // One wave of the workgroup reads the token's parameters and hands them on through LDS.  The
    // counters start at zero behind the same barrier, the only s_barrier of the kernel, before
    // anybody requests anything of the cache.
    // (the context length of a decode step | the position of the first of a verify step's rows: one scalar load)
    static_assert(offsetof(saetta_token_params, position) == 4 && offsetof(saetta_token_params, kv_len) == 8, "dwords 1 and 2");
    if constexpr (PREP) {
        if (threadIdx.x < 32) {
            const uint32_t position = reinterpret_cast<const volatile uint32_t *>(a.tp)[1], kv_len = reinterpret_cast<const volatile uint32_t *>(a.tp)[2];
            sync_lds[threadIdx.x] = threadIdx.x == W::C_LENGTH ? tokens_before(a, position, kv_len) : threadIdx.x == W::C_POSITION ? position : 0u;
        }
    } else {
        if (threadIdx.x < 32) sync_lds[threadIdx.x] = threadIdx.x == W::C_LENGTH ? reinterpret_cast<const uint32_t *>(a.tp)[a.decode_len ? 2 : 1] : 0u;
    }
    __syncthreads();
    const uint32_t tp_first = __builtin_amdgcn_readfirstlane(sync_lds[W::C_LENGTH]);
    // tokens row r sees; the last row's are the launch's
    auto len_of = [&](int r) -> uint32_t { return min<uint32_t>(PREP || a.decode_len ? tp_first : tp_first + uint32_t(r) + 1, a.capacity); };
    const uint32_t max_len = len_of(M - 1);
    const uint32_t nblocks = (max_len + BLOCK - 1) / BLOCK;
    uint32_t blk_begin, blk_end;
    if (nblocks <= context_splits) {
        blk_begin = split;
        blk_end = split + 1;
        if (split >= nblocks) return;
    } else {
        blk_begin = split * nblocks / context_splits;
        blk_end = (split + 1) * nblocks / context_splits;
    }
    const uint32_t limit = min(max_len, blk_end * BLOCK);  // tokens of this share end here
    const uint32_t last_tok = limit - 1;                   // rows past it are never read: loads are clamped to it
    const uint32_t range = blk_end - blk_begin;
    // rounds of equal size (the last may be shorter), none longer than 17 blocks
    // (one row and two: one round of up to 17 blocks, or rounds of up to 8; three and four rows: of up to 12)
    constexpr uint32_t LONG_ROUND = W::ALTERNATE ? W::ALT_BLOCKS : W::SHORT_BLOCKS;
    const uint32_t n_rounds = range > uint32_t(RBK) ? (range + LONG_ROUND - 1) / LONG_ROUND : 1;
    const bool alt = W::ALTERNATE && n_rounds > 1;  // rounds in alternate halves of LDS
    const uint32_t per_round = (range + n_rounds - 1) / n_rounds;
    const uint32_t v_off = W::V_OFF + (M > 1 && n_rounds > 1 ? uint32_t(W::V_SHORT) : 0u);  // where the rounds' values lie
    auto blocks_of = [&](uint32_t round) { return min(range - round * per_round, per_round); };
    // The rounds in the order in which the splits take them: four in a row start a quarter of the share apart.  Started all at
    // the front they read addresses one share apart at every moment, and shares of nearly a power of two then meet in the
    // same memory channels: 40.5 us per layer at 131000 tokens (8-bit, one row) against 34.2 so, where 128000 take 32.5
    // and 33.0.  (Fewer rounds than 8: nothing to gain, and 60000 tokens took 21.8 us instead of 21.3.)
    const uint32_t first_round = n_rounds >= 8 ? (split & 3) * n_rounds / 4 : 0;
    auto place = [&](uint32_t round) { return round + first_round < n_rounds ? round + first_round : round + first_round - n_rounds; };

    auto dma = [&](uint32_t lds_addr, uint32_t voff, const void *src) {
        asm volatile("s_mov_b32 m0, %0\n"
                     "s_nop 0\n"
                     "global_load_lds_dwordx4 %1, %2\n"
                     :
                     : "s"(lds_addr), "v"(voff), "s"(src)
                     : "memory", "m0");
    };
    auto dma4 = [&](uint32_t lds_addr, uint32_t voff, const void *src) {
        asm volatile("s_mov_b32 m0, %0\n"
                     "s_nop 0\n"
                     "global_load_lds_dword %1, %2\n"
                     :
                     : "s"(lds_addr), "v"(voff), "s"(src)
                     : "memory", "m0");
    };
    // counters: raised by one lane after the wave's LDS writes (LDS takes a wave's instructions in
    // order); a waiting wave polls, a bounded number of times
    auto raise = [&](int c) {
        asm volatile("" ::: "memory");
        if (lane == 0) __hip_atomic_fetch_add(sync_lds + c, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        asm volatile("" ::: "memory");
    };
    auto peek = [&](int c) {
        asm volatile("" ::: "memory");
        const uint32_t v = __hip_atomic_load(sync_lds + c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        asm volatile("" ::: "memory");
        return uint32_t(__builtin_amdgcn_readfirstlane(v));
    };
    // A wait that runs out must not pass for a result: the wave notes which counter it was, goes on to its
    // end like any wave, and there (`leave`) leaves a code in the device's status word and l = NaN in the
    // workgroup's partials (wait_gave_up, out of line: it never runs); the wave that stores the maxima and
    // sums writes l = NaN itself if it has given up.  (The polling loop is kept rolled up: there are some
    // twenty waits in the kernel, and its code has to come through the instruction cache at every launch.)
    uint32_t lost = 0;
    auto await = [&](int c, uint32_t want) {
        asm volatile("" ::: "memory");
        uint32_t left = W::SPIN_LIMIT;
#pragma nounroll
        do {
            const uint32_t v = __hip_atomic_load(sync_lds + c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            if (__builtin_amdgcn_readfirstlane(v) >= want) break;
            __builtin_amdgcn_s_sleep(1);
        } while (--left);
        if (__builtin_expect(left == 0, 0)) lost = 0x100u + uint32_t(c);
        asm volatile("" ::: "memory");
    };
    auto leave = [&]() {
        if (__builtin_expect(lost != 0, 0)) wait_gave_up(a.status, a.part_ml, lost, M, a.nsplits, split, a.heads, kv);
    };
    // l of a partial as the writer of the maxima and sums stores it
    auto marked = [&](float l) { return lost ? __builtin_nanf("") : l; };

    if (loader && wave_all < W::K_LOADERS) {
        // ---- a key-loader wave: scales and biases of tokens 128 L .. 128 L + 127, keys of blocks L, L + 2, ...;
        // loader 0 then block 16 with its scales and biases ----
        const uint32_t L = uint32_t(wave_all);
        const void *sb_src[4] = {a.kscales, a.kbiases, a.vscales, a.vbiases};
        if constexpr (W::ALTERNATE) if (alt) {
            // ---- rounds of up to 8 blocks in alternate halves of LDS: loader L takes the rounds L, L + 2, ... whole, so
            // that two rounds' keys can be on their way at once.  A round goes out when the values of the round before
            // have been requested (the stream keeps the order keys, values, keys, ...) and when the round before last,
            // which lay in the same half, has been used up: its scales are read until every wave has built its operands,
            // its keys until every wave has its scores. ----
            for (uint32_t round = L; round < n_rounds; round += 2) {
                const uint32_t base = (blk_begin + place(round) * per_round) * BLOCK, nb = blocks_of(place(round));
                const uint32_t half = L * W::ALT_BLOCKS;  // the blocks of LDS this round goes to start here
                if (round > 1) await(W::C_BUILT, W::WAVES * (round - 1));
                if (round > 0) await(W::C_VREQ, round);
#pragma unroll
                for (int h = 0; h < W::ALT_BLOCKS / 4; h++) {
                    const uint32_t voff = (min(base + 64 * h + lane, last_tok) * kvh + kv) * 8;
#pragma unroll
                    for (int arr = 0; arr < 4; arr++) {
#pragma unroll
                        for (int pl = 0; pl < 2; pl++) dma4(lds0 + W::SB_OFF + arr * W::SB_ARRAY + (pl * RT + BLOCK * half + 64 * h) * 4, voff + 4 * pl, sb_src[arr]);
                    }
                }
#pragma unroll
                for (int r = 0; r < W::ALT_BLOCKS; r++) {
                    if (uint32_t(r) < nb) {
                        const uint32_t tok = min(base + BLOCK * r + (lane >> 2), last_tok);
                        const uint32_t voff = (tok * kvh + kv) * RB + (lane & 3) * 16;
#pragma unroll
                        for (int i = 0; i < W::PER_BLOCK; i++) dma(lds0 + W::K_OFF + (half + r) * W::K_BLOCK_BYTES + i * 1024, voff + 64 * i, a.kdata);
                    }
                }
                raise(W::C_KEYS);
                __builtin_amdgcn_s_waitcnt(vmcnt_only(0));
                raise(W::C_KPART + int(L));
            }
            leave();
            return;
        }
        // (one row: more than one round is taken above)
        for (uint32_t round = 0; round < (M == 1 ? 1u : n_rounds); round++) {
            const uint32_t at = M == 1 ? 0 : place(round), base = (blk_begin + at * per_round) * BLOCK, nb = blocks_of(at);
            // the round before: its scales are read until every wave has built its operands, its keys until every wave has its scores
            if (round > 0) await(W::C_BUILT, W::WAVES * round);
#pragma unroll
            for (int h = 0; h < 2; h++) {
                // a dword per lane and load: the token's four f16 of an array go to two planes
                const uint32_t voff = (min(base + 128 * L + 64 * h + lane, last_tok) * kvh + kv) * 8;
#pragma unroll
                for (int arr = 0; arr < 4; arr++) {
#pragma unroll
                    for (int pl = 0; pl < 2; pl++) dma4(lds0 + W::SB_OFF + arr * W::SB_ARRAY + (pl * RT + 128 * L + 64 * h) * 4, voff + 4 * pl, sb_src[arr]);
                }
            }
            auto request_block = [&](uint32_t blk) {
                // lane -> (token lane / 4, 16 bytes lane % 4 of the token's 64-byte piece i): four
                // neighbouring lanes read 64 contiguous bytes
                const uint32_t tok = min(base + BLOCK * blk + (lane >> 2), last_tok);
                const uint32_t voff = (tok * kvh + kv) * RB + (lane & 3) * 16;
#pragma unroll
                for (int i = 0; i < W::PER_BLOCK; i++) dma(lds0 + W::K_OFF + blk * W::K_BLOCK_BYTES + i * 1024, voff + 64 * i, a.kdata);
            };
#pragma unroll
            for (int r = 0; r < 8; r++) {
                if (L + 2 * r < nb) request_block(L + 2 * r);
            }
            const bool extra = nb == uint32_t(RBK) && L == 0;
            if (extra) {
                if (lane < BLOCK) {
                    const uint32_t voff = (min(base + 256 + lane, last_tok) * kvh + kv) * 8;
#pragma unroll
                    for (int arr = 0; arr < 4; arr++) {
#pragma unroll
                        for (int pl = 0; pl < 2; pl++) dma4(lds0 + W::SB_OFF + arr * W::SB_ARRAY + (pl * RT + 256) * 4, voff + 4 * pl, sb_src[arr]);
                    }
                }
                request_block(16);
            }
            if (round == 0) raise(W::C_KEYS);
            // loads return in order (a round of less than 16 blocks: all at once)
            if (extra) {
                __builtin_amdgcn_s_waitcnt(vmcnt_only(W::K_LOADS / 2 + W::X_LOADS));
                raise(W::C_KPART + 0);
                __builtin_amdgcn_s_waitcnt(vmcnt_only(W::X_LOADS));
                raise(W::C_KPART + 1);
            } else if (nb >= 16) {
                __builtin_amdgcn_s_waitcnt(vmcnt_only(W::K_LOADS / 2));
                raise(W::C_KPART + 0);
                __builtin_amdgcn_s_waitcnt(vmcnt_only(0));
                raise(W::C_KPART + 1);
            } else {
                __builtin_amdgcn_s_waitcnt(vmcnt_only(0));
                raise(W::C_KPART + 0);
                raise(W::C_KPART + 1);
            }
            __builtin_amdgcn_s_waitcnt(vmcnt_only(0));
            raise(W::C_KPART + 2);
        }
        leave();
        return;
    }
    if (loader) {
        // ---- a value-loader wave: blocks L, L + 2, ... of every round, two of them in each 64-token slot;
        // loader 0 then block 16 (slot 4) ----
        const uint32_t L = uint32_t(wave_all) - W::K_LOADERS;
        if constexpr (W::ALTERNATE) if (alt) {
            // ---- alternate halves: loader L takes the values of the rounds L, L + 2, ... whole, each behind its round's
            // keys in the stream, into the half that the round before last has left (every wave through with its values) ----
            for (uint32_t round = L; round < n_rounds; round += 2) {
                const uint32_t base = (blk_begin + place(round) * per_round) * BLOCK, nb = blocks_of(place(round));
                const uint32_t half = L * W::ALT_BLOCKS;
                await(W::C_KEYS, round + 1);
                if (round > 1) await(W::C_DONE, W::WAVES * (round - 1));
#pragma unroll
                for (int r = 0; r < W::ALT_BLOCKS; r++) {
                    if (uint32_t(r) < nb) {
#pragma unroll
                        for (int i = 0; i < W::PER_BLOCK; i++) {
                            const uint32_t t = BLOCK * r + W::V_GROUP_TOKENS * i + lane / W::PIECES;  // token of the round
                            const uint32_t piece = (lane % W::PIECES + W::PIECES - ((t >> 3) & 3) * (W::PIECES / 4)) % W::PIECES;
                            dma(lds0 + W::V_OFF + (W::PER_BLOCK * (half + r) + i) * 1024, (min(base + t, last_tok) * kvh + kv) * RB + piece * 16, a.vdata);
                        }
                    }
                }
                raise(W::C_VREQ);
                __builtin_amdgcn_s_waitcnt(vmcnt_only(0));
                raise(W::C_SLOT + int(L));
            }
            leave();
            return;
        }
        for (uint32_t round = 0; round < (M == 1 ? 1u : n_rounds); round++) {
            const uint32_t at = M == 1 ? 0 : place(round), base = (blk_begin + at * per_round) * BLOCK, nb = blocks_of(at);
            // the keys of the first round have been requested | every wave is through with the values before
            if (round == 0) {
                await(W::C_KEYS, W::K_LOADERS);
            } else {
                await(W::C_DONE, W::WAVES * round);
            }
            auto request_block = [&](uint32_t blk) {
#pragma unroll
                for (int i = 0; i < W::PER_BLOCK; i++) {
                    // lane -> (token lane / PIECES of the instruction's group, the piece that goes to place lane % PIECES
                    // of the row, which is rotated by (token / 8) % 4 quarters: the same for the group's tokens)
                    const uint32_t t = BLOCK * blk + W::V_GROUP_TOKENS * i + lane / W::PIECES;  // token of the round
                    const uint32_t piece = (lane % W::PIECES + W::PIECES - ((t >> 3) & 3) * (W::PIECES / 4)) % W::PIECES;
                    dma(lds0 + v_off + (W::PER_BLOCK * blk + i) * 1024, (min(base + t, last_tok) * kvh + kv) * RB + piece * 16, a.vdata);
                }
            };
#pragma unroll
            for (int r = 0; r < 8; r++) {
                if (L + 2 * r < nb) request_block(L + 2 * r);
            }
            const bool extra = nb == uint32_t(RBK) && L == 0;
            if (extra) request_block(16);
            // loads return in order (a round of less than 16 blocks: all at once)
            if (extra) {
                __builtin_amdgcn_s_waitcnt(vmcnt_only(W::V_LOADS * 3 / 4 + W::PER_BLOCK));
                raise(W::C_SLOT + 0);
                __builtin_amdgcn_s_waitcnt(vmcnt_only(W::V_LOADS * 2 / 4 + W::PER_BLOCK));
                raise(W::C_SLOT + 1);
                __builtin_amdgcn_s_waitcnt(vmcnt_only(W::V_LOADS * 1 / 4 + W::PER_BLOCK));
                raise(W::C_SLOT + 2);
                __builtin_amdgcn_s_waitcnt(vmcnt_only(W::PER_BLOCK));
                raise(W::C_SLOT + 3);
            } else if (nb >= 16) {
                __builtin_amdgcn_s_waitcnt(vmcnt_only(W::V_LOADS * 3 / 4));
                raise(W::C_SLOT + 0);
                __builtin_amdgcn_s_waitcnt(vmcnt_only(W::V_LOADS * 2 / 4));
                raise(W::C_SLOT + 1);
                __builtin_amdgcn_s_waitcnt(vmcnt_only(W::V_LOADS * 1 / 4));
                raise(W::C_SLOT + 2);
                __builtin_amdgcn_s_waitcnt(vmcnt_only(0));
                raise(W::C_SLOT + 3);
            } else {
                __builtin_amdgcn_s_waitcnt(vmcnt_only(0));
                raise(W::C_SLOT + 0);
                raise(W::C_SLOT + 1);
                raise(W::C_SLOT + 2);
                raise(W::C_SLOT + 3);
            }
            __builtin_amdgcn_s_waitcnt(vmcnt_only(0));
            raise(W::C_SLOT + 4);
        }
        leave();
        return;
    }

    // ---- computing waves ------------------------------------------------------------------------
    half8 *q_lds = reinterpret_cast<half8 *>(lds_raw + W::Q_OFF);
    _Float16 *qz_lds = reinterpret_cast<_Float16 *>(lds_raw + W::QZ_OFF);
    const uint32_t *sb_lds = reinterpret_cast<const uint32_t *>(lds_raw + W::SB_OFF);
    float *bmax_lds = reinterpret_cast<float *>(lds_raw + W::BMAX_OFF);
    float *bsum_lds = reinterpret_cast<float *>(lds_raw + W::BSUM_OFF);
    float *zs_lds = reinterpret_cast<float *>(lds_raw + W::ZS_OFF);
    if constexpr (PREP) {
        // The norm and the rotation of the query rows, while the first keys are on their way: wave w has k-step w of every
        // row, the waves 0 and 1 the dims 0-63 that are rotated (lane 16 row + i of them computes angle i of the wave's 16).
        float sine = 0.0f, cosine = 0.0f;
#pragma unroll
        for (int p = 0; p < W::PAIRS; p++) {
            float sum = 0.0f;
#pragma unroll
            for (int e = 0; e < 8; e++) sum += qv[p][e] * qv[p][e];
            sum = across_rows<16, 64>(sum, SumOp());
            if (j == 0) zs_lds[(wave * W::PAIRS + p) * 16 + n] = sum;
        }
        raise(W::C_NORM);
        if (wave < 2) rope_angle(sync_lds[W::C_POSITION] + min(j, M - 1), rope_frequency(16 * (n >> 3) + 8 * wave + (n & 7), 32, prep->p.log2_theta), sine, cosine);
        await(W::C_NORM, W::WAVES);
#pragma unroll
        for (int p = 0; p < W::PAIRS; p++) {
            float total = 0.0f;
#pragma unroll
            for (int w = 0; w < W::WAVES; w++) total += zs_lds[(w * W::PAIRS + p) * 16 + n];
            const float scale = query_scale(total, prep->p.eps);
#pragma unroll
            for (int e = 0; e < 8; e++) qv[p][e] *= scale * norm_w[e];
            if (wave < 2) {
                const int row = M == 1 ? 0 : min(2 * p + (n >> 3), M - 1);
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    const float s = __shfl(sine, 16 * row + 8 * (j & 1) + e), c = __shfl(cosine, 16 * row + 8 * (j & 1) + e);
                    const float x = qv[p][e], other = half_swap(x, j < 2);
                    qv[p][e] = j < 2 ? rope_first(x, other, s, c) : rope_second(other, x, s, c);
                }
            }
        }
    }
    // the scores of block b, row r: [head][token] f32 over the block's keys
    auto s_block = [&](int b, int r) { return reinterpret_cast<float *>(lds_raw + W::K_OFF + b * W::K_BLOCK_BYTES + r * 512); };

    // the value codes of k-step ks for group g: the lane's dword of tokens 32 ks + 8j .. + 7
    auto read_values = [&](int ks, int g, ValRegs<BITS> &vreg) {
        const int jj = ks == 8 ? (j & 1) : j;
        // (tokens 8 jj .. 8 jj + 7 of a k-step: their rows are rotated by jj quarters)
        const unsigned char *vb = lds_raw + v_off + 8 * jj * RB + ((val_lane_offset<BITS>(g, n) + jj * W::V_ROT) & (RB - 1));
#pragma unroll
        for (int e = 0; e < 8; e++) vreg.w[e] = *reinterpret_cast<const uint32_t *>(vb + (32 * ks + e) * RB);
    };
    // a row's maximum per head over the round's blocks
    auto round_max = [&](int r, float start) {
        const float *bmx = bmax_lds + r * W::BROW + (n & 7) * W::BSTRIDE;
        float v = start;
        if constexpr (M == 1) {
#pragma unroll
            for (int i = 0; i < W::BSINGLE / 4; i++) {
                const floatx4 w = reinterpret_cast<const floatx4 *>(bmx)[i];
                v = fmaxf(v, fmaxf(fmaxf(w[0], w[1]), fmaxf(w[2], w[3])));
            }
        } else {
#pragma unroll
            for (int i = 0; i < RBK; i++) v = fmaxf(v, bmx[i]);
        }
        return v;
    };
    // a row's sum of P of head n & 7 over the round's blocks, relative to the maximum nm: lane group j adds blocks j, j + 4, ...
    auto round_sum = [&](int r, float nm) {
        float sum = 0.0f;
        if constexpr (M == 1) {
            // lane group j adds blocks 5j .. 5j + 4
#pragma unroll
            for (int i = 0; i < W::BSINGLE / 4; i++) {
                const int b = (W::BSINGLE / 4) * j + i;
                sum += bsum_lds[r * W::BROW + (n & 7) * W::BSTRIDE + b] * __builtin_amdgcn_exp2f(bmax_lds[r * W::BROW + (n & 7) * W::BSTRIDE + b] - nm);
            }
            return across_rows<16, 64>(sum, SumOp());
        }
#pragma unroll
        for (int i = 0; i < (RBK + 3) / 4; i++) {
            const int b = j + 4 * i;
            if (b < RBK) sum += bsum_lds[r * W::BROW + (n & 7) * W::BSTRIDE + b] * __builtin_amdgcn_exp2f(bmax_lds[r * W::BROW + (n & 7) * W::BSTRIDE + b] - nm);  // (a block that is not there: sum 0)
        }
        return across_rows<16, 64>(sum, SumOp());
    };
    constexpr float unscale = code_up<BITS>() / P_UP;
    const int g = wave >> 1, b2 = wave & 1;  // O += P V: the wave's group and which k-steps of a slot

    if constexpr (M > 1) {
        // ---- several rows ------------------------------------------------------------------------
        // Two rows share a tile: its 16 columns are (row of the pair, head), and the hi and the lo parts of
        // an operand go through two MFMAs into one accumulator, so that every lane of a result holds a
        // whole score (or output) of its own column.  Three rows: the second pair's upper columns repeat
        // row 2 and are not written out.
        // Scores: with one pair every wave takes its blocks (wave, wave + 8; wave 0 also 16); with two
        // pairs waves 0-3 take the first and waves 4-7 the second, blocks w % 4 + 4 i.  The pair's query
        // operands stay in registers: they go through the one place in LDS, the hi parts and then the lo
        // parts of a pair, while the first keys are on their way.
        // O += P V: as with one row, waves 2g and 2g + 1 share group g and take alternate k-steps, for
        // every pair, the byte permutes of a value operand serving both pairs.
        constexpr int PAIRS = W::PAIRS, WT = W::WAVES / PAIRS;
        const int at = wave / WT, wt = wave % WT;
        const int col_row = n >> 3;  // the row of the pair that this lane's column belongs to
        auto row_of = [&](int pair, int half) { return min(2 * pair + half, M - 1); };
        if (range > uint32_t(RBK)) {
            // ---- a share of more than one round (a context of more than 17 blocks per split) ----------
            // Rounds of up to SHORT_BLOCKS blocks, in the first blocks of the keys' and the values' places.  What
            // a round leaves behind, per column: the maximum so far, the sums so far relative to it (O in
            // registers, l with wave 0), both brought to the new maximum before the next round's values are
            // added.  The query operands of every pair wait in LDS (the blocks that short rounds never fill) and
            // are read again for every round's scores, so that they hold no registers while the values are taken.
            constexpr int SB = W::SHORT_BLOCKS, A_SHORT = SB / WT, S_SLOTS = SB / 4;
            half8 *qp_lds = reinterpret_cast<half8 *>(lds_raw + W::QP_OFF);
            _Float16 *qpz_lds = reinterpret_cast<_Float16 *>(lds_raw + W::QPZ_OFF);
            {
                const float qmul = a.scale * 1.4426950408889634f * Q_UP;
#pragma unroll
                for (int pair = 0; pair < PAIRS; pair++) {
                    // this thread's item: k-step `wave`, lane `lane`: column n = (row n / 8 of the pair, head n % 8)
                    half8 hi, lo;
                    float sum = 0.0f;
#pragma unroll
                    for (int e = 0; e < 8; e++) {
                        _Float16 h, lw;
                        split_hi_lo(qv[pair][key_slot_dim<BITS>(e)] * qmul, h, lw);
                        hi[e] = h, lo[e] = lw;
                        sum += (float)h + (float)lw;
                    }
                    qp_lds[((pair * 2 + 0) * 8 + wave) * 64 + lane] = hi;
                    qp_lds[((pair * 2 + 1) * 8 + wave) * 64 + lane] = lo;
                    _Float16 h, lw;
                    split_hi_lo(sum * (1.0f / Q_UP), h, lw);
                    qpz_lds[((pair * 2 + 0) * 64 + lane) * 8 + wave] = h;
                    qpz_lds[((pair * 2 + 1) * 64 + lane) * 8 + wave] = lw;
                }
                // blocks that a short round never has: maximum "none", sum 0 (the table of this wave's pair, by its first wave)
                if (wt == 0 && j == 0) {
                    const int my_row = row_of(at, col_row);
#pragma unroll
                    for (int b = SB; b < RBK; b++) bmax_lds[my_row * W::BROW + (n & 7) * W::BSTRIDE + b] = NO_SCORE, bsum_lds[my_row * W::BROW + (n & 7) * W::BSTRIDE + b] = 0.0f;
                }
            }
            raise(W::C_QUERY);

            float m_run[PAIRS], l_run[PAIRS], zacc[PAIRS];
            floatx4 acc[PAIRS][4];  // [pair][tile of 16 dims 4n' + e]: rows 4j .. 4j+3 (columns of the pair), column n'
#pragma unroll
            for (int p = 0; p < PAIRS; p++) {
                m_run[p] = NO_SCORE, l_run[p] = 0.0f, zacc[p] = 0.0f;
#pragma unroll
                for (int e = 0; e < 4; e++) acc[p][e] = floatx4{0, 0, 0, 0};
            }
            uint32_t taken = 0;  // blocks whose scores this wave has written (two pairs: the handshake over a block's keys counts them)
            await(W::C_QUERY, W::WAVES);
#pragma unroll 1
            for (uint32_t round = 0; round < n_rounds; round++) {
                const uint32_t base = (blk_begin + place(round) * per_round) * BLOCK, nb = blocks_of(place(round));
                const uint32_t round_limit = min(limit, base + nb * BLOCK);  // tokens of this round end here
                const uint32_t live_blocks = (nb + 1) & ~1u;  // k-steps are two blocks: the blocks of the k-steps that have tokens

                // ---- phase A: the scores of this wave's blocks for its pair of rows ----
                {
                    const int my_row = row_of(at, col_row);
                    const uint32_t my_limit = min<uint32_t>(round_limit, len_of(my_row));
#pragma unroll 1
                    for (int i = 0; i < A_SHORT; i++) {
                        const int blk = wt + WT * i;
                        if (uint32_t(blk) >= live_blocks) {
                            // (no scores to take, and no operands will be made of this block; the table still holds the
                            // round before's entries until every wave has built its operands from them)
                            if (round > 0) await(W::C_BUILT, W::WAVES * round);
                            if (j == 0) bmax_lds[my_row * W::BROW + (n & 7) * W::BSTRIDE + blk] = NO_SCORE, bsum_lds[my_row * W::BROW + (n & 7) * W::BSTRIDE + blk] = 0.0f;
                            continue;
                        }
                        await(W::C_KPART + 0, W::K_LOADERS * (round + 1));  // the round's keys and scales are in LDS
                        const unsigned char *kb = lds_raw + W::K_OFF + blk * W::K_BLOCK_BYTES;
                        KeyRegs<BITS> kreg[4];
#pragma unroll
                        for (int gg = 0; gg < 4; gg++) {
                            if constexpr (BITS == 8) {
                                const u32x4 v = *reinterpret_cast<const u32x4 *>(kb + gg * 1024 + n * 64 + j * 16);
                                kreg[gg].w[0] = v.x, kreg[gg].w[1] = v.y, kreg[gg].w[2] = v.z, kreg[gg].w[3] = v.w;
                            } else {
                                const u32x2 v = *reinterpret_cast<const u32x2 *>(kb + (gg >> 1) * 1024 + n * 64 + (gg & 1) * 32 + j * 8);
                                kreg[gg].w[0] = v.x, kreg[gg].w[1] = v.y;
                            }
                        }
                        const int tok0 = BLOCK * blk + 4 * j;  // this lane's 4 tokens of the round in C layout
                        const uint32_t *sb_w = sb_lds + BLOCK * blk;
                        const u32x2 zr = {sb_w[W::SB_ARRAY / 4 + n], sb_w[W::SB_ARRAY / 4 + RT + n]};
                        const half8 zop = as_half8(perm(0, zr.x, 0x01000100u), perm(0, zr.x, 0x03020302u), perm(0, zr.y, 0x01000100u), perm(0, zr.y, 0x03020302u));
                        const u32x4 s01 = *reinterpret_cast<const u32x4 *>(sb_w + 4 * j);
                        const u32x4 s23 = *reinterpret_cast<const u32x4 *>(sb_w + RT + 4 * j);
                        const uint32_t sw[8] = {s01.x, s23.x, s01.y, s23.y, s01.z, s23.z, s01.w, s23.w};
                        floatx4 sc = {0, 0, 0, 0}, rr[4] = {{0, 0, 0, 0}, {0, 0, 0, 0}, {0, 0, 0, 0}, {0, 0, 0, 0}};
                        sc = __builtin_amdgcn_mfma_f32_16x16x32_f16(zop, *reinterpret_cast<const half8 *>(qpz_lds + ((at * 2 + 0) * 64 + lane) * 8), sc, 0, 0, 0);
                        sc = __builtin_amdgcn_mfma_f32_16x16x32_f16(zop, *reinterpret_cast<const half8 *>(qpz_lds + ((at * 2 + 1) * 64 + lane) * 8), sc, 0, 0, 0);
                        // the hi parts of the pair's query operands, then the lo parts: one set in registers at a time
                        // (the accumulators of the rounds so far are held as well), the key operands made once for each
#pragma unroll
                        for (int part = 0; part < 2; part++) {
                            half8 q_part[8];
#pragma unroll
                            for (int k = 0; k < 8; k++) q_part[k] = qp_lds[((at * 2 + part) * 8 + k) * 64 + lane];
#pragma unroll
                            for (int gg = 0; gg < 4; gg++) {
#pragma unroll
                                for (int ab = 0; ab < 2; ab++) {
                                    rr[gg] = __builtin_amdgcn_mfma_f32_16x16x32_f16(key_operand<BITS>(kreg[gg], ab), q_part[gg * 2 + ab], rr[gg], 0, 0, 0);
                                }
                            }
                            asm volatile("" ::: "memory");  // (the lo parts are not to be fetched while the hi parts are held)
                        }
                        constexpr float C1 = code_up<BITS>() / Q_UP;
#pragma unroll
                        for (int tk = 0; tk < 4; tk++) {
                            float d = 0.0f;
#pragma unroll
                            for (int gg = 0; gg < 4; gg++) d += half_bits_to_float(sw[2 * tk + (gg >> 1)] >> (16 * (gg & 1))) * rr[gg][tk];
                            const float v = sc[tk] + d * C1;
                            sc[tk] = base + tok0 + tk < my_limit ? v : NO_SCORE;  // (also whatever a block past the round left in LDS)
                        }
                        // the block's softmax relative to its own maximum, per column
                        float cm = fmaxf(fmaxf(sc[0], sc[1]), fmaxf(sc[2], sc[3]));
                        cm = across_rows<16, 64>(cm, MaxOp());
                        float sum = 0.0f;
#pragma unroll
                        for (int tk = 0; tk < 4; tk++) {
                            sc[tk] = sc[tk] > 0.5f * NO_SCORE ? __builtin_amdgcn_exp2f(sc[tk] - cm) : 0.0f;
                            sum += sc[tk];
                        }
                        sum = across_rows<16, 64>(sum, SumOp());
                        if (j == 0) bmax_lds[my_row * W::BROW + (n & 7) * W::BSTRIDE + blk] = cm, bsum_lds[my_row * W::BROW + (n & 7) * W::BSTRIDE + blk] = sum;
                        // the scores go over the block's own keys: when this wave has them in registers, and with
                        // two pairs the other pair's wave of the same blocks, which takes them in the same order
                        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                        taken++;
                        if constexpr (PAIRS > 1) {
                            raise(W::C_MERGE + wt);
                            await(W::C_MERGE + wt, PAIRS * taken);
                        }
                        *reinterpret_cast<floatx4 *>(s_block(blk, my_row) + (n & 7) * BLOCK + 4 * j) = sc;
                    }
                }
                raise(W::C_SCORES);
                await(W::C_SCORES, W::WAVES * (round + 1));

                // ---- the columns' maxima; what was summed so far brought to them; the probability operands ----
                float al[PAIRS];
#pragma unroll
                for (int p = 0; p < PAIRS; p++) {
                    const float nm = round_max(row_of(p, col_row), m_run[p]);
                    al[p] = __builtin_amdgcn_exp2f(m_run[p] - nm);  // (nothing summed so far: whatever it is, it scales zeros)
                    m_run[p] = nm;
                    zacc[p] *= al[p];
                    if (wave == 0) l_run[p] = l_run[p] * al[p] + round_sum(row_of(p, col_row), nm);
                }
                half8 p_hi[PAIRS][S_SLOTS], p_lo[PAIRS][S_SLOTS];
#pragma unroll
                for (int sl = 0; sl < S_SLOTS; sl++) {
                    if (uint32_t(2 * (2 * sl + b2)) >= nb) {  // the k-step has no tokens
#pragma unroll
                        for (int p = 0; p < PAIRS; p++) p_hi[p][sl] = p_lo[p][sl] = half8{0, 0, 0, 0, 0, 0, 0, 0};
                        continue;
                    }
                    const int ks = 2 * sl + b2;  // tokens 32 ks ..: blocks 2 ks and 2 ks + 1
                    const int blk = 2 * ks + (j >> 1);
                    const int sh = 16 * (g & 1);
                    const uint32_t *vsp = sb_lds + 2 * (W::SB_ARRAY / 4) + (g >> 1) * RT + 32 * ks + 8 * j;
                    const u32x4 sv0 = *reinterpret_cast<const u32x4 *>(vsp), sv1 = *reinterpret_cast<const u32x4 *>(vsp + 4);
                    const u32x4 zv0 = *reinterpret_cast<const u32x4 *>(vsp + W::SB_ARRAY / 4), zv1 = *reinterpret_cast<const u32x4 *>(vsp + W::SB_ARRAY / 4 + 4);
                    const uint32_t sw[8] = {sv0.x, sv0.y, sv0.z, sv0.w, sv1.x, sv1.y, sv1.z, sv1.w};
                    const uint32_t zw[8] = {zv0.x, zv0.y, zv0.z, zv0.w, zv1.x, zv1.y, zv1.z, zv1.w};
                    float vscale[8], vbias[8];
#pragma unroll
                    for (int e = 0; e < 8; e++) vscale[e] = half_bits_to_float(sw[e] >> sh), vbias[e] = half_bits_to_float(zw[e] >> sh);
#pragma unroll
                    for (int p = 0; p < PAIRS; p++) {
                        const int r = row_of(p, col_row);
                        const float *sp = s_block(blk, r) + (n & 7) * BLOCK + 8 * (j & 1);
                        const floatx4 pt0 = *reinterpret_cast<const floatx4 *>(sp), pt1 = *reinterpret_cast<const floatx4 *>(sp + 4);
                        const float pt[8] = {pt0[0], pt0[1], pt0[2], pt0[3], pt1[0], pt1[1], pt1[2], pt1[3]};
                        // 2^(block maximum - maximum so far) * P_UP (2^8, so that the lo part stays a normal f16)
                        const float f = __builtin_amdgcn_exp2f(bmax_lds[r * W::BROW + (n & 7) * W::BSTRIDE + blk] - m_run[p] + 8.0f);
                        float x[8], lo[8], zb = 0.0f;
#pragma unroll
                        for (int e = 0; e < 8; e++) {
                            zb += pt[e] * vbias[e];
                            x[e] = pt[e] * f * vscale[e];
                            lo[e] = x[e] - __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, x[e]) & 0xffffe000u);
                        }
                        zacc[p] += zb * f;
                        uint32_t o[8];
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            // round toward zero: exact truncation to the hi part
                            o[e] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(x[2 * e], x[2 * e + 1]));
                            o[4 + e] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(lo[2 * e], lo[2 * e + 1]));
                        }
                        asm volatile("" : "+v"(o[0]), "+v"(o[1]), "+v"(o[2]), "+v"(o[3]), "+v"(o[4]), "+v"(o[5]), "+v"(o[6]), "+v"(o[7]));
                        p_hi[p][sl] = as_half8(o[0], o[1], o[2], o[3]);
                        p_lo[p][sl] = as_half8(o[4], o[5], o[6], o[7]);
                    }
                }
                raise(W::C_BUILT);  // this wave is through with the round's scores, scales and biases

                // ---- phase C: O = O * 2^(old maximum - new) + P V ----
                if (round > 0) {
#pragma unroll
                    for (int p = 0; p < PAIRS; p++) {
                        // accumulator rows 4j + i are the pair's columns 4j + i: lane c (j = 0, n = c) holds column c's factor
                        floatx4 al4;
#pragma unroll
                        for (int i = 0; i < 4; i++) al4[i] = __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(4 * (4 * j + i), __builtin_bit_cast(int, al[p])));
#pragma unroll
                        for (int e = 0; e < 4; e++) acc[p][e] *= al4;
                    }
                }
#pragma unroll
                for (int sl = 0; sl < S_SLOTS; sl++) {
                    if (uint32_t(2 * (2 * sl + b2)) >= nb) continue;
                    await(W::C_SLOT + sl, W::V_LOADERS * (round + 1));  // value slot sl is in LDS
                    ValRegs<BITS> vreg;
                    read_values(2 * sl + b2, g, vreg);
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const half8 vop = val_operand<BITS>(vreg, e, n);
#pragma unroll
                        for (int p = 0; p < PAIRS; p++) {
                            acc[p][e] = __builtin_amdgcn_mfma_f32_16x16x32_f16(p_hi[p][sl], vop, acc[p][e], 0, 0, 0);
                            acc[p][e] = __builtin_amdgcn_mfma_f32_16x16x32_f16(p_lo[p][sl], vop, acc[p][e], 0, 0, 0);
                        }
                    }
                }
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the value codes are in registers
                raise(W::C_DONE);
            }

            // ---- epilogue: the two waves of a group add up, wave 2g writes the partials ----
#pragma unroll
            for (int p = 0; p < PAIRS; p++) {
                const float z = across_rows<16, 64>(zacc[p], SumOp());
                if (j == 0) zs_lds[(wave * PAIRS + p) * 16 + n] = z;
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            floatx4 mine[PAIRS][4];  // column 4j + i of the pair, dims 64 g + 4n .. + 3
#pragma unroll
            for (int p = 0; p < PAIRS; p++) {
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const float zb = zs_lds[(wave * PAIRS + p) * 16 + 4 * j + i] * (1.0f / P_UP);
#pragma unroll
                    for (int e = 0; e < 4; e++) mine[p][i][e] = acc[p][e][i] * unscale + zb;
                }
            }
            // (the merge lies over the keys, which hold the last round's scores until every wave has built its operands;
            // the key loaders request nothing after the last round)
            floatx4 *x_o = reinterpret_cast<floatx4 *>(lds_raw + W::K_OFF);  // [pair][group][lane][4 columns]
            static_assert(PAIRS * 4 * 64 * 4 * 16 <= W::SHORT_BLOCKS * W::K_BLOCK_BYTES || BITS == 4, "the merge stays clear of the query operands");
            await(W::C_BUILT, W::WAVES * n_rounds);
            if (b2 == 1) {
#pragma unroll
                for (int p = 0; p < PAIRS; p++) {
#pragma unroll
                    for (int i = 0; i < 4; i++) x_o[((p * 4 + g) * 64 + lane) * 4 + i] = mine[p][i];
                }
                raise(W::C_MERGE + 4 + g);
                leave();
                return;
            }
            if (wave == 0) {
#pragma unroll
                for (int p = 0; p < PAIRS; p++) {
                    const int r = 2 * p + col_row;
                    if (j == 0 && r < M) {
                        const size_t slot = (size_t(r) * a.nsplits + split) * a.heads + kv * 8 + (n & 7);
                        *reinterpret_cast<floatx2 *>(a.part_ml + 2 * slot) = floatx2{m_run[p], marked(l_run[p])};
                    }
                }
            }
            await(W::C_MERGE + 4 + g, 1);
#pragma unroll
            for (int p = 0; p < PAIRS; p++) {
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const int c = 4 * j + i, r = 2 * p + (c >> 3);
                    if (r < M) {
                        const size_t slot = (size_t(r) * a.nsplits + split) * a.heads + kv * 8 + (c & 7);
                        __builtin_nontemporal_store(mine[p][i] + x_o[((p * 4 + g) * 64 + lane) * 4 + i], reinterpret_cast<floatx4 *>(a.part_o + slot * DIM + 64 * g + 4 * n));
                    }
                }
            }
            leave();
            return;
        }
        const uint32_t base = blk_begin * BLOCK;
        const bool extra = range >= uint32_t(RBK);  // the round has block 16
        const uint32_t live_blocks = (range + 1) & ~1u;  // k-steps are two blocks: the blocks of the k-steps that have tokens

        half8 q_hi[8], q_lo[8], qz_reg[2];
        {
            const float qmul = a.scale * 1.4426950408889634f * Q_UP;
#pragma unroll
            for (int pass = 0; pass < 2 * PAIRS; pass++) {
                const int pair = pass >> 1, lo_part = pass & 1;
                // this thread's item: k-step `wave`, lane `lane`: column n = (row n / 8 of the pair, head n % 8)
                half8 op;
                float sum = 0.0f;
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    _Float16 h, lw;
                    split_hi_lo(qv[pair][key_slot_dim<BITS>(e)] * qmul, h, lw);
                    op[e] = lo_part ? lw : h;
                    sum += (float)h + (float)lw;
                }
                // the place is free when the readers of the pass before (the waves of its pair) have it in registers
                if (pass > 0) await(W::C_QREAD, WT * pass);
                q_lds[wave * 64 + lane] = op;
                if (!lo_part) {
                    // key bias term: slot `k-step` of this lane in the B operand of one more MFMA, as hi and lo halves
                    _Float16 h, lw;
                    split_hi_lo(sum * (1.0f / Q_UP), h, lw);
                    qz_lds[(0 * 64 + lane) * 8 + wave] = h;
                    qz_lds[(1 * 64 + lane) * 8 + wave] = lw;
                }
                raise(W::C_QUERY);
                if (pair == at) {
                    await(W::C_QUERY, W::WAVES * (pass + 1));
#pragma unroll
                    for (int i = 0; i < 8; i++) {
                        const half8 v = q_lds[i * 64 + lane];
                        if (lo_part) q_lo[i] = v; else q_hi[i] = v;
                    }
                    if (!lo_part) {
                        qz_reg[0] = *reinterpret_cast<const half8 *>(qz_lds + lane * 8);
                        qz_reg[1] = *reinterpret_cast<const half8 *>(qz_lds + (64 + lane) * 8);
                    }
                    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                    raise(W::C_QREAD);
                }
            }
        }

        // ---- phase A: the scores of this wave's blocks for its pair of rows ----
        {
            const int my_row = row_of(at, col_row);
            const uint32_t my_limit = min<uint32_t>(limit, len_of(my_row));
            constexpr int A_BLOCKS = (RBK + WT - 1) / WT;
#pragma unroll 1
            for (int i = 0; i < A_BLOCKS; i++) {
                const int blk = wt + WT * i;
                if (blk >= (extra ? RBK : RBK - 1)) break;
                if (uint32_t(blk) >= live_blocks) {
                    // (a short share: no scores to take, and no operands will be made of this block; the other
                    // pair's wave of the same blocks leaves it out as well)
                    if (j == 0) bmax_lds[my_row * W::BROW + (n & 7) * W::BSTRIDE + blk] = NO_SCORE, bsum_lds[my_row * W::BROW + (n & 7) * W::BSTRIDE + blk] = 0.0f;
                    continue;
                }
                await(W::C_KPART + (blk >> 3), W::K_LOADERS);  // this part of the keys is in LDS (first: and the scales)
                const unsigned char *kb = lds_raw + W::K_OFF + blk * W::K_BLOCK_BYTES;
                KeyRegs<BITS> kreg[4];
#pragma unroll
                for (int gg = 0; gg < 4; gg++) {
                    if constexpr (BITS == 8) {
                        const u32x4 v = *reinterpret_cast<const u32x4 *>(kb + gg * 1024 + n * 64 + j * 16);
                        kreg[gg].w[0] = v.x, kreg[gg].w[1] = v.y, kreg[gg].w[2] = v.z, kreg[gg].w[3] = v.w;
                    } else {
                        const u32x2 v = *reinterpret_cast<const u32x2 *>(kb + (gg >> 1) * 1024 + n * 64 + (gg & 1) * 32 + j * 8);
                        kreg[gg].w[0] = v.x, kreg[gg].w[1] = v.y;
                    }
                }
                const int tok0 = BLOCK * blk + 4 * j;  // this lane's 4 tokens of the round in C layout
                const uint32_t *sb_w = sb_lds + BLOCK * blk;
                const u32x2 zr = {sb_w[W::SB_ARRAY / 4 + n], sb_w[W::SB_ARRAY / 4 + RT + n]};
                const half8 zop = as_half8(perm(0, zr.x, 0x01000100u), perm(0, zr.x, 0x03020302u), perm(0, zr.y, 0x01000100u), perm(0, zr.y, 0x03020302u));
                const u32x4 s01 = *reinterpret_cast<const u32x4 *>(sb_w + 4 * j);
                const u32x4 s23 = *reinterpret_cast<const u32x4 *>(sb_w + RT + 4 * j);
                const uint32_t sw[8] = {s01.x, s23.x, s01.y, s23.y, s01.z, s23.z, s01.w, s23.w};
                floatx4 s = {0, 0, 0, 0}, rr[4];
                s = __builtin_amdgcn_mfma_f32_16x16x32_f16(zop, qz_reg[0], s, 0, 0, 0);
                s = __builtin_amdgcn_mfma_f32_16x16x32_f16(zop, qz_reg[1], s, 0, 0, 0);
#pragma unroll
                for (int gg = 0; gg < 4; gg++) {
                    rr[gg] = floatx4{0, 0, 0, 0};
#pragma unroll
                    for (int ab = 0; ab < 2; ab++) {
                        const half8 kop = key_operand<BITS>(kreg[gg], ab);
                        rr[gg] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kop, q_hi[gg * 2 + ab], rr[gg], 0, 0, 0);
                        rr[gg] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kop, q_lo[gg * 2 + ab], rr[gg], 0, 0, 0);
                    }
                }
                constexpr float C1 = code_up<BITS>() / Q_UP;
#pragma unroll
                for (int tk = 0; tk < 4; tk++) {
                    float d = 0.0f;
#pragma unroll
                    for (int gg = 0; gg < 4; gg++) d += half_bits_to_float(sw[2 * tk + (gg >> 1)] >> (16 * (gg & 1))) * rr[gg][tk];
                    const float v = s[tk] + d * C1;
                    s[tk] = base + tok0 + tk < my_limit ? v : NO_SCORE;  // (also whatever a block past the round left in LDS)
                }
                // the block's softmax relative to its own maximum, per column
                float cm = fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]));
                cm = across_rows<16, 64>(cm, MaxOp());
                float sum = 0.0f;
#pragma unroll
                for (int tk = 0; tk < 4; tk++) {
                    s[tk] = s[tk] > 0.5f * NO_SCORE ? __builtin_amdgcn_exp2f(s[tk] - cm) : 0.0f;
                    sum += s[tk];
                }
                sum = across_rows<16, 64>(sum, SumOp());
                if (j == 0) bmax_lds[my_row * W::BROW + (n & 7) * W::BSTRIDE + blk] = cm, bsum_lds[my_row * W::BROW + (n & 7) * W::BSTRIDE + blk] = sum;
                // the scores go over the block's own keys: when this wave has them in registers, and with
                // two pairs the other pair's wave of the same blocks, which takes them in the same order
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                if constexpr (PAIRS > 1) {
                    // (the blocks a wave leaves out are its last ones: i counts the ones it takes)
                    raise(W::C_MERGE + wt);
                    await(W::C_MERGE + wt, PAIRS * (i + 1));
                }
                *reinterpret_cast<floatx4 *>(s_block(blk, my_row) + (n & 7) * BLOCK + 4 * j) = s;
            }
            if (wt == 0 && !extra && j == 0) bmax_lds[my_row * W::BROW + (n & 7) * W::BSTRIDE + 16] = NO_SCORE, bsum_lds[my_row * W::BROW + (n & 7) * W::BSTRIDE + 16] = 0.0f;
        }
        raise(W::C_SCORES);
        await(W::C_SCORES, W::WAVES);

        // ---- the columns' maxima, the probability operands of this wave's k-steps ----
        // A operand: lane (n, j) holds tokens 8j .. 8j + 7 of the k-step for column n, as hi and as lo parts.
        float nm[PAIRS], zacc[PAIRS];
#pragma unroll
        for (int p = 0; p < PAIRS; p++) nm[p] = round_max(row_of(p, col_row), NO_SCORE), zacc[p] = 0.0f;
        const bool fifth = extra && b2 == 0;  // k-step 8: block 16 (lane groups 0 and 1; the others repeat them with factor 0)
        half8 p_hi[PAIRS][W::SLOTS], p_lo[PAIRS][W::SLOTS];
#pragma unroll
        for (int sl = 0; sl < W::SLOTS; sl++) {
            // (no block 16 | a short share: the k-step has no tokens)
            if ((sl == 4 && !fifth) || uint32_t(2 * (2 * sl + b2)) >= range) {
#pragma unroll
                for (int p = 0; p < PAIRS; p++) p_hi[p][sl] = p_lo[p][sl] = half8{0, 0, 0, 0, 0, 0, 0, 0};
                continue;
            }
            const int ks = 2 * sl + b2;  // tokens 32 ks ..: blocks 2 ks and 2 ks + 1
            const int jj = sl == 4 ? (j & 1) : j;
            const int blk = 2 * ks + (jj >> 1);
            const int sh = 16 * (g & 1);
            // value scales and biases of group g: half g % 2 of the tokens' dwords of groups (g, g ^ 1).
            // (Tokens past the share have probability 0 and the scales of the share's last token:
            // every load is clamped to it, so nothing but cache rows in use is ever read.)
            const uint32_t *vsp = sb_lds + 2 * (W::SB_ARRAY / 4) + (g >> 1) * RT + 32 * ks + 8 * jj;
            const u32x4 sv0 = *reinterpret_cast<const u32x4 *>(vsp), sv1 = *reinterpret_cast<const u32x4 *>(vsp + 4);
            const u32x4 zv0 = *reinterpret_cast<const u32x4 *>(vsp + W::SB_ARRAY / 4), zv1 = *reinterpret_cast<const u32x4 *>(vsp + W::SB_ARRAY / 4 + 4);
            const uint32_t sw[8] = {sv0.x, sv0.y, sv0.z, sv0.w, sv1.x, sv1.y, sv1.z, sv1.w};
            const uint32_t zw[8] = {zv0.x, zv0.y, zv0.z, zv0.w, zv1.x, zv1.y, zv1.z, zv1.w};
            float vscale[8], vbias[8];
#pragma unroll
            for (int e = 0; e < 8; e++) vscale[e] = half_bits_to_float(sw[e] >> sh), vbias[e] = half_bits_to_float(zw[e] >> sh);
            const int fb = 2 * ks + (j >> 1);  // block 17 does not exist: factor 0
#pragma unroll
            for (int p = 0; p < PAIRS; p++) {
                const int r = row_of(p, col_row);
                const float *sp = s_block(blk, r) + (n & 7) * BLOCK + 8 * (jj & 1);
                const floatx4 pt0 = *reinterpret_cast<const floatx4 *>(sp), pt1 = *reinterpret_cast<const floatx4 *>(sp + 4);
                const float pt[8] = {pt0[0], pt0[1], pt0[2], pt0[3], pt1[0], pt1[1], pt1[2], pt1[3]};
                // 2^(block maximum - round maximum) * P_UP (2^8, so that the lo part stays a normal f16)
                const float f = fb < RBK ? __builtin_amdgcn_exp2f(bmax_lds[r * W::BROW + (n & 7) * W::BSTRIDE + (fb < RBK ? fb : 0)] - nm[p] + 8.0f) : 0.0f;
                float x[8], lo[8], zb = 0.0f;
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    zb += pt[e] * vbias[e];
                    x[e] = pt[e] * f * vscale[e];
                    lo[e] = x[e] - __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, x[e]) & 0xffffe000u);
                }
                zacc[p] += zb * f;
                uint32_t o[8];
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    // round toward zero: exact truncation to the hi part
                    o[e] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(x[2 * e], x[2 * e + 1]));
                    o[4 + e] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(lo[2 * e], lo[2 * e + 1]));
                }
                // (pinned: left alone, the compiler moves an operand's arithmetic down to its use, behind the wait for the values)
                asm volatile("" : "+v"(o[0]), "+v"(o[1]), "+v"(o[2]), "+v"(o[3]), "+v"(o[4]), "+v"(o[5]), "+v"(o[6]), "+v"(o[7]));
                p_hi[p][sl] = as_half8(o[0], o[1], o[2], o[3]);
                p_lo[p][sl] = as_half8(o[4], o[5], o[6], o[7]);
            }
        }
        raise(W::C_BUILT);  // this wave is through with the scores

        // ---- phase C: O += P V, one k-step per value slot as the slots land ----
        floatx4 acc[PAIRS][4];  // [pair][tile of 16 dims 4n' + e]: rows 4j .. 4j+3 (columns of the pair), column n'
#pragma unroll
        for (int p = 0; p < PAIRS; p++) {
#pragma unroll
            for (int e = 0; e < 4; e++) acc[p][e] = floatx4{0, 0, 0, 0};
        }
#pragma unroll
        for (int sl = 0; sl < W::SLOTS; sl++) {
            if ((sl == 4 && !fifth) || uint32_t(2 * (2 * sl + b2)) >= range) continue;
            await(W::C_SLOT + sl, W::V_LOADERS);  // value slot sl is in LDS
            ValRegs<BITS> vreg;
            read_values(sl == 4 ? 8 : 2 * sl + b2, g, vreg);
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const half8 vop = val_operand<BITS>(vreg, e, n);
#pragma unroll
                for (int p = 0; p < PAIRS; p++) {
                    acc[p][e] = __builtin_amdgcn_mfma_f32_16x16x32_f16(p_hi[p][sl], vop, acc[p][e], 0, 0, 0);
                    acc[p][e] = __builtin_amdgcn_mfma_f32_16x16x32_f16(p_lo[p][sl], vop, acc[p][e], 0, 0, 0);
                }
            }
        }

        // ---- epilogue: the two waves of a group add up, wave 2g writes the partials ----
#pragma unroll
        for (int p = 0; p < PAIRS; p++) {
            // a column's bias sum: over the four lane groups
            const float z = across_rows<16, 64>(zacc[p], SumOp());
            if (j == 0) zs_lds[(wave * PAIRS + p) * 16 + n] = z;
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        floatx4 mine[PAIRS][4];  // column 4j + i of the pair, dims 64 g + 4n .. + 3
#pragma unroll
        for (int p = 0; p < PAIRS; p++) {
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float zb = zs_lds[(wave * PAIRS + p) * 16 + 4 * j + i] * (1.0f / P_UP);
#pragma unroll
                for (int e = 0; e < 4; e++) mine[p][i][e] = acc[p][e][i] * unscale + zb;
            }
        }
        // (the merge lies over the keys, which hold the scores until every wave has built its operands)
        floatx4 *x_o = reinterpret_cast<floatx4 *>(lds_raw + W::K_OFF);  // [pair][group][lane][4 columns]
        await(W::C_BUILT, W::WAVES);
        if (b2 == 1) {
#pragma unroll
            for (int p = 0; p < PAIRS; p++) {
#pragma unroll
                for (int i = 0; i < 4; i++) x_o[((p * 4 + g) * 64 + lane) * 4 + i] = mine[p][i];
            }
            raise(W::C_MERGE + 4 + g);
            leave();
            return;
        }
        if (wave == 0) {
#pragma unroll
            for (int p = 0; p < PAIRS; p++) {
                const int r = 2 * p + col_row;
                const float l = round_sum(row_of(p, col_row), nm[p]);
                if (j == 0 && r < M) {
                    const size_t slot = (size_t(r) * a.nsplits + split) * a.heads + kv * 8 + (n & 7);
                    *reinterpret_cast<floatx2 *>(a.part_ml + 2 * slot) = floatx2{nm[p], marked(l)};
                }
            }
        }
        await(W::C_MERGE + 4 + g, 1);
#pragma unroll
        for (int p = 0; p < PAIRS; p++) {
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int c = 4 * j + i, r = 2 * p + (c >> 3);
                if (r < M) {
                    const size_t slot = (size_t(r) * a.nsplits + split) * a.heads + kv * 8 + (c & 7);
                    // (nobody on this CU reads the partials again: past the caches)
                    __builtin_nontemporal_store(mine[p][i] + x_o[((p * 4 + g) * 64 + lane) * 4 + i], reinterpret_cast<floatx4 *>(a.part_o + slot * DIM + 64 * g + 4 * n));
                }
            }
        }
    } else {
        // ---- one row -----------------------------------------------------------------------------
        // Scores: wave w takes the blocks w and w + 8 (wave 0 also 16).  O += P V: waves 2g and 2g + 1 share
        // group g and take alternate k-steps, so that each value slot gives every wave one k-step.
        // ---- prologue: the query row to f16 hi/lo operands in LDS (operand row n: head n & 7, hi part in
        // rows 0-7 and lo part in rows 8-15 of the one tile) ---------------------------------------------
        {
            const float qmul = a.scale * 1.4426950408889634f * Q_UP;
            half8 op;
            float sum = 0.0f;
#pragma unroll
            for (int e = 0; e < 8; e++) {
                _Float16 h, lw;
                split_hi_lo(qv[0][key_slot_dim<BITS>(e)] * qmul, h, lw);
                const _Float16 x = n < 8 ? h : lw;
                op[e] = x;
                sum += (float)x;
            }
            q_lds[wave * 64 + lane] = op;
            // key bias term: slot `k-step` of this lane in the B operand of one more MFMA, as hi and lo halves
            _Float16 h, lw;
            split_hi_lo(sum * (1.0f / Q_UP), h, lw);
            qz_lds[(0 * 64 + lane) * 8 + wave] = h;
            qz_lds[(1 * 64 + lane) * 8 + wave] = lw;
            // blocks that never exist
            if (wave == 0 && lane < 8 * (W::BSINGLE - RBK)) {
                const int idx = (lane / (W::BSINGLE - RBK)) * W::BSTRIDE + RBK + lane % (W::BSINGLE - RBK);
                bmax_lds[idx] = NO_SCORE, bsum_lds[idx] = 0.0f;
            }
        }
        raise(W::C_QUERY);

        // ---- running state -------------------------------------------------------------
        float m_run = NO_SCORE;
        float l_run = 0.0f;    // sum of P of head n & 7 (wave 0 keeps it)
        float zacc = 0.0f;     // sum of P * P_UP * value bias of group g over this lane's tokens
        floatx4 acc[4];        // [tile of 16 dims 4n' + e]: rows 4j .. 4j+3 (operand rows), column n'
#pragma unroll
        for (int e = 0; e < 4; e++) acc[e] = floatx4{0, 0, 0, 0};
        await(W::C_QUERY, W::WAVES);

        if constexpr (W::ALTERNATE) if (alt) {
            // ---- a share of more than one round: rounds of up to ALT_BLOCKS blocks in alternate halves of LDS ----
            // Round r lies in the blocks ALT_BLOCKS (r % 2) .. of the keys' and the values' places, of the scales and of
            // the block table: every computing wave takes the scores of one block and two k-steps
            // of O += P V per round, and the loaders fill the other half meanwhile.  A half is free for round r + 2 when
            // every wave has built its operands (keys, scales, scores) and is through with the values of round r.
            constexpr int AB = W::ALT_BLOCKS, WAVE_BLOCKS = AB / W::WAVES, WAVE_STEPS = AB / 4;
            // The query operands are held over the rounds: read anew in each they were 80 KB of the round's way through LDS, in front of its
            // first product.  What makes a round of 4-bit codes shorter, us a layer at 60000 | 150000 | 216000 tokens, without -> with it: the operands held
            // 18.2 -> 17.8 | 31.0 -> 30.05 | 39.8 -> 38.4; one_row_operand 18.1 | 30.6 | 39.2 (a single round of 32768 tokens 13.3 -> 13.05); the mask in the last
            // block only 17.95 | 30.4 | 39.0; RawMaxOp 17.85 | 30.25 | 38.7.  8-bit codes, whose rounds wait for memory: the mask 20.9 -> 20.6 at 60000,
            // 15.4 -> 15.3 at 32768, the others nothing.  What the loaders alone take at 150000 tokens of 4 bits, with no arithmetic
            // at all, is 25.4.  Tried here: scores a round ahead of the operands, so that no wave waits for another's (32.7); four
            // places of 8 blocks for 4-bit codes, two rounds of every loader on their way (34.4: what has landed is told of later); the
            // values and the next keys read as soon as they are there, under the operands (31.9).
            half8 q_reg[8], qz_reg[2];
#pragma unroll
            for (int i = 0; i < 8; i++) q_reg[i] = q_lds[i * 64 + lane];
            qz_reg[0] = *reinterpret_cast<const half8 *>(qz_lds + lane * 8);
            qz_reg[1] = *reinterpret_cast<const half8 *>(qz_lds + (64 + lane) * 8);
#pragma unroll
            for (int i = 0; i < 8; i++) asm volatile("" : "+v"(q_reg[i]));
            asm volatile("" : "+v"(qz_reg[0]), "+v"(qz_reg[1]));
#pragma unroll 1
            for (uint32_t round = 0; round < n_rounds; round++) {
                const uint32_t base = (blk_begin + place(round) * per_round) * BLOCK, nb = blocks_of(place(round));
                const int half = int(round & 1) * AB;  // the round's first block in LDS
                const uint32_t round_limit = min(limit, base + nb * BLOCK);  // tokens of this round end here
                const uint32_t live_blocks = (nb + 1) & ~1u;  // k-steps are two blocks: the blocks of the k-steps that have tokens
                // ---- phase A: the scores of the blocks wave (, wave + 8) of the round ----
#pragma unroll 1
                for (int part = 0; part < WAVE_BLOCKS; part++) {
                    const int rblk = wave + W::WAVES * part;  // of the round
                    const int blk = half + rblk;              // in LDS
                    if (uint32_t(rblk) >= live_blocks) {
                        // (no scores to take, and no operands will be made of this block; the table still holds the entries of
                        // the round before last until every wave has built its operands from them)
                        if (round > 1) await(W::C_BUILT, W::WAVES * (round - 1));
                        if (j == 0 && n < 8) bmax_lds[n * W::BSTRIDE + blk] = NO_SCORE, bsum_lds[n * W::BSTRIDE + blk] = 0.0f;
                    } else {
                        await(W::C_KPART + int(round & 1), round / 2 + 1);  // the round's keys and scales are in LDS (its loader's counter)
                        const unsigned char *kb = lds_raw + W::K_OFF + blk * W::K_BLOCK_BYTES;
                        KeyRegs<BITS> kreg[4];
#pragma unroll
                        for (int gg = 0; gg < 4; gg++) {
                            if constexpr (BITS == 8) {
                                const u32x4 v = *reinterpret_cast<const u32x4 *>(kb + gg * 1024 + n * 64 + j * 16);
                                kreg[gg].w[0] = v.x, kreg[gg].w[1] = v.y, kreg[gg].w[2] = v.z, kreg[gg].w[3] = v.w;
                            } else {
                                const u32x2 v = *reinterpret_cast<const u32x2 *>(kb + (gg >> 1) * 1024 + n * 64 + (gg & 1) * 32 + j * 8);
                                kreg[gg].w[0] = v.x, kreg[gg].w[1] = v.y;
                            }
                        }
                        const int tok0 = BLOCK * rblk + 4 * j;  // this lane's 4 tokens of the round in C layout
                        const uint32_t *sb_w = sb_lds + BLOCK * blk;  // the block's dwords of groups (0, 1); + RT: groups (2, 3)
                        floatx4 sc;
                        {
                            const u32x2 zr = {sb_w[W::SB_ARRAY / 4 + n], sb_w[W::SB_ARRAY / 4 + RT + n]};
                            const half8 zop = as_half8(perm(0, zr.x, 0x01000100u), perm(0, zr.x, 0x03020302u), perm(0, zr.y, 0x01000100u),
                                                       perm(0, zr.y, 0x03020302u));
                            sc = floatx4{0, 0, 0, 0};
                            sc = __builtin_amdgcn_mfma_f32_16x16x32_f16(zop, qz_reg[0], sc, 0, 0, 0);
                            sc = __builtin_amdgcn_mfma_f32_16x16x32_f16(zop, qz_reg[1], sc, 0, 0, 0);
                        }
                        floatx4 r[4];
#pragma unroll
                        for (int gg = 0; gg < 4; gg++) {
                            r[gg] = floatx4{0, 0, 0, 0};
#pragma unroll
                            for (int ab = 0; ab < 2; ab++) {
                                r[gg] = __builtin_amdgcn_mfma_f32_16x16x32_f16(key_operand<BITS>(kreg[gg], ab), q_reg[gg * 2 + ab], r[gg], 0, 0, 0);
                            }
                        }
                        const u32x4 s01 = *reinterpret_cast<const u32x4 *>(sb_w + 4 * j);
                        const u32x4 s23 = *reinterpret_cast<const u32x4 *>(sb_w + RT + 4 * j);
                        const uint32_t sw[8] = {s01.x, s23.x, s01.y, s23.y, s01.z, s23.z, s01.w, s23.w};
                        constexpr float C1 = code_up<BITS>() / Q_UP;
#pragma unroll
                        for (int tk = 0; tk < 4; tk++) {
                            float d = 0.0f;
#pragma unroll
                            for (int gg = 0; gg < 4; gg++) d += half_bits_to_float(sw[2 * tk + (gg >> 1)] >> (16 * (gg & 1))) * r[gg][tk];
                            const float v = sc[tk] + d * C1;
                            sc[tk] = v + dpp<0x128>(v);  // row_ror 8: the other part (hi | lo) of the same head
                        }
                        if (base + BLOCK * (rblk + 1) > round_limit) {
#pragma unroll
                            for (int tk = 0; tk < 4; tk++) sc[tk] = base + tok0 + tk < round_limit ? sc[tk] : NO_SCORE;  // (also whatever a block past the round left in LDS)
                        }
                        float cm = fmaxf(fmaxf(sc[0], sc[1]), fmaxf(sc[2], sc[3]));
                        cm = across_rows<16, 64>(cm, RawMaxOp());
                        float sum = 0.0f;
#pragma unroll
                        for (int tk = 0; tk < 4; tk++) {
                            sc[tk] = sc[tk] > 0.5f * NO_SCORE ? __builtin_amdgcn_exp2f(sc[tk] - cm) : 0.0f;
                            sum += sc[tk];
                        }
                        sum = across_rows<16, 64>(sum, SumOp());
                        // over the block's own keys (every lane of the wave has its key registers by now)
                        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                        if (n < 8) *reinterpret_cast<floatx4 *>(s_block(blk, 0) + n * BLOCK + 4 * j) = sc;
                        if (j == 0 && n < 8) bmax_lds[n * W::BSTRIDE + blk] = cm, bsum_lds[n * W::BSTRIDE + blk] = sum;
                    }
                }
                raise(W::C_SCORES);
                await(W::C_SCORES, W::WAVES * (round + 1));

                // ---- the round's maximum per head, and what was summed so far brought to it ----
                float nm = m_run;
                {
                    const floatx4 *bmx = reinterpret_cast<const floatx4 *>(bmax_lds + (n & 7) * W::BSTRIDE + half);
#pragma unroll
                    for (int i = 0; i < AB / 4; i++) {
                        const floatx4 w = bmx[i];
                        nm = fmaxf(nm, fmaxf(fmaxf(w[0], w[1]), fmaxf(w[2], w[3])));
                    }
                }
                const float al = __builtin_amdgcn_exp2f(m_run - nm);  // (first round: 2^(-1e30 - nm) = 0, and nothing to scale)
                if (round > 0) {
                    zacc *= al;
                    floatx4 al4;
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        al4[i] = __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(4 * ((4 * j + i) & 7), __builtin_bit_cast(int, al)));
                    }
#pragma unroll
                    for (int e = 0; e < 4; e++) acc[e] *= al4;
                }
                m_run = nm;
                if (wave == 0) {
                    // the round's sum of P of head n & 7: lane group j adds the blocks (AB / 4) j ..
                    float sum = 0.0f;
#pragma unroll
                    for (int i = 0; i < AB / 4; i++) {
                        const int b = half + (AB / 4) * j + i;
                        sum += bsum_lds[(n & 7) * W::BSTRIDE + b] * __builtin_amdgcn_exp2f(bmax_lds[(n & 7) * W::BSTRIDE + b] - nm);  // (a block that is not there: sum 0)
                    }
                    l_run = l_run * al + across_rows<16, 64>(sum, SumOp());
                }

                // ---- probability operands of this wave's k-steps (as in a single round) ----
                half8 p_alt[WAVE_STEPS];
                {
                    const int hh = n >> 3;  // this lane makes tokens 8j + 4 hh .. + 3 of a k-step
                    const uint32_t sel = group_sel(g);
#pragma unroll
                    for (int i = 0; i < WAVE_STEPS; i++) {
                        if (uint32_t(2 * (2 * i + b2)) >= nb) {  // the k-step has no tokens
                            p_alt[i] = half8{0, 0, 0, 0, 0, 0, 0, 0};
                            continue;
                        }
                        const int ks = half / 2 + 2 * i + b2;  // in LDS: tokens 32 ks ..: blocks 2 ks and 2 ks + 1
                        const int blk = 2 * ks + (j >> 1);
                        const floatx4 pt = *reinterpret_cast<const floatx4 *>(s_block(blk, 0) + (n & 7) * BLOCK + 8 * (j & 1) + 4 * hh);
                        const uint32_t *vsp = sb_lds + 2 * (W::SB_ARRAY / 4) + (g >> 1) * RT + 32 * ks + 8 * j + 4 * hh;
                        const u32x4 sv = *reinterpret_cast<const u32x4 *>(vsp);
                        const u32x4 zv = *reinterpret_cast<const u32x4 *>(vsp + W::SB_ARRAY / 4);
                        // 2^(block maximum - maximum so far) * P_UP (2^8, so that the lo part stays a normal f16)
                        const float f = __builtin_amdgcn_exp2f(bmax_lds[(n & 7) * W::BSTRIDE + blk] - nm + 8.0f);
                        p_alt[i] = one_row_operand(pt, f, sv, zv, sel, zacc);
                    }
                }
                raise(W::C_BUILT);  // this wave is through with the round's keys, scores, scales and biases

                // ---- phase C: O += P V of the wave's k-steps ----
                await(W::C_SLOT + int(round & 1), round / 2 + 1);  // the round's values are in LDS (its loader's counter)
                {
                    ValRegs<BITS> vreg[WAVE_STEPS];
#pragma unroll
                    for (int i = 0; i < WAVE_STEPS; i++) {
                        if (uint32_t(2 * (2 * i + b2)) >= nb) continue;
#pragma unroll
                        for (int e = 0; e < 8; e++) {
                            const int tk = BLOCK * half + 32 * (2 * i + b2) + 8 * j + e;
                            vreg[i].w[e] = *reinterpret_cast<const uint32_t *>(lds_raw + W::V_OFF + tk * RB + ((val_lane_offset<BITS>(g, n) + j * (RB / 4)) & (RB - 1)));
                        }
                    }
#pragma unroll
                    for (int i = 0; i < WAVE_STEPS; i++) {
                        if (uint32_t(2 * (2 * i + b2)) >= nb) continue;
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            acc[e] = __builtin_amdgcn_mfma_f32_16x16x32_f16(p_alt[i], val_operand<BITS>(vreg[i], e, n), acc[e], 0, 0, 0);
                        }
                    }
                }
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the value codes are in registers
                raise(W::C_DONE);
            }
        }
        if (!alt) {
            // ---- a share of up to 17 blocks: one round ----
            constexpr uint32_t round = 0;  // (written as the first of several rounds)
            constexpr bool more = false;
            const uint32_t base = (blk_begin + round * per_round) * BLOCK, nb = blocks_of(round);
            const bool extra = nb == uint32_t(RBK);  // the round has block 16
            const uint32_t round_limit = min(limit, base + nb * BLOCK);  // tokens of this round end here
            const uint32_t live_blocks = (nb + 1) & ~1u;  // k-steps are two blocks: the blocks of the k-steps that have tokens

            // ---- phase A: scores of blocks wave, wave + 8 (and wave 0: 16) --------------------------
            // (the query operands are read again in every round: they are not needed between the scores
            // of one round and the next, and the registers are)
            {
                half8 q_reg[8], qz_reg[2];
#pragma unroll
                for (int i = 0; i < 8; i++) q_reg[i] = q_lds[i * 64 + lane];
                qz_reg[0] = *reinterpret_cast<const half8 *>(qz_lds + lane * 8);
                qz_reg[1] = *reinterpret_cast<const half8 *>(qz_lds + (64 + lane) * 8);
                const int parts = (wave == 0 && extra) ? 3 : 2;
#pragma unroll 1
                for (int part = 0; part < parts; part++) {
                    const int blk = wave + 8 * part;
                    if (uint32_t(blk) >= live_blocks) {
                        // (a short round: no scores to take, and no operands will be made of this block; the
                        // table still holds the round before's entries until every wave has built its operands
                        // from them, which is also what the key loader waits for before it overwrites the keys)
                        if (round > 0) await(W::C_BUILT, W::WAVES * round);
                        if (j == 0 && n < 8) bmax_lds[n * W::BSTRIDE + blk] = NO_SCORE, bsum_lds[n * W::BSTRIDE + blk] = 0.0f;
                        continue;
                    }
                    await(W::C_KPART + part, W::K_LOADERS * (round + 1));  // this part of the keys is in LDS (first: and the scales)
                    const unsigned char *kb = lds_raw + W::K_OFF + blk * W::K_BLOCK_BYTES;
                    KeyRegs<BITS> kreg[4];
#pragma unroll
                    for (int gg = 0; gg < 4; gg++) {
                        if constexpr (BITS == 8) {
                            // the group's 64 bytes of token n are piece gg: 16 bytes j of them
                            const u32x4 v = *reinterpret_cast<const u32x4 *>(kb + gg * 1024 + n * 64 + j * 16);
                            kreg[gg].w[0] = v.x, kreg[gg].w[1] = v.y, kreg[gg].w[2] = v.z, kreg[gg].w[3] = v.w;
                        } else {
                            // the group's 32 bytes of token n are half gg % 2 of piece gg / 2: 8 bytes j of them
                            const u32x2 v = *reinterpret_cast<const u32x2 *>(kb + (gg >> 1) * 1024 + n * 64 + (gg & 1) * 32 + j * 8);
                            kreg[gg].w[0] = v.x, kreg[gg].w[1] = v.y;
                        }
                    }
                    const int tok0 = BLOCK * blk + 4 * j;  // this lane's 4 tokens of the round in C layout
                    const uint32_t *sb_w = sb_lds + BLOCK * blk;  // the block's dwords of groups (0, 1); + RT: groups (2, 3)
                    floatx4 s;
                    {
                        // bias term: slot e of every lane group belongs to group e / 2 of token n
                        const u32x2 zr = {sb_w[W::SB_ARRAY / 4 + n], sb_w[W::SB_ARRAY / 4 + RT + n]};
                        const half8 zop = as_half8(perm(0, zr.x, 0x01000100u), perm(0, zr.x, 0x03020302u), perm(0, zr.y, 0x01000100u),
                                                   perm(0, zr.y, 0x03020302u));
                        s = floatx4{0, 0, 0, 0};
                        s = __builtin_amdgcn_mfma_f32_16x16x32_f16(zop, qz_reg[0], s, 0, 0, 0);
                        s = __builtin_amdgcn_mfma_f32_16x16x32_f16(zop, qz_reg[1], s, 0, 0, 0);
                    }
                    floatx4 r[4];
#pragma unroll
                    for (int gg = 0; gg < 4; gg++) {
                        r[gg] = floatx4{0, 0, 0, 0};
#pragma unroll
                        for (int ab = 0; ab < 2; ab++) {
                            r[gg] = __builtin_amdgcn_mfma_f32_16x16x32_f16(key_operand<BITS>(kreg[gg], ab), q_reg[gg * 2 + ab], r[gg], 0, 0, 0);
                        }
                    }
                    // scales of the lane's tokens 4j .. 4j+3 of the block: groups (0, 1) and groups (2, 3)
                    const u32x4 s01 = *reinterpret_cast<const u32x4 *>(sb_w + 4 * j);
                    const u32x4 s23 = *reinterpret_cast<const u32x4 *>(sb_w + RT + 4 * j);
                    const uint32_t sw[8] = {s01.x, s23.x, s01.y, s23.y, s01.z, s23.z, s01.w, s23.w};
                    constexpr float C1 = code_up<BITS>() / Q_UP;
#pragma unroll
                    for (int tk = 0; tk < 4; tk++) {
                        float d = 0.0f;
#pragma unroll
                        for (int gg = 0; gg < 4; gg++) d += half_bits_to_float(sw[2 * tk + (gg >> 1)] >> (16 * (gg & 1))) * r[gg][tk];
                        const float v = s[tk] + d * C1;
                        s[tk] = v + dpp<0x128>(v);  // row_ror 8: the other part (hi | lo) of the same head
                    }
                    if (base + BLOCK * (blk + 1) > round_limit) {
#pragma unroll
                        for (int tk = 0; tk < 4; tk++) s[tk] = base + tok0 + tk < round_limit ? s[tk] : NO_SCORE;  // (also whatever a block past the round left in LDS)
                    }
                    // the block's softmax relative to its own maximum, per head
                    float cm = fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]));
                    cm = across_rows<16, 64>(cm, RawMaxOp());
                    float sum = 0.0f;
#pragma unroll
                    for (int tk = 0; tk < 4; tk++) {
                        s[tk] = s[tk] > 0.5f * NO_SCORE ? __builtin_amdgcn_exp2f(s[tk] - cm) : 0.0f;
                        sum += s[tk];
                    }
                    sum = across_rows<16, 64>(sum, SumOp());
                    // over the block's own keys (every lane of the wave has its key registers by now)
                    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                    if (n < 8) *reinterpret_cast<floatx4 *>(s_block(blk, 0) + n * BLOCK + 4 * j) = s;
                    if (j == 0 && n < 8) bmax_lds[n * W::BSTRIDE + blk] = cm, bsum_lds[n * W::BSTRIDE + blk] = sum;
                }
                if (wave == 0 && !extra) {
                    // (block 16 of the round before, if it had one, is read until every wave has built its operands)
                    if (round > 0) await(W::C_BUILT, W::WAVES * round);
                    if (j == 0 && n < 8) bmax_lds[n * W::BSTRIDE + 16] = NO_SCORE, bsum_lds[n * W::BSTRIDE + 16] = 0.0f;
                }
            }
            raise(W::C_SCORES);
            await(W::C_SCORES, W::WAVES * (round + 1));

            // ---- the round's maximum per head, and what was summed so far brought to it -------------
            float nm = m_run;
            {
                const floatx4 *bmx = reinterpret_cast<const floatx4 *>(bmax_lds + (n & 7) * W::BSTRIDE);
#pragma unroll
                for (int i = 0; i < W::BSINGLE / 4; i++) {
                    const floatx4 w = bmx[i];
                    nm = fmaxf(nm, fmaxf(fmaxf(w[0], w[1]), fmaxf(w[2], w[3])));
                }
            }
            const float al = __builtin_amdgcn_exp2f(m_run - nm);  // (first round: 2^(-1e30 - nm) = 0, and nothing to scale)
            if (round > 0) {
                zacc *= al;
                // accumulator rows 4j + i are heads (4j + i) & 7: lane h (j = 0, n = h) holds head h's factor
                floatx4 al4;
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    al4[i] = __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(4 * ((4 * j + i) & 7), __builtin_bit_cast(int, al)));
                }
#pragma unroll
                for (int e = 0; e < 4; e++) acc[e] *= al4;
            }
            m_run = nm;
            if (wave == 0) {
                // the round's sum of P of head n & 7: lane group j adds blocks 5j .. 5j + 4
                float sum = 0.0f;
#pragma unroll
                for (int i = 0; i < W::BSINGLE / 4; i++) {
                    const int b = (W::BSINGLE / 4) * j + i;
                    sum += bsum_lds[(n & 7) * W::BSTRIDE + b] * __builtin_amdgcn_exp2f(bmax_lds[(n & 7) * W::BSTRIDE + b] - nm);  // (a block that is not there: sum 0)
                }
                l_run = l_run * al + across_rows<16, 64>(sum, SumOp());
            }

            // ---- probability operands of this wave's k-steps: P * value scale of group g, hi part in
            // operand rows 0-7 and lo part in rows 8-15.  The two lanes of a head (n and n + 8) make four of
            // the lane group's eight tokens each, both parts, and exchange what the other one feeds. ----
            half8 p_op[W::SLOTS];
            {
                const int hh = n >> 3;  // this lane makes tokens 8j + 4 hh .. + 3 of a k-step
                const uint32_t sel = group_sel(g);
                const bool fifth = extra && b2 == 0;  // k-step 8: block 16 (lane groups 0 and 1; the others repeat them with factor 0)
#pragma unroll
                for (int sl = 0; sl < W::SLOTS; sl++) {
                    // (no block 16 | a short round: the k-step has no tokens)
                    if ((sl == 4 && !fifth) || uint32_t(2 * (2 * sl + b2)) >= nb) {
                        p_op[sl] = half8{0, 0, 0, 0, 0, 0, 0, 0};
                        continue;
                    }
                    const int ks = 2 * sl + b2;  // tokens 32 ks ..: blocks 2 ks and 2 ks + 1
                    const int jj = sl == 4 ? (j & 1) : j;
                    const int blk = 2 * ks + (jj >> 1);
                    const floatx4 pt = *reinterpret_cast<const floatx4 *>(s_block(blk, 0) + (n & 7) * BLOCK + 8 * (jj & 1) + 4 * hh);
                    // value scales and biases of group g: half g % 2 of the tokens' dwords of groups (g, g ^ 1).
                    // (Tokens past the share have probability 0 and the scales of the share's last token:
                    // every load is clamped to it, so nothing but cache rows in use is ever read.)
                    const uint32_t *vsp = sb_lds + 2 * (W::SB_ARRAY / 4) + (g >> 1) * RT + 32 * ks + 8 * jj + 4 * hh;
                    const u32x4 sv = *reinterpret_cast<const u32x4 *>(vsp);
                    const u32x4 zv = *reinterpret_cast<const u32x4 *>(vsp + W::SB_ARRAY / 4);
                    // 2^(block maximum - round maximum) * P_UP (2^8, so that the lo part stays a normal f16)
                    const float f = __builtin_amdgcn_exp2f(bmax_lds[(n & 7) * W::BSTRIDE + 2 * ks + (j >> 1)] - nm + 8.0f);
                    p_op[sl] = one_row_operand(pt, f, sv, zv, sel, zacc);
                }
            }
            if (more) raise(W::C_BUILT);  // this wave is through with the round's scores, scales and biases

            // ---- phase C: O += P V, one k-step per value slot as the slots land ---------------------
            const unsigned char *vb = lds_raw + W::V_OFF;
            auto read_values = [&](int sl, ValRegs<BITS> &vreg) {
                const int jj = sl == 4 ? (j & 1) : j;
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    const int tk = 32 * (2 * sl + b2) + 8 * jj + e;
                    vreg.w[e] = *reinterpret_cast<const uint32_t *>(vb + tk * RB + ((val_lane_offset<BITS>(g, n) + jj * (RB / 4)) & (RB - 1)));
                }
            };
            auto add_values = [&](int sl, const ValRegs<BITS> &vreg) {
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    acc[e] = __builtin_amdgcn_mfma_f32_16x16x32_f16(p_op[sl], val_operand<BITS>(vreg, e, n), acc[e], 0, 0, 0);
                }
            };
            const bool fifth = extra && b2 == 0;
            // (a short round: not every k-step of this wave has tokens)
            auto has_tokens = [&](int sl) { return uint32_t(2 * (2 * sl + b2)) < nb; };
            if (nb >= 16 && peek(W::C_SLOT + 3) >= W::V_LOADERS * (round + 1)) {
                // slots 0-3 are there already (the slots land in order): every read at once
                ValRegs<BITS> vreg[4];
#pragma unroll
                for (int sl = 0; sl < 4; sl++) read_values(sl, vreg[sl]);
#pragma unroll
                for (int sl = 0; sl < 4; sl++) add_values(sl, vreg[sl]);
            } else {
#pragma unroll
                for (int sl = 0; sl < 4; sl++) {
                    if (!has_tokens(sl)) continue;
                    await(W::C_SLOT + sl, W::V_LOADERS * (round + 1));  // value slot sl is in LDS
                    ValRegs<BITS> vreg;
                    read_values(sl, vreg);
                    add_values(sl, vreg);
                }
            }
            if (fifth) {
                await(W::C_SLOT + 4, W::V_LOADERS * (round + 1));
                ValRegs<BITS> vreg;
                read_values(4, vreg);
                add_values(4, vreg);
            }
            if (more) {
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the value codes are in registers
                raise(W::C_DONE);
            }
        }

        // ---- epilogue: the two waves of a group add up, wave 2g writes the partial ---------------------
        {
            // the head's bias sum: over the four lane groups and the two lanes of the head
            float z = across_rows<16, 64>(zacc, SumOp());
            z += dpp<0x128>(z);
            if (j == 0 && n < 8) zs_lds[wave * 8 + n] = z;
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
        floatx4 mine[4];  // head 4j + i (j < 2), dims 64 g + 4n .. + 3
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float zb = zs_lds[wave * 8 + ((4 * j + i) & 7)] * (1.0f / P_UP);
#pragma unroll
            for (int e = 0; e < 4; e++) mine[i][e] = across_rows<32, 64>(acc[e][i], SumOp()) * unscale + zb;
        }
        // (the key area is free: the key loaders request nothing after the last round, and every wave is
        // past the last round's scores, having built its operands from them)
        floatx4 *x_o = reinterpret_cast<floatx4 *>(lds_raw + W::X_OFF);  // [group][lane < 32][4 rows]
        if (b2 == 1) {
            if (j < 2) {
#pragma unroll
                for (int i = 0; i < 4; i++) x_o[(g * 32 + lane) * 4 + i] = mine[i];
            }
            raise(W::C_MERGE + g);
            leave();
            return;
        }
        await(W::C_MERGE + g, 1);
        if (wave == 0 && j == 0 && n < 8) {
            const size_t slot = size_t(split) * a.heads + kv * 8 + n;
            *reinterpret_cast<floatx2 *>(a.part_ml + 2 * slot) = floatx2{m_run, marked(l_run)};
        }
        if (j < 2) {
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const size_t slot = size_t(split) * a.heads + kv * 8 + 4 * j + i;
                *reinterpret_cast<floatx4 *>(a.part_o + slot * DIM + 64 * g + 4 * n) = mine[i] + x_o[(g * 32 + lane) * 4 + i];
            }
        }
    }
    leave();
}

template <int BITS, int M>
__global__ __launch_bounds__((KeysFirst<BITS, M>::THREADS_)) void attention_partial_kernel_s(PartialArgs a) {
    attention_partial_s_body<BITS, M, false>(a, nullptr);
}
template <int BITS, int M>
__global__ __launch_bounds__((KeysFirst<BITS, M>::THREADS_)) void attention_token_kernel_s(TokenArgs t) {
    attention_partial_s_body<BITS, M, true>(t.a, &t.prep);
}

#include "decode_rows.hpp"
#include "decode_half_rows.hpp"
#include "decode_code_rows.hpp"

// Merges the splits of one (q head, row): weights 2^(m_c - M), then the gate
// (reference: attention_reduce / attention_reduce_rows,
// kernels/attention.metal:367-409, kernels/attention_rows.metal:296-342).
struct ReduceArgs {
    const float *part_o;
    const float *part_ml;
    const float *q_and_gate;
    float *out;
    uint32_t heads, capacity, nsplits, rows;
    const saetta_token_params *tp;
    uint32_t decode_len;
    uint32_t last_is_new;  // 1: the last split is the new tokens' (attention_token_kernel_*), the others the context before them
};

constexpr uint32_t MAX_SPLITS = 256;  // workgroups per kv head: 2 kv heads fill 512 slots of 256 CUs

// Partials of saetta_attn_decode_quant_static, the entry point that allocates nothing: room for one
// query row, 16 q heads and the most splits a launch uses: part_o f32 [256][16][256] (4 MiB), then
// part_ml f32 [256][16][2] (32 KiB).  Every device the library runs on holds its own copy of the
// array at its own address, until the process ends.  In host code the array's name is only a
// stand-in for hipGetSymbolAddress, never a device address: setup_decode asks for the address once
// per device and everything else uses g_static_scratch[device].
constexpr uint32_t STATIC_MAX_HEADS = 16;
constexpr size_t STATIC_PART_O_FLOATS = size_t(MAX_SPLITS) * STATIC_MAX_HEADS * DIM;
constexpr size_t STATIC_PART_ML_FLOATS = size_t(MAX_SPLITS) * STATIC_MAX_HEADS * 2;
static __device__ __align__(256) float scratch[STATIC_PART_O_FLOATS + STATIC_PART_ML_FLOATS];
constexpr int STATIC_MAX_DEVICES = 64;
float *g_static_scratch[STATIC_MAX_DEVICES] = {};

// One workgroup per (q head, row, DIMS dims of the head): wave w takes a quarter of the splits, lane
// (slot = lane / QUADS, quad = lane % QUADS) PER_LANE of them and four dims.  Latency is all there is to it: every load is
// requested before anything is waited for (buffer loads, whose slots past the last split read zero: with a branch around each
// the compiler waited for one before it asked for the next, and for the position before the first), a wave sums its splits
// relative to its own maximum, so that the four waves meet once, through LDS.
// A layer's token step, us, ten layers in a graph: 8-bit 300 tokens of 8192 9.1 -> 8.6, halves 4096 of 8192 10.9 -> 10.3, 8-bit 32768
// 16.8 -> 16.0; eight rows at 1000 tokens 18.3 -> 17.3.
// DIMS: a split's maximum and sum are a line of their own, read by every workgroup of a head, and 16 dims are half a line of its O,
// so one row, which is latency, has many workgroups, and more rows, which are bytes, have wide ones.  Us a layer's step, 16, 32, 64, 128
// dims: one row 8-bit 32768 tokens 15.67, 15.75, 15.91; two 16.98, 16.61, 16.86; three 22.24, 22.10, 21.90, 22.85; six of halves 57123 35.08,
// 34.42, 34.40; eight 20000 28.2, 26.9, 26.8, 8-bit 30.2, 29.1, 28.9, 29.5.  (The maxima and sums of a head in a row, as [row][head][split]: three
// rows 22.2 -> 21.8, but four of 4 bits at 3000 13.4 -> 13.8, one row 15.3 -> 15.4: eight scattered stores a split.)
// WAIT: slots past the splits at work are left out of the requests, which have to wait for the position then.  One and two
// rows read them all the same: the wait costs more than up to 2 MB of old partials a row.
template <int DIMS, int PER_LANE, bool WAIT>
__global__ __launch_bounds__(256) void attention_reduce_kernel(ReduceArgs a) {
    constexpr uint32_t QUADS = DIMS / 4, SLOTS = 64 / QUADS;
    __shared__ float wave_m[4], wave_l[4];
    __shared__ floatx4 wave_o[4][QUADS];
    const uint32_t h = blockIdx.x, row = blockIdx.y, slice = blockIdx.z;
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, slot = lane / QUADS, quad = lane % QUADS;
    const size_t qh = size_t(row) * a.heads + h;
    const uint32_t position = a.tp->position, kv_len = a.tp->kv_len;
    uint32_t parts = 0, fresh = 0;
    auto splits_at_work = [&]() {
        const uint32_t seen = min(a.decode_len ? kv_len : position + a.rows, a.capacity);
        const uint32_t max_len = a.last_is_new ? min(seen, position) : seen;
        parts = min(a.nsplits - a.last_is_new, (max_len + BLOCK - 1) / BLOCK), fresh = a.last_is_new ? a.nsplits - 1 : ~0u;
    };
    if constexpr (WAIT) splits_at_work();
    const uint32_t records = a.nsplits * a.heads;
    const __amdgpu_buffer_rsrc_t o_rsrc = make_rsrc(a.part_o + size_t(row) * records * DIM, records * DIM * 4);
    const __amdgpu_buffer_rsrc_t ml_rsrc = make_rsrc(a.part_ml + size_t(row) * records * 2, records * 8);
    const __amdgpu_buffer_rsrc_t g_rsrc = make_rsrc(a.q_and_gate + (qh * 2 + 1) * DIM, DIM * 4);
    auto split_of = [&](int i) { return SLOTS * PER_LANE * wave + slot + SLOTS * i; };
    floatx2 mlv[PER_LANE];
    floatx4 pv[PER_LANE];
#pragma unroll
    for (int i = 0; i < PER_LANE; i++) {
        const uint32_t c = split_of(i), record = c * a.heads + h;
        const bool need = c < (WAIT ? parts : a.nsplits) || (WAIT && c == fresh);
        mlv[i] = __builtin_bit_cast(floatx2, __builtin_amdgcn_raw_buffer_load_b64(ml_rsrc, need ? int(record * 8) : OOB, 0, 0));
        pv[i] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(o_rsrc, need ? int(record * (DIM * 4) + (DIMS * slice + 4 * quad) * 4) : OOB, 0, 0));
    }
    const float g = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(g_rsrc, tid < DIMS ? int(DIMS * slice + tid) * 4 : OOB, 0, 0));
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (!WAIT) splits_at_work();
    float m[PER_LANE], mx = NO_SCORE;
#pragma unroll
    for (int i = 0; i < PER_LANE; i++) {
        // (slots past the splits at work hold old values: dropped by select, never multiplied)
        const uint32_t c = split_of(i);
        const bool live = c < parts || c == fresh;
        m[i] = live ? mlv[i][0] : NO_SCORE;
        if (!live) mlv[i][1] = 0.0f, pv[i] = floatx4{0, 0, 0, 0};
        mx = fmaxf(mx, m[i]);
    }
    // the wave's maximum; like the sums, over the SLOTS slots, whose lanes are QUADS apart: with 4 quads two steps inside a row of 16
    // lanes, with 8 one, with 16 none, then two across rows.  The quads of a slot have the same m and l.
    if constexpr (QUADS <= 4) mx = fmaxf(mx, dpp<0x124>(mx));  // row_ror 4
    if constexpr (QUADS <= 8) mx = fmaxf(mx, dpp<0x128>(mx));  // row_ror 8
    mx = across_rows<16, 64>(mx, MaxOp());
    auto over_slots = [](float x) {
        if constexpr (QUADS <= 4) x += dpp<0x124>(x);
        if constexpr (QUADS <= 8) x += dpp<0x128>(x);
        return across_rows<16, 64>(x, SumOp());
    };
    float l = 0.0f;
    floatx4 o = {0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < PER_LANE; i++) {
        const float w = m[i] > 0.5f * NO_SCORE ? __builtin_amdgcn_exp2f(m[i] - mx) : 0.0f;
        l += w * mlv[i][1];
        o += pv[i] * w;
    }
    l = over_slots(l);
#pragma unroll
    for (int e = 0; e < 4; e++) o[e] = over_slots(o[e]);
    if (lane == 0) wave_m[wave] = mx, wave_l[wave] = l;
    if (lane < QUADS) wave_o[wave][lane] = o;  // (lane = quad)
    const float open = __builtin_amdgcn_rcpf(1.0f + __expf(-g));
    __syncthreads();
    if (tid < DIMS) {
        const float M = fmaxf(fmaxf(wave_m[0], wave_m[1]), fmaxf(wave_m[2], wave_m[3]));
        float total = 0.0f, sum = 0.0f;
#pragma unroll
        for (int w = 0; w < 4; w++) {
            const float f = wave_m[w] > 0.5f * NO_SCORE ? __builtin_amdgcn_exp2f(wave_m[w] - M) : 0.0f;
            total += f * wave_l[w];
            sum += f * wave_o[w][tid >> 2][tid & 3];
        }
        a.out[qh * DIM + DIMS * slice + tid] = sum * __builtin_amdgcn_rcpf(total) * open;
    }
}

// (more rows than one have a workgroup per CU, and half as many splits at most: run_attention)
template <int DIMS, bool WAIT>
int launch_reduce(hipStream_t stream, const ReduceArgs &a) {
    constexpr uint32_t ONE = DIMS / 16, HALF = MAX_SPLITS / 2;  // splits a lane takes, of 64
    static_assert(4 * (64 / (DIMS / 4)) * ONE == 64 && HALF <= 2 * 64 && MAX_SPLITS <= 4 * 64, "a split has a place");
    const dim3 grid(a.heads, a.rows, DIM / DIMS);
    if (a.nsplits <= 64) {
        launch(attention_reduce_kernel<DIMS, ONE, WAIT>, grid, 256, 0, stream, a);
    } else if (a.nsplits <= HALF) {
        launch(attention_reduce_kernel<DIMS, 2 * ONE, WAIT>, grid, 256, 0, stream, a);
    } else {
        SAETTA_REQUIRE(DIMS == 16, SAETTA_E_SHAPE, "merge of %u rows: %u splits, %u at most", a.rows, a.nsplits, HALF);
        if constexpr (DIMS == 16) launch(attention_reduce_kernel<DIMS, 4 * ONE, WAIT>, grid, 256, 0, stream, a);
    }
    return SAETTA_OK;
}

// ---- a token step of a cache of up to three splits: one launch --------------------------------------
//
// In a cache of up to 128 tokens (SAETTA_CHUNK) there is one split, so the step is neither work for the matrix cores nor anything to merge:
// three launches and their trips through memory.  Here a workgroup of 512 threads takes a q head of a row: it makes the head's query and,
// for itself, the new keys and values (make_rows; the first head's workgroup of a row stores them), and has the whole context beside them.
// Sixteen lanes hold a token, 16 dims each, keys and values alike; what is in the cache is asked for before anything is known, as
// far as the cache goes, and dropped by select where no token is.  Products and sums in f32, of halves as the cache gives them, of codes as numbers:
// a token's scale and bias are the same for a lane's sixteen and go into their sums (relative error against 64 bits 4e-7 to 9e-7, where the
// three launches have 8e-7 to 8e-6; each value made first 1.5e-7 to 2.8e-7 at 0.9 us more a 128 tokens).
// A layer's step, us, ten layers in a graph, three launches -> one:
//   cache  rows  in use   halves          8-bit           4-bit
//    128     1       4     8.7 ->  6.5     9.3 ->  6.7     9.4 ->  7.3
//                  119    11.3 ->  6.4    11.2 ->  6.8    11.1 ->  7.3
//            2     119    12.2 ->  6.6    11.6 ->  6.8    11.8 ->  7.3
//            8     119    17.4 ->  7.6    19.5 ->  8.1    20.2 ->  8.8
//    256     2       4     9.6 ->  8.3    10.2 ->  8.7    10.3 ->  9.6
//                  240    12.4 ->  9.3    11.8 ->  8.7    11.9 ->  9.6
//            3       4    10.4 ->  8.3    12.4 ->  8.7    12.7 ->  9.6
//                  240    14.6 ->  9.3    14.5 ->  8.7    14.5 ->  9.7
//    384     3       4    10.5 ->  9.9    12.5 -> 11.1    12.7 -> 11.7
//                  370    14.6 -> 11.5    14.5 -> 11.0    14.6 -> 11.7
//            4       4    11.0 -> 10.3    12.8 -> 11.6    13.1 -> 12.3
//            8       4    13.2 -> 10.7    14.2 -> 12.3    14.6 -> 13.0
//                  370    17.7 -> 12.3    19.5 -> 12.2    20.3 -> 13.0
// Ahead at every length, which matters: it is not known where a step is recorded.  Halves in more than 128 leave out the passes that have no
// token in use; without that, three rows of 384 take 11.6 at any length, behind the three launches up to some 100 tokens.  Codes, ahead as
// they are, don't: the branches would cost a full cache 3 to 5 % (8-bit, three rows of 384 at 370, 11.0 -> 11.3, 4-bit 11.7 -> 12.2; at 4 tokens 9.0 and
// 8.5); nor do halves in 128 (6.1 at 4 tokens, 6.5 at 119).
// What is left is the launch, the trips to the position and to the rows, the chain of the new rows (norm, rotation, quantizer) and 2 us per
// 128 tokens of cache, vector instructions.  Threads: 256 take 7.3 (halves, one row; 6.9 then) and 9.4 (eight; 8.1), 8.3 and 11.1 (8-bit; 7.8 and 9.2);
// 1024 7.5 and 8.2, 8.2 and 9.0.
// The line: two rows in a cache of 384 are even (halves 11.2 -> 11.4, 4-bit 11.7 -> 11.5).  One row would be ahead in one of 256 too (156 in use 10.2 -> 9.4 | 10.2 -> 8.6 |
// 10.4 -> 9.4) and five and more in one of 512: slower than it could be, for those steps are the three launches that test_gpu_token_step.py counts.
constexpr int ALONE_THREADS = 512, ALONE_PASS = ALONE_THREADS / 16;
uint32_t alone_tokens(uint32_t rows) { return rows == 1 ? SAETTA_CHUNK : rows == 2 ? 2 * SAETTA_CHUNK : 3 * SAETTA_CHUNK; }
struct AloneArgs {
    PartialArgs a;
    PrepArgs prep;
    float *out;
    uint32_t keep;  // 1: the step's partials go to its scratch too, everything in the first split (0.1 to 0.2 us)
};

template <int BITS, int TOKENS>
__global__ __launch_bounds__(ALONE_THREADS) void attention_token_alone_kernel(AloneArgs t) {
    constexpr int R = SAETTA_MAX_ROWS, WORDS = BITS / 2, PASSES = TOKENS / ALONE_PASS;  // WORDS: dwords of 16 values
    constexpr int ROWS_BYTES = R * 32 * 8 + (2 * R + 1) * DIM * 4;
    __shared__ __attribute__((aligned(16))) unsigned char rows_lds[ROWS_BYTES];
    __shared__ float score_lds[TOKENS + R], prob_lds[TOKENS + R];
    __shared__ __attribute__((aligned(16))) float o_lds[ALONE_THREADS / 64][DIM];
    const PartialArgs &a = t.a;
    const uint32_t tid = threadIdx.x, lane = tid & 63, part = tid & 15, sub = tid >> 4;  // part: dims 16 part .. + 15; sub: token of a pass
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t row = blockIdx.x / SAETTA_GQA_GROUP, head0 = blockIdx.x % SAETTA_GQA_GROUP, kv = blockIdx.y, kvh = a.kv_heads;
    const uint32_t position = a.tp->position, kv_len = a.tp->kv_len;
    const size_t of_head = size_t(row) * a.heads + kv * SAETTA_GQA_GROUP + head0;

    // ---- the cache ----
    struct Sixteen {
        uint32_t w[WORDS];
        uint32_t scale, bias;
    };
    Sixteen key[PASSES], value[PASSES];
    auto ask = [&](Sixteen &x, const void *data, const uint16_t *scales, const uint16_t *biases, uint32_t token) {
        const size_t at = size_t(token) * kvh + kv;
        const uint32_t *src = static_cast<const uint32_t *>(data) + at * (DIM * BITS / 32) + part * WORDS;
        if constexpr (BITS == 4) {
            const u32x2 v = *reinterpret_cast<const u32x2 *>(src);
            x.w[0] = v.x, x.w[1] = v.y;
        } else {
#pragma unroll
            for (int i = 0; i < WORDS / 4; i++) {
                const u32x4 v = reinterpret_cast<const u32x4 *>(src)[i];
                x.w[4 * i] = v.x, x.w[4 * i + 1] = v.y, x.w[4 * i + 2] = v.z, x.w[4 * i + 3] = v.w;
            }
        }
        if constexpr (BITS != 16) x.scale = scales[at * 4 + part / 4], x.bias = biases[at * 4 + part / 4];
    };
#pragma unroll
    for (int i = 0; i < PASSES; i++) ask(key[i], a.kdata, a.kscales, a.kbiases, min(uint32_t(i * ALONE_PASS) + sub, a.capacity - 1));  // (no branch: each would wait)
#pragma unroll
    for (int i = 0; i < PASSES; i++) ask(value[i], a.vdata, a.vscales, a.vbiases, min(uint32_t(i * ALONE_PASS) + sub, a.capacity - 1));
    const float gate = t.prep.q_and_gate[(of_head * 2 + 1) * DIM + (tid & (DIM - 1))];
    // (codes as numbers: scale and bias are the same for the sixteen, and go into their sums)
    auto sixteen = [](const Sixteen &x, float (&v)[16]) {
#pragma unroll
        for (int e = 0; e < 16; e++) {
            if constexpr (BITS == 16) {
                v[e] = half_bits_to_float(x.w[e / 2] >> (16 * (e & 1)));
            } else if constexpr (BITS == 8) {
                v[e] = float((x.w[e / 4] >> (8 * (e & 3))) & 255);
            } else {
                v[e] = float((((x.w[e / 8] >> (4 * (e & 1))) & 0x0f0f0f0fu) >> (8 * (e / 2 & 3))) & 255);
            }
        }
    };

    // ---- the new rows ----
    const auto [keys, values, queries] = make_rows<BITS, R>(a, t.prep, rows_lds, ALONE_THREADS / 64, row, 1, head0, 1, position);

    // ---- the scores, in units of log2(e): tokens of the cache that the row sees, then the new ones ----
    const uint32_t before = tokens_before(a, position, kv_len), fresh = tokens_new(a, position, kv_len, row);
    // (a decode sees min(kv_len, capacity) tokens: where the record says more than position + 1, rows past the new one too)
    const uint32_t past = a.decode_len ? min(kv_len, a.capacity) : 0;
    // (what is in use is told by the token's number all through, never by its score: a NaN in the cache is a NaN in the outputs)
    auto live = [&](uint32_t token) { return token < before || (token > position && token < past); };
    // (SKIP: a pass of tokens none of which is in use is left out)
    constexpr bool SKIP = BITS == 16 && TOKENS > SAETTA_CHUNK;
    const uint32_t end = max(before, past);
    auto in_use = [&](int pass) { return !SKIP || uint32_t(pass * ALONE_PASS) < end; };
    const float c = a.scale * 1.4426950408889634f;
    float q[16], q_sum = 0.0f;
#pragma unroll
    for (int e = 0; e < 16; e++) q[e] = queries[part * 16 + e] * c, q_sum += q[e];
#pragma unroll
    for (int i = 0; i < PASSES; i++) {
        const uint32_t token = i * ALONE_PASS + sub;
        float s = NO_SCORE;
        if (in_use(i)) {
            float k[16];
            sixteen(key[i], k);
            s = 0.0f;
#pragma unroll
            for (int e = 0; e < 16; e++) s += q[e] * k[e];
            if constexpr (BITS != 16) s = half_bits_to_float(key[i].scale) * s + half_bits_to_float(key[i].bias) * q_sum;
            s = group_reduce<16>(s, SumOp());
        }
        if (part == 0) score_lds[token] = live(token) ? s : NO_SCORE;
    }
    for (uint32_t n = wave; n < uint32_t(R); n += ALONE_THREADS / 64) {
        float s = NO_SCORE;
        if (n < fresh) {
            s = 0.0f;
#pragma unroll
            for (int i = 0; i < 4; i++) s += queries[64 * i + lane] * c * keys[n * DIM + 64 * i + lane];
            s = group_reduce<64>(s, SumOp());
        }
        if (lane == 0) score_lds[TOKENS + n] = s;
    }
    __syncthreads();

    // ---- the softmax: every wave for itself, the first hands the probabilities out ----
    constexpr int OLD = TOKENS / 64;
    constexpr float UNUSED = -1.0f;  // in a probability's place
    float s[OLD + 1], m = s[OLD] = lane < uint32_t(R) ? score_lds[TOKENS + lane] : NO_SCORE, l = 0.0f;
#pragma unroll
    for (int i = 0; i < OLD; i++) s[i] = score_lds[64 * i + lane], m = fmaxf(m, s[i]);
    m = group_reduce<64>(m, MaxOp());
#pragma unroll
    for (int i = 0; i <= OLD; i++) {
        const bool used = i < OLD ? live(64 * i + lane) : lane < fresh;
        s[i] = __builtin_amdgcn_exp2f(s[i] - m);
        l += used ? s[i] : 0.0f, s[i] = used ? s[i] : UNUSED;
    }
    l = group_reduce<64>(l, SumOp());
    if (wave == 0) {
#pragma unroll
        for (int i = 0; i < OLD; i++) prob_lds[64 * i + lane] = s[i];
        if (lane < uint32_t(R)) prob_lds[TOKENS + lane] = s[OLD];
    }
    __syncthreads();

    // ---- the values ----
    float o[16], biases = 0.0f;
#pragma unroll
    for (int e = 0; e < 16; e++) o[e] = 0.0f;
#pragma unroll
    for (int i = 0; i < PASSES; i++) {
        if (!in_use(i)) continue;
        float p = prob_lds[i * ALONE_PASS + sub];
        const bool used = !(p < 0.0f);  // (never a product with what lies where no token is)
        Sixteen &x = value[i];
        if constexpr (BITS == 16) {
#pragma unroll
            for (int w = 0; w < WORDS; w++) x.w[w] = used ? x.w[w] : 0;
        } else {
            biases += used ? p * half_bits_to_float(x.bias) : 0.0f;
            p = used ? p * half_bits_to_float(x.scale) : 0.0f;
        }
        float v[16];
        sixteen(x, v);
#pragma unroll
        for (int e = 0; e < 16; e++) o[e] += p * v[e];
    }
#pragma unroll
    for (int e = 0; e < 16; e++) o[e] = across_rows<16, 64>(o[e] + biases, SumOp());
    if (lane < 16) {
#pragma unroll
        for (int e = 0; e < 16; e += 4) *reinterpret_cast<floatx4 *>(&o_lds[wave][16 * part + e]) = floatx4{o[e], o[e + 1], o[e + 2], o[e + 3]};
    }
    __syncthreads();
    if (tid >= uint32_t(DIM)) return;
    float sum = 0.0f;
#pragma unroll
    for (int w = 0; w < ALONE_THREADS / 64; w++) sum += o_lds[w][tid];
    for (uint32_t n = 0; n < fresh; n++) sum += prob_lds[TOKENS + n] * values[n * DIM + tid];
    t.out[of_head * DIM + tid] = sum * __builtin_amdgcn_rcpf(l) * __builtin_amdgcn_rcpf(1.0f + __expf(-gate));
    if (!t.keep) return;
    const size_t first = size_t(row) * a.nsplits * a.heads + kv * SAETTA_GQA_GROUP + head0;
    a.part_o[first * DIM + tid] = sum;
    for (uint32_t split = 1; split < a.nsplits; split++) a.part_o[(first + split * a.heads) * DIM + tid] = 0.0f;
    if (tid < a.nsplits) *reinterpret_cast<floatx2 *>(a.part_ml + 2 * (first + tid * a.heads)) = tid == 0 ? floatx2{m, l} : floatx2{NO_SCORE, 0.0f};
}

uint32_t splits_for(uint32_t capacity, uint32_t wanted) {
    // Never more than the 128-token chunks of the capacity, so that scratch sized as
    // rows * ceil(capacity / 128) * heads partials is always enough.
    const uint32_t chunks = (capacity + SAETTA_CHUNK - 1) / SAETTA_CHUNK;
    uint32_t s = chunks < MAX_SPLITS ? chunks : MAX_SPLITS;
    if (wanted && wanted < s) s = wanted;
    return s ? s : 1;
}

// One to four rows over codes: from this capacity on the kernel whose loader waves keep a workgroup's share in
// LDS, the keys first, is the faster one at every length (one row, 8-bit, against the register kernels: 10.0
// against 11.0 us per layer at 4k tokens, 10.1 against 12.5 at 32k, 29.7 against 31.1 at 131k; shares of more
// than one round in alternate halves of LDS: 13.4 against 14.1 us at 40k for the ring of four 64-token slots
// that served there before, 28.3 against 29.7 at 150k, 4-bit, for the two-workgroups-per-CU kernel).
constexpr uint32_t KEYS_FIRST_FROM = 24 * 1024;
// Rows over a half cache that take the kernel with loader waves, at any capacity (figures there): two rows are one computing
// wave, which the register kernel's four are ahead of.
constexpr uint32_t HALF_ROWS_FROM = 3;
// Five rows and more take the store in, where their kernel has loader waves, from this capacity on.  This is no crossover: one launch
// is ahead in smaller caches too (6 rows at 300 tokens of 8192 13.7 -> 12.5 us a layer, at 30000 of 32768 29.3 -> 26.7), but in those a
// step of many rows is the three launches that test_gpu_token_step.py counts (at up to 40960 tokens).
constexpr uint32_t MANY_NEW_ROWS_FROM = 48 * 1024;

// Rows over codes that take the kernel with waves of their own (attention_partial_kernel_c), by the cache's capacity; us a
// layer in a plan with the store taken in, the kernel before it -> this one:
//   two rows from 48k: behind up to a length of 34k, where a share is a single round of the keys-first kernel (of 65536, 8-bit: 2000 13.4
//   -> 13.7, 12000 14.7 -> 15.6, 32768 17.4 -> 19.2; 4-bit 13.5 -> 13.9, 14.8 -> 15.5, 17.0 -> 18.9) and ahead from there (37000 21.8 ->
//   20.1, 44000 22.8 -> 21.2, 57123 26.6 -> 23.7; 20.8 -> 19.6, 21.7 -> 19.7, 26.4 -> 21.6; 131000 45.1 -> 30.6).  The length is not known
//   where a launch is recorded, and one launch cannot hold both (twelve waves of 168 registers, six of 256): over all lengths that a
//   cache has room for the two sides weigh the same at 48k.
//   three and four rows from 24k, at every length but a full 24k of 4-bit codes: 3 rows, 8-bit, 2000 17.5 -> 15.0, 12000 19.4 -> 18.4, 24400
//   21.7 -> 21.3, 32768 23.6 -> 22.7, 57123 35.7 -> 27.6; 4 rows, 4-bit, 19.0 -> 16.7, 21.3 -> 20.1, 22.9 -> 23.6, 25.0 -> 25.0, 36.7 -> 29.6
//   five rows and more: 6 rows, 8-bit, 300 16.8 -> 15.4, 12000 26.9 -> 25.7, 57123 47.1 -> 38; 8 rows 19.1 -> 15.6, 31.6 -> 28.6, 54.8 ->
//   42; 5 and 6 rows of 4-bit codes from 28k: 6 rows 4000 24.0 -> 22.7, 8000 24.9 -> 25.7, 20000 29.5 -> 29.3, 30000 34.8 -> 32.3
// Attention by itself has 128 splits for the context instead of 127 and less, and the keys-first kernel is further ahead in its
// single round: two rows from 64k (8-bit, 6000 11.7 -> 13.2, 32768 15.5 -> 17.5, 37000 20.0 -> 19.4, 57123 25.1 -> 22.1), four rows of 8
// bits from 36k (300 12.7 -> 11.2, 12000 18.1 -> 18.0, 24500 19.4 -> 20.1, 32768 20.7 -> 21.6, 34700 22.2 -> 23.4, 37000 26.7 -> 23.5); three
// rows (8-bit, 24500 18.3 -> 18.8, 32768 20.5 -> 20.5, 37000 25.8 -> 22.2) and 4-bit codes as above.
// It is ahead in larger caches still (4 rows, 8-bit, at 150000 tokens 66.5 -> 48.4, 8 rows 107 -> 79), but stops at 64k tokens, 2 to
// 4 rows of 4-bit codes at 128k, so that results stay what they were: the sums of the codes and of the biases nearly cancel, the
// more the longer the context, and the order in which 32-bit sums are taken shows as 4e-6 to 8e-6 of the results at 64000 tokens,
// 1.0e-5 to 1.5e-5 at 131000 (2 to 4 rows, 4-bit, 7e-6).  Either kernel is further than that from 64 bits.
constexpr bool code_rows(int bits, uint32_t rows, uint32_t capacity, bool with_store) {
    constexpr uint32_t K = 1024;
    const uint32_t few = rows == 2 ? (with_store ? 48 * K : 64 * K) : rows == 4 && bits == 8 && !with_store ? 36 * K : 24 * K;
    const uint32_t from = rows >= 7 || (rows >= 5 && bits == 8) ? 0 : rows >= 5 ? 28 * K : few;
    const uint32_t to = rows <= 4 && bits == 4 ? 128 * K : 64 * K;
    return bits != 16 && rows >= 2 && capacity >= from && capacity <= to;
}

// token: with the step before the scores taken in (nullptr: not)
template <int BITS, int TILES, bool PACKED>
void launch_partial(hipStream_t stream, const PartialArgs &a, bool one_per_cu, bool keys_first, const TokenArgs *token) {
    void (*kernel)(PartialArgs);
    int lds_bytes;
    const dim3 grid(a.nsplits, a.kv_heads);
    if constexpr (BITS == 16 && !PACKED && TILES >= 2) {
        if (keys_first) {
            using W = HalfRows<TILES>;
            if (token) launch(attention_token_kernel_h<TILES>, dim3(token->a.nsplits - 1 + a.rows, a.kv_heads), W::THREADS_, W::LDS_BYTES, stream, *token);
            else launch(attention_partial_kernel_h<TILES>, grid, W::THREADS_, W::LDS_BYTES, stream, a);
            return;
        }
    }
    if constexpr (BITS != 16 && !PACKED) {
        if (keys_first && code_rows(BITS, a.rows, a.capacity, token != nullptr)) {
            using W = CodeRows<BITS, TILES>;
            if (token) launch(attention_token_kernel_c<BITS, TILES>, dim3(token->a.nsplits - 1 + a.rows, a.kv_heads), W::THREADS_, W::LDS_BYTES, stream, *token);
            else launch(attention_partial_kernel_c<BITS, TILES>, grid, W::THREADS_, W::LDS_BYTES, stream, a);
            return;
        }
    }
    if constexpr (BITS != 16) {
        if (keys_first) {
            auto launch_rows = [&](auto rows_c) {
                constexpr int MR = decltype(rows_c)::value;
                using W = KeysFirst<BITS, MR>;
                if (token) launch(attention_token_kernel_s<BITS, MR>, dim3(token->a.nsplits, a.kv_heads), W::THREADS_, W::LDS_BYTES, stream, *token);
                else launch(attention_partial_kernel_s<BITS, MR>, grid, W::THREADS_, W::LDS_BYTES, stream, a);
            };
            if (a.rows == 1) launch_rows(std::integral_constant<int, 1>());
            else if (a.rows == 2) launch_rows(std::integral_constant<int, 2>());
            else if (a.rows == 3) launch_rows(std::integral_constant<int, 3>());
            else launch_rows(std::integral_constant<int, 4>());
            return;
        }
    }
    if constexpr (TILES == 1 && BITS != 16 && PACKED) {
        if (one_per_cu) {
            kernel = attention_partial_kernel_p<BITS>;
            lds_bytes = Shape<BITS, TILES, PACKED, ITB_ONE_PER_CU>::LDS_BYTES;
        } else {
            kernel = attention_partial_kernel_1<BITS>;
            lds_bytes = Shape<BITS, TILES, PACKED, ITB_TWO_PER_CU>::LDS_BYTES;
        }
    } else if constexpr (PACKED) {
        kernel = attention_partial_kernel_p<BITS>;  // f16 cache: its registers do not fit two waves
        lds_bytes = Shape<BITS, TILES, PACKED, ITB_ONE_PER_CU>::LDS_BYTES;
    } else {
        kernel = attention_partial_kernel_n<BITS, TILES>;
        lds_bytes = Shape<BITS, TILES, PACKED, itb_rows<TILES>()>::LDS_BYTES;
    }
    // (the dynamic LDS limit of every variant was raised in setup_decode)
    if (token) {
        const dim3 both(token->a.nsplits - 1 + a.rows * (SAETTA_GQA_GROUP / token->new_heads), a.kv_heads);
        if constexpr (PACKED) launch(attention_token_kernel_p<BITS>, both, THREADS, lds_bytes, stream, *token);
        else if constexpr (TILES <= 2) launch(attention_token_kernel_n<BITS, TILES>, both, THREADS, lds_bytes, stream, *token);
        return;
    }
    launch(kernel, grid, THREADS, lds_bytes, stream, a);
}

template <int BITS>
void launch_partial_rows(hipStream_t stream, const PartialArgs &a, bool one_per_cu, bool keys_first, const TokenArgs *token = nullptr) {
    if (a.rows == 1) {
        launch_partial<BITS, 1, true>(stream, a, one_per_cu, keys_first, token);
    } else if (a.rows == 2) {
        launch_partial<BITS, 1, false>(stream, a, one_per_cu, keys_first, token);
    } else if (a.rows <= 4) {
        launch_partial<BITS, 2, false>(stream, a, one_per_cu, keys_first, token);
    } else if (a.rows <= 6) {
        launch_partial<BITS, 3, false>(stream, a, one_per_cu, keys_first, token);
    } else {
        launch_partial<BITS, 4, false>(stream, a, one_per_cu, keys_first, token);
    }
}

// Whether the last two launches of a plan in the making are the step before the scores and the partial stage `a` of the
// same rows over the same buffers, so that the reduce stage about to be recorded makes them one layer's token step, which
// the kernels of TokenArgs do in one launch less.  They are written for 64 rotary dims and for what rope_angle and
// inverse_root take, and the new tokens take a split of their own: with fewer than 4 the context would be left with too few
// workgroups.  (The branch to the library's sine and cosine inside them was 1 to 1.6 % of a step at 32768 tokens of 8 bits,
// taken or not.)
// out: where the step is to be one launch, which then writes it (a cache of up to alone_tokens), else nullptr.
bool token_step(const LaunchList &list, const PartialArgs &a, int bits, const float *q_and_gate, const float *out, bool keys_first, TokenArgs &token) {
    const size_t n = list.launches.size();
    if (n < 2 || (!out && a.nsplits < 4)) return false;
    const LaunchRecord &before = list.launches[n - 2], &partial = list.launches[n - 1];
    if (before.kind != LAUNCH_PREP || partial.kind != LAUNCH_PARTIAL || int(before.bits) != bits || int(partial.bits) != bits || before.rows != a.rows) return false;
    const PartialArgs &b = list.arg<PartialArgs>(partial, 0);
    if (b.q != a.q || b.kdata != a.kdata || b.vdata != a.vdata || b.kscales != a.kscales || b.kbiases != a.kbiases || b.vscales != a.vscales || b.vbiases != a.vbiases ||
        b.part_o != a.part_o || b.part_ml != a.part_ml || b.heads != a.heads || b.kv_heads != a.kv_heads || b.capacity != a.capacity || b.scale != a.scale ||
        b.rows != a.rows || b.nsplits != a.nsplits || b.tp != a.tp || b.decode_len != a.decode_len) return false;
    const PrepArgs prep = list.arg<PrepArgs>(before, 0);
    const bool cache = bits == 16 ? prep.keys_half == a.kdata && prep.values_half == a.vdata
                                  : prep.kq.data == a.kdata && prep.kq.scales == a.kscales && prep.kq.biases == a.kbiases && prep.vq.data == a.vdata &&
                                        prep.vq.scales == a.vscales && prep.vq.biases == a.vbiases;
    if (!(cache && prep.q_out == a.q && prep.q_and_gate == q_and_gate && prep.tp == a.tp && prep.capacity == a.capacity && prep.p.heads == a.heads &&
          prep.p.kv_heads == a.kv_heads && prep.p.half_dims == 32 && prep.p.log2_theta >= 0.0f && prep.p.eps >= INVERSE_ROOT_FROM &&
          aligned(prep.q_and_gate, 16) && aligned(prep.q_norm, 16))) return false;
    // One launch only where its buffers lie apart.  In three, the step's inputs are done with when the store has run, so a
    // program may write the key back in the place of `k` (the reference's in-place key) or lay the partials over any of
    // them; in one, workgroups still read the inputs while others write.
    const size_t row_kv = size_t(a.rows) * a.kv_heads * DIM * sizeof(float), row_q = size_t(a.rows) * a.heads * DIM * sizeof(float);
    const size_t partials = size_t(a.rows) * a.nsplits * a.heads, cached = size_t(a.capacity) * a.kv_heads * DIM;
    const size_t data = cached * size_t(bits) / 8, scales = bits == 16 ? 0 : cached / SAETTA_QUANT_GROUP * sizeof(uint16_t);
    const Span inputs[] = {{prep.q_and_gate, 2 * row_q}, {prep.k, row_kv}, {prep.v, row_kv}, {prep.q_norm, DIM * sizeof(float)},
                           {prep.k_norm, DIM * sizeof(float)}, {a.tp, sizeof(saetta_token_params)}},
               outputs[] = {{prep.k_back, prep.k_back ? row_kv : 0}, {prep.q_out, row_q}, {a.part_o, partials * DIM * sizeof(float)},
                            {a.part_ml, partials * 2 * sizeof(float)}, {a.kdata, data}, {a.vdata, data}, {a.kscales, scales},
                            {a.kbiases, scales}, {a.vscales, scales}, {a.vbiases, scales}, {out, out ? row_q : 0}};
    for (const Span &o : outputs) {
        for (const Span &i : inputs) {
            if (!apart(o, i)) return false;
        }
        for (const Span &other : outputs) {
            if (&other != &o && !apart(o, other)) return false;
        }
    }
    token = TokenArgs{a, prep, SAETTA_GQA_GROUP};
    if (out) return true;
    const uint32_t room = MAX_SPLITS / 2;  // workgroups of a kv head, one to a CU
    if (keys_first && (bits == 16 || code_rows(bits, a.rows, a.capacity, true))) {
        // a workgroup per new row, for which a full context gives up CUs (two rows to one: 6 rows at 57123 tokens 36.2 against
        // 35.5 us a layer)
        if (a.rows > NEW_ROWS && a.capacity < MANY_NEW_ROWS_FROM) return false;
        token.a.nsplits = min(a.nsplits, room - a.rows + 1);
    } else if (!keys_first) {
        // more rows than four: the workgroups of the new rows need longer than the launch takes (18.7 against 18.2 us per
        // layer at 8 rows and 300 tokens, f16)
        if (a.rows > NEW_ROWS) return false;
        // as many splits as before, one of them the new tokens'.  Their workgroups beside the context's: two heads to one
        // while all fit one to a CU, a whole row to one where the context gives up CUs for them.
        if (a.nsplits - 1 + 4 * a.rows <= room) token.new_heads = 2;
        else if (a.nsplits - 1 + a.rows > room) token.a.nsplits = room - a.rows + 1;
    }
    return true;
}

// A further reduce stage is recorded over the scratch of `a`: of the partials as the step that was the last to use it divides them, where
// that is a step in fewer launches.  One in a single launch leaves them there only for this.
void read_again(LaunchList &list, const PartialArgs &a, uint32_t &nsplits, uint32_t &last_is_new) {
    for (size_t n = list.launches.size(); n-- > 0;) {
        const LaunchRecord &r = list.launches[n];
        if (r.kind == LAUNCH_PARTIAL && list.arg<PartialArgs>(r, 0).part_o == a.part_o) return;
        if (r.kind == LAUNCH_REDUCE && list.arg<ReduceArgs>(r, 0).part_o == a.part_o) {
            const ReduceArgs &b = list.arg<ReduceArgs>(r, 0);
            if (b.last_is_new && b.rows == a.rows && b.heads == a.heads && b.capacity == a.capacity) nsplits = b.nsplits, last_is_new = 1;
            return;
        }
        if (r.kind == LAUNCH_ALONE && list.arg<AloneArgs>(r, 0).a.part_o == a.part_o) {
            list.arg<AloneArgs>(r, 0).keep = 1;
            return;
        }
    }
}

int run_attention(hipStream_t stream, int bits, const float *q, const void *kdata, const void *vdata,
                  const uint16_t *ks, const uint16_t *kz, const uint16_t *vs, const uint16_t *vz,
                  float *part_o, float *part_ml, const float *q_and_gate, float *out, uint32_t heads,
                  uint32_t kv_heads, uint32_t capacity, float scale, uint32_t rows, uint32_t wanted_splits,
                  const saetta_token_params *d_tp, bool decode_len, uint32_t stages, const char *what) {
    SAETTA_REQUIRE(bits == 16 || bits == 8 || bits == 4, SAETTA_E_BITS, "%s: bits %d", what, bits);
    SAETTA_REQUIRE(kv_heads > 0 && heads == kv_heads * SAETTA_GQA_GROUP, SAETTA_E_SHAPE,
                   "%s needs 8 q heads per kv head (heads %u, kv heads %u)", what, heads, kv_heads);
    SAETTA_REQUIRE(rows >= 1 && rows <= SAETTA_MAX_ROWS, SAETTA_E_SHAPE, "%s: %u rows (1..8)", what, rows);
    // Byte offsets into the cache are 32-bit: capacity * kv_heads * 512 B (the f16 row) must fit.
    SAETTA_REQUIRE(capacity > 0 && uint64_t(capacity) * kv_heads * 512 < (uint64_t(1) << 31), SAETTA_E_SHAPE,
                   "%s: capacity %u out of range", what, capacity);
    // Whole 16-token blocks are read: the last one must lie inside the cache (the reference's caches
    // are multiples of 128, src/gpu_layers.rs:199).
    SAETTA_REQUIRE(capacity % BLOCK == 0, SAETTA_E_SHAPE, "%s: capacity %u is not a multiple of 16", what, capacity);
    SAETTA_REQUIRE(q && kdata && vdata && part_o && part_ml && q_and_gate && out && d_tp, SAETTA_E_NULL,
                   "%s: null buffer", what);
    SAETTA_REQUIRE(bits == 16 || (ks && kz && vs && vz), SAETTA_E_NULL, "%s: null scales or biases", what);
    SAETTA_REQUIRE(aligned(q, 16) && aligned(kdata, 16) && aligned(vdata, 16) && aligned(part_o, 16) &&
                       aligned(part_ml, 8) && aligned(q_and_gate, 4) && aligned(out, 4),
                   SAETTA_E_ALIGN, "%s: q, cache and scratch must be 16-byte aligned", what);
    SAETTA_REQUIRE(bits == 16 || (aligned(ks, 8) && aligned(kz, 8) && aligned(vs, 8) && aligned(vz, 8)),
                   SAETTA_E_ALIGN, "%s: scales and biases must be 8-byte aligned", what);
    if (int rc = ensure_device()) return rc;
    uint32_t nsplits = splits_for(capacity, wanted_splits);
    // One to four rows over codes in a cache of 24k tokens and more go to the kernel with loader waves, a
    // one-workgroup-per-CU kernel at every length: a share of up to 17 blocks (the kernel sees the length
    // when it runs: a step at 32k tokens is one round in a cache of any size) is one round, a longer one
    // rounds of 8 blocks (three and four rows: 12).  Three rows and more over halves, and the rows over codes that
    // code_rows names, go to the kernels with a wave per tile.  SAETTA_STAGE_NO_LOADERS keeps to the register kernels (the caller's choice of
    // kernel family, as DecodeAttention.kernel is in the reference, src/attention.rs:36-38).
    // The register kernels: one workgroup per CU (half as many splits, each twice as long) or two.  Two
    // rows and more and a half cache need the whole register file anyway; one row over codes fits two
    // workgroups per CU, which pays only for long contexts: up to 64k tokens the shorter merge of half as
    // many partials is worth more (measured: 19.4 against 20.6 us per layer at 32k, 28.3 against 29.7 at
    // 64k, but 44 against 35 at 146k, 4-bit).  Both stages of a call derive the same number from the same arguments; where
    // a plan's reduce stage makes a token step of the launches before it, the number is the token step's.
    const bool loaders = bits == 16 ? rows >= HALF_ROWS_FROM : code_rows(bits, rows, capacity, false) || (rows <= 4 && capacity >= KEYS_FIRST_FROM);
    const bool keys_first = loaders && !(stages & SAETTA_STAGE_NO_LOADERS);
    const bool one_per_cu = rows >= 2 || bits == 16 || capacity <= 80 * 1024 || keys_first;
    if (one_per_cu && nsplits > MAX_SPLITS / 2) nsplits = MAX_SPLITS / 2;
    const PartialArgs a{q,     kdata,    vdata,    ks,    kz,   vs,      vz,   part_o, part_ml,
                        heads, kv_heads, capacity, scale, rows, nsplits, d_tp, decode_len ? 1u : 0u, device_status_word()};
    auto partial = [&](const TokenArgs *token) {
        if (bits == 8) {
            launch_partial_rows<8>(stream, a, one_per_cu, keys_first, token);
        } else if (bits == 4) {
            launch_partial_rows<4>(stream, a, one_per_cu, keys_first, token);
        } else {
            launch_partial_rows<16>(stream, a, one_per_cu, keys_first, token);
        }
    };
    if (stages & SAETTA_STAGE_PARTIAL) {
        partial(nullptr);
        tag_launch(LAUNCH_PARTIAL, uint32_t(bits), rows);
    }
    if (stages & SAETTA_STAGE_REDUCE) {
        uint32_t last_is_new = 0;
        if (LaunchList *list = recording()) {
            TokenArgs token;
            if (capacity <= alone_tokens(rows) && token_step(*list, a, bits, q_and_gate, out, keys_first, token)) {
                list->launches.pop_back(), list->launches.pop_back();
                const AloneArgs alone{token.a, token.prep, out, 0};
                auto of = [&](auto tokens) {
                    constexpr int TOKENS = decltype(tokens)::value;
                    launch(bits == 16 ? attention_token_alone_kernel<16, TOKENS> : bits == 8 ? attention_token_alone_kernel<8, TOKENS> : attention_token_alone_kernel<4, TOKENS>,
                           dim3(rows * SAETTA_GQA_GROUP, kv_heads), ALONE_THREADS, 0, stream, alone);
                };
                if (capacity <= SAETTA_CHUNK) of(std::integral_constant<int, SAETTA_CHUNK>{});
                else if (capacity <= 2 * SAETTA_CHUNK) of(std::integral_constant<int, 2 * SAETTA_CHUNK>{});
                else of(std::integral_constant<int, 3 * SAETTA_CHUNK>{});
                tag_launch(LAUNCH_ALONE, uint32_t(bits), rows);
                return launch_status(what);
            }
            if (one_per_cu && token_step(*list, a, bits, q_and_gate, nullptr, keys_first, token)) {
                list->launches.pop_back(), list->launches.pop_back();
                partial(&token);
                last_is_new = 1;
                nsplits = token.a.nsplits;
            } else {
                read_again(*list, a, nsplits, last_is_new);
            }
        }
        ReduceArgs r{part_o, part_ml, q_and_gate, out, heads, capacity, nsplits, rows, d_tp, decode_len ? 1u : 0u, last_is_new};
        if (int rc = rows == 1 ? launch_reduce<16, false>(stream, r) : rows == 2 ? launch_reduce<32, false>(stream, r) : launch_reduce<64, true>(stream, r)) return rc;
        tag_launch(LAUNCH_REDUCE, uint32_t(bits), rows);
    }
    return launch_status(what);
}

}  // namespace

namespace {
template <int BITS, int TILES, bool PACKED, int ITB, class Args>
int raise_lds(void (*kernel)(Args)) {
    static_assert(Shape<BITS, TILES, PACKED, ITB>::LDS_BYTES <= 160 * 1024, "LDS of a CU");
    if (Shape<BITS, TILES, PACKED, ITB>::LDS_BYTES <= 48 * 1024) return 0;
    return int(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                   Shape<BITS, TILES, PACKED, ITB>::LDS_BYTES));
}
template <int BITS, int M>
int raise_lds_keys_first() {
    if (int rc = int(hipFuncSetAttribute(reinterpret_cast<const void *>(attention_token_kernel_s<BITS, M>), hipFuncAttributeMaxDynamicSharedMemorySize,
                                         KeysFirst<BITS, M>::LDS_BYTES))) return rc;
    return int(hipFuncSetAttribute(reinterpret_cast<const void *>(attention_partial_kernel_s<BITS, M>),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, KeysFirst<BITS, M>::LDS_BYTES));
}
template <int BITS, int TILES>
int raise_lds_code_rows_of() {
    if (int rc = int(hipFuncSetAttribute(reinterpret_cast<const void *>(attention_token_kernel_c<BITS, TILES>), hipFuncAttributeMaxDynamicSharedMemorySize,
                                         CodeRows<BITS, TILES>::LDS_BYTES))) return rc;
    return int(hipFuncSetAttribute(reinterpret_cast<const void *>(attention_partial_kernel_c<BITS, TILES>), hipFuncAttributeMaxDynamicSharedMemorySize,
                                   CodeRows<BITS, TILES>::LDS_BYTES));
}
template <int BITS>
int raise_lds_code_rows() {
    if (int rc = raise_lds_code_rows_of<BITS, 1>()) return rc;
    if (int rc = raise_lds_code_rows_of<BITS, 2>()) return rc;
    if (int rc = raise_lds_code_rows_of<BITS, 3>()) return rc;
    return raise_lds_code_rows_of<BITS, 4>();
}
template <int TILES>
int raise_lds_half_rows() {
    if (int rc = int(hipFuncSetAttribute(reinterpret_cast<const void *>(attention_token_kernel_h<TILES>), hipFuncAttributeMaxDynamicSharedMemorySize,
                                         HalfRows<TILES>::LDS_BYTES))) return rc;
    return int(hipFuncSetAttribute(reinterpret_cast<const void *>(attention_partial_kernel_h<TILES>), hipFuncAttributeMaxDynamicSharedMemorySize,
                                   HalfRows<TILES>::LDS_BYTES));
}
template <int BITS>
int raise_lds_of_bits() {
    if (int rc = raise_lds<BITS, 1, true, ITB_ONE_PER_CU>(attention_partial_kernel_p<BITS>)) return rc;
    if (int rc = raise_lds<BITS, 1, true, ITB_ONE_PER_CU>(attention_token_kernel_p<BITS>)) return rc;
    if (int rc = raise_lds<BITS, 1, false, itb_rows<1>()>(attention_token_kernel_n<BITS, 1>)) return rc;
    if (int rc = raise_lds<BITS, 2, false, itb_rows<2>()>(attention_token_kernel_n<BITS, 2>)) return rc;
    if (int rc = raise_lds<BITS, 1, false, itb_rows<1>()>(attention_partial_kernel_n<BITS, 1>)) return rc;
    if (int rc = raise_lds<BITS, 2, false, itb_rows<2>()>(attention_partial_kernel_n<BITS, 2>)) return rc;
    if (int rc = raise_lds<BITS, 3, false, itb_rows<3>()>(attention_partial_kernel_n<BITS, 3>)) return rc;
    return raise_lds<BITS, 4, false, itb_rows<4>()>(attention_partial_kernel_n<BITS, 4>);
}
}  // namespace

int setup_decode() {
    if (int rc = load_kernel(reinterpret_cast<const void *>(attention_reduce_kernel<16, 1, false>))) return rc;
    {
        // (runs once per device, with that device current)
        int dev = 0;
        if (hipError_t e = hipGetDevice(&dev)) return int(e);
        if (dev < 0 || dev >= STATIC_MAX_DEVICES) return int(hipErrorInvalidDevice);
        float *ptr = nullptr;
        if (hipError_t e = hipGetSymbolAddress(reinterpret_cast<void **>(&ptr), HIP_SYMBOL(scratch))) return int(e);
        g_static_scratch[dev] = ptr;
    }
    if (int rc = raise_lds_keys_first<8, 1>()) return rc;
    if (int rc = raise_lds_keys_first<8, 2>()) return rc;
    if (int rc = raise_lds_keys_first<8, 3>()) return rc;
    if (int rc = raise_lds_keys_first<8, 4>()) return rc;
    if (int rc = raise_lds_keys_first<4, 1>()) return rc;
    if (int rc = raise_lds_keys_first<4, 2>()) return rc;
    if (int rc = raise_lds_keys_first<4, 3>()) return rc;
    if (int rc = raise_lds_keys_first<4, 4>()) return rc;
    if (int rc = raise_lds_code_rows<8>()) return rc;
    if (int rc = raise_lds_code_rows<4>()) return rc;
    if (int rc = raise_lds_half_rows<2>()) return rc;
    if (int rc = raise_lds_half_rows<3>()) return rc;
    if (int rc = raise_lds_half_rows<4>()) return rc;
    if (int rc = raise_lds_of_bits<8>()) return rc;
    if (int rc = raise_lds_of_bits<4>()) return rc;
    if (int rc = raise_lds_of_bits<16>()) return rc;
    if (int rc = raise_lds<8, 1, true, ITB_TWO_PER_CU>(attention_partial_kernel_1<8>)) return rc;
    return raise_lds<4, 1, true, ITB_TWO_PER_CU>(attention_partial_kernel_1<4>);
}
}  // namespace saetta

using namespace saetta;

extern "C" size_t saetta_part_o_bytes(uint32_t heads, uint32_t capacity, uint32_t rows) {
    return size_t(rows) * splits_for(capacity, 0) * heads * DIM * sizeof(float);
}

extern "C" size_t saetta_part_ml_bytes(uint32_t heads, uint32_t capacity, uint32_t rows) {
    return size_t(rows) * splits_for(capacity, 0) * heads * 2 * sizeof(float);
}

extern "C" int saetta_attn_decode(saetta_stream_t stream, const float *q, const uint16_t *keys,
                                  const uint16_t *values, float *part_o, float *part_ml,
                                  const float *q_and_gate, float *out, saetta_decode_params p,
                                  const saetta_token_params *d_tp, uint32_t stages) {
    return run_attention(as_stream(stream), 16, q, keys, values, nullptr, nullptr, nullptr, nullptr, part_o,
                         part_ml, q_and_gate, out, p.heads, p.kv_heads, p.capacity, p.scale, 1, 0, d_tp,
                         true, stages, "attn_decode");
}

extern "C" int saetta_attn_decode_quant(saetta_stream_t stream, int bits, const float *q,
                                        saetta_quant_rows keys, saetta_quant_rows values, float *part_o,
                                        float *part_ml, const float *q_and_gate, float *out,
                                        saetta_decode_params p, const saetta_token_params *d_tp,
                                        uint32_t stages) {
    SAETTA_REQUIRE(bits == 8 || bits == 4, SAETTA_E_BITS, "attn_decode_quant: bits %d (8 or 4)", bits);
    return run_attention(as_stream(stream), bits, q, keys.data, values.data, keys.scales, keys.biases,
                         values.scales, values.biases, part_o, part_ml, q_and_gate, out, p.heads,
                         p.kv_heads, p.capacity, p.scale, 1, 0, d_tp, true, stages, "attn_decode_quant");
}

extern "C" size_t saetta_static_scratch_bytes(void) { return sizeof(float) * (STATIC_PART_O_FLOATS + STATIC_PART_ML_FLOATS); }

extern "C" int saetta_attn_decode_quant_static(saetta_stream_t stream, int bits, const float *q,
                                               saetta_quant_rows keys, saetta_quant_rows values,
                                               const float *q_and_gate, float *out, saetta_decode_params p,
                                               const saetta_token_params *d_tp, uint32_t stages) {
    SAETTA_REQUIRE(bits == 8 || bits == 4, SAETTA_E_BITS, "attn_decode_quant_static: bits %d (8 or 4)", bits);
    // What the partials of this launch need against what the static array holds (the number of
    // splits never exceeds 256, so only the heads can outgrow it).
    const size_t need = saetta_part_o_bytes(p.heads, p.capacity, 1) + saetta_part_ml_bytes(p.heads, p.capacity, 1);
    SAETTA_REQUIRE(p.heads <= STATIC_MAX_HEADS && need <= saetta_static_scratch_bytes(), SAETTA_E_SCRATCH,
                   "attn_decode_quant_static: %u heads need %zu bytes of partials, the static scratch holds %zu "
                   "(up to %u heads); use saetta_attn_decode_quant with scratch of the caller's",
                   p.heads, need, saetta_static_scratch_bytes(), STATIC_MAX_HEADS);
    if (int rc = ensure_device()) return rc;
    int dev = 0;
    if (hipError_t e = hipGetDevice(&dev)) return fail(int(e), "attn_decode_quant_static: %s", hipGetErrorString(e));
    float *part_o = (dev >= 0 && dev < STATIC_MAX_DEVICES) ? g_static_scratch[dev] : nullptr;
    SAETTA_REQUIRE(part_o, SAETTA_E_DEVICE, "attn_decode_quant_static: no static scratch on device %d", dev);
    return run_attention(as_stream(stream), bits, q, keys.data, values.data, keys.scales, keys.biases,
                         values.scales, values.biases, part_o, part_o + STATIC_PART_O_FLOATS, q_and_gate, out,
                         p.heads, p.kv_heads, p.capacity, p.scale, 1, 0, d_tp, true, stages,
                         "attn_decode_quant_static");
}

extern "C" int saetta_attn_rows(saetta_stream_t stream, const float *q, const uint16_t *keys,
                                const uint16_t *values, float *part_o, float *part_ml,
                                const float *q_and_gate, float *out, saetta_rows_params p,
                                const saetta_token_params *d_tp, uint32_t stages) {
    return run_attention(as_stream(stream), 16, q, keys, values, nullptr, nullptr, nullptr, nullptr, part_o,
                         part_ml, q_and_gate, out, p.heads, p.kv_heads, p.capacity, p.scale, p.rows,
                         p.splits, d_tp, false, stages, "attn_rows");
}

extern "C" int saetta_attn_rows_quant(saetta_stream_t stream, int bits, const float *q,
                                      saetta_quant_rows keys, saetta_quant_rows values, float *part_o,
                                      float *part_ml, const float *q_and_gate, float *out,
                                      saetta_rows_params p, const saetta_token_params *d_tp,
                                      uint32_t stages) {
    SAETTA_REQUIRE(bits == 8 || bits == 4, SAETTA_E_BITS, "attn_rows_quant: bits %d (8 or 4)", bits);
    return run_attention(as_stream(stream), bits, q, keys.data, values.data, keys.scales, keys.biases,
                         values.scales, values.biases, part_o, part_ml, q_and_gate, out, p.heads,
                         p.kv_heads, p.capacity, p.scale, p.rows, p.splits, d_tp, false, stages,
                         "attn_rows_quant");
}
