// Verify rows (3..8) over a half cache: one wave per tile of 16 (row, head) pairs, loader waves in front of them.
// Included by decode.hip, inside its namespace.
//
// What bounds it: the cache's bytes, 2 KB a token and kv head, then the partials (48 KB a workgroup for six rows).  In
// attention_partial_kernel_n four waves load, score, exponentiate and multiply in common phases, one wave per SIMD, and
// each of these is on the path of the next.  Here they run side by side:
//  * two loader waves stream slots of 32 tokens (16 KB of keys, then 16 KB of values) into a ring of four places in LDS
//    (global_load_lds_dwordx4, no registers), so up to 128 KB per CU are on their way at any time;
//  * a computing wave takes every slot for its tile and needs no other wave: S^T = K Q^T leaves four tokens of one (row,
//    head) pair in a lane, which is the operand that O^T += V^T P^T wants if the 32 tokens of its k index are taken in that
//    order, and ds_read_b64_tr_b16 hands out the values transposed in any order of tokens: the probabilities never leave the
//    registers, maximum, sum and rescaling are per lane, no value is permuted.
// The waves meet through counters in LDS (see attention_partial_kernel_s): per place, the loads that have landed and the
// waves that are through with the keys, and with the values.
// Rows in LDS are whole token rows of 512 bytes, their 16-byte pieces (keys) or 32-byte chunks (values) at places
// exclusive-or'ed with the token's number: the 16 tokens of a read then fall on different banks, and a load instruction
// still brings two whole rows of the cache.
// Measured per layer in a plan, ten layers in a graph, attention_partial_kernel_n -> this: 6 rows at 57123 tokens 46.8 ->
// 35.8 us, of which 2.7 the store taken in (a stream of the same loads without the products, 12 MB of partials and the merge
// are 36.1 with it apart), at 12000 24.6 -> 21.7, 300 15.0 -> 13.4; 8 rows 51.2 -> 38.2, 27.1 -> 24.7, 17.1 -> 15.0; 3 rows
// 37.4 -> 32.8, 18.6 -> 17.5, 11.7 -> 10.0; 4 rows at 200000 tokens 96.5 -> 82.  Two rows, one computing wave, are behind:
// 30.7 -> 32.4 at 57123.  Error against 64 bits, rel, means of six seeds: 6 rows at 57123 tokens 4.4e-7 -> 4.3e-7, 3 at
// 200000 5.8e-7 -> 5.6e-7, 5 at 700 3.2e-7 -> 2.9e-7.
// Tried: two computing waves a tile on alternate slots (6 rows 39.4: two places are held instead of one, so less is on its
// way); the next slot's scores beside a slot's exponentials (even at 57123 tokens, 23.6 against 22.2 at 12000); partials
// through LDS, a kilobyte a store (even).  The operands of a slot are asked for four at a time, one lot ahead of the
// products: left to the compiler every read stood in front of its product (8 rows 43.6 instead of 38.6).
template <int TILES>
struct HalfRows {
    static constexpr int COMPUTE = TILES, LOADERS = 2;         // waves
    static constexpr int THREADS_ = (COMPUTE + LOADERS) * 64;
    static constexpr int ROW = DIM * 2;
    static constexpr int SLOT_TOKENS = 2 * BLOCK, PART = SLOT_TOKENS * ROW, SLOT = 2 * PART;  // keys, then values
    static constexpr int PLACES = 4;
    static constexpr int LOADS = PART / 1024;                  // load instructions of a slot's keys, and of its values
    static_assert(2 * LOADS * PLACES / LOADERS <= 64, "a loader's requests out at once");
    // LDS map, in bytes
    static constexpr int SYNC_OFF = PLACES * SLOT;             // counters, u32
    static constexpr int ROPE_OFF = SYNC_OFF + 128;            // [computing wave][row of the tile][32] sine, cosine
    static constexpr int LDS_BYTES = ROPE_OFF + COMPUTE * 512;
    static constexpr int C_KEYS = 0, C_VALUES = 4;             // [place]: slots whose keys | values have landed there
    static constexpr int C_KFREE = 8, C_VFREE = 12;            // [place]: computing waves through with a slot's keys | values
    static constexpr uint32_t SPIN_LIMIT = 1u << 20;
    static_assert(LDS_BYTES <= 160 * 1024, "LDS of a CU");
    static_assert(SAETTA_MAX_ROWS * 32 * 8 + SAETTA_MAX_ROWS * 10 * DIM * 4 <= LDS_BYTES, "the new rows' workgroup fits");
};
// A row's maximum is followed only when it has grown by this much (log2): until then its probabilities are up to twice
// P_UP and the sums so far need no rescaling.  It is followed in whole numbers: what is rescaled, and what
// the merge multiplies a split with, is a power of two then, and the exponentials' arguments are rounded once.
constexpr float MAX_SLACK = 1.0f;

template <int TILES, bool PREP>
__device__ __forceinline__ void attention_half_rows_body(const PartialArgs &a, const PrepArgs *prep) {
    using W = HalfRows<TILES>;
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds_raw[];
    const uint32_t lane = threadIdx.x & 63, n = lane & 15, j = lane >> 4;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t split = blockIdx.x, kv = blockIdx.y, kvh = a.kv_heads;
    uint32_t *sync_lds = reinterpret_cast<uint32_t *>(lds_raw + W::SYNC_OFF);
    const uint32_t lds0 = uint32_t(reinterpret_cast<uintptr_t>(lds_raw));
    const uint32_t context_splits = PREP ? a.nsplits - 1 : a.nsplits;
    if constexpr (PREP) {
        if (split >= context_splits) {
            new_rows<16, 2 * TILES>(a, *prep, lds_raw, W::COMPUTE + W::LOADERS, split - context_splits, 1, 0, SAETTA_GQA_GROUP);
            return;
        }
    }
    const uint32_t position = a.tp->position, kv_len = a.tp->kv_len;
    const uint32_t real_rows = a.rows * 8;  // (row, head) pairs of this kv head
    const uint32_t tile = wave;  // of a computing wave
    // ---- a computing wave's query values, requested before anything else: k-step s of lane (n, j) is dims 32 s + 8 j .. + 7
    // of pair 16 tile + n (past the last pair: the last one again, whose results nobody stores) ----
    const uint32_t pair = min(16 * tile + n, real_rows - 1);
    float q[8][8];
    if (wave < uint32_t(W::COMPUTE)) {
        const size_t of_head = size_t(pair >> 3) * a.heads + kv * 8 + (pair & 7);
        const float *src = (PREP ? prep->q_and_gate + of_head * 2 * DIM : a.q + of_head * DIM) + 8 * j;
#pragma unroll
        for (int s = 0; s < 8; s++) {
            const float4 f0 = *reinterpret_cast<const float4 *>(src + 32 * s), f1 = *reinterpret_cast<const float4 *>(src + 32 * s + 4);
            q[s][0] = f0.x, q[s][1] = f0.y, q[s][2] = f0.z, q[s][3] = f0.w, q[s][4] = f1.x, q[s][5] = f1.y, q[s][6] = f1.z, q[s][7] = f1.w;
        }
    }
    if (threadIdx.x < 16) sync_lds[threadIdx.x] = 0;
    __syncthreads();

    // ---- the context and this workgroup's share of it, as in attention_partial_body ----
    const uint32_t max_len = PREP ? tokens_before(a, position, kv_len) : min(position + a.rows, a.capacity);
    const uint32_t nblocks = (max_len + BLOCK - 1) / BLOCK;
    uint32_t blk_begin = split, blk_end = split + 1;
    if (nblocks <= context_splits) {
        if (split >= nblocks) return;
    } else {
        blk_begin = split * nblocks / context_splits;
        blk_end = (split + 1) * nblocks / context_splits;
    }
    const uint32_t first_tok = blk_begin * BLOCK, limit = min(max_len, blk_end * BLOCK);  // tokens of this share
    const uint32_t slots = (limit - first_tok + W::SLOT_TOKENS - 1) / W::SLOT_TOKENS;
    // four splits in a row start a quarter of their share apart (see attention_partial_body)
    const uint32_t first_slot = (split & 3) * slots / 4;
    auto start_of = [&](uint32_t u) {
        const uint32_t at = u + first_slot < slots ? u + first_slot : u + first_slot - slots;
        return first_tok + at * W::SLOT_TOKENS;
    };
    LdsCounters<W::SPIN_LIMIT, 0x200u> sync{sync_lds, lane};

    floatx4 acc[16];  // O^T: dims 16 T + 4 j .. + 3 of the lane's pair
    float m_run = NO_SCORE, l_run = 0.0f;
    if (wave >= uint32_t(W::COMPUTE)) {
        // ---- a loader wave: the slots L, L + 2, ... ----
        const uint32_t L = wave - W::COMPUTE;
        auto dma = [&](uint32_t lds_addr, uint32_t voff, const void *src) {
            asm volatile("s_mov_b32 m0, %0\n"
                         "s_nop 0\n"
                         "global_load_lds_dwordx4 %1, %2\n"
                         :
                         : "s"(lds_addr), "v"(voff), "s"(src)
                         : "memory", "m0");
        };
        // instruction i brings the rows 2 i and 2 i + 1; rows past the share are the last one again (their scores are masked)
        const uint32_t last = limit - 1, half = lane >> 5, piece = lane & 31;
        auto request = [&](uint32_t u, bool values) {
            const uint32_t t0 = start_of(u), to = lds0 + (u % W::PLACES) * W::SLOT + (values ? W::PART : 0);
            const void *src = values ? a.vdata : a.kdata;
#pragma unroll
            for (int i = 0; i < W::LOADS; i++) {
                const uint32_t row = 2 * i + half, turn = row & 15;
                dma(to + i * 1024, (min(t0 + row, last) * kvh + kv) * W::ROW + ((piece ^ (values ? 2 * turn : turn)) << 4), src);
            }
        };
        uint32_t mine = 0;
        for (uint32_t u = L; u < slots; u += W::LOADERS, mine++) {
            const uint32_t at = u % W::PLACES, use = u / W::PLACES, before = (u - W::LOADERS) % W::PLACES;
            if (use) sync.await(W::C_KFREE + at, TILES * use);
            request(u, false);
            if (use == 0) request(u, true);
            if (mine) {
                if (use == 0) __builtin_amdgcn_s_waitcnt(vmcnt_only(3 * W::LOADS));
                else __builtin_amdgcn_s_waitcnt(vmcnt_only(2 * W::LOADS));
                sync.raise(W::C_KEYS + before);
            }
            if (use) {
                sync.await(W::C_VFREE + at, TILES * use);
                request(u, true);
            }
            if (mine) {
                __builtin_amdgcn_s_waitcnt(vmcnt_only(2 * W::LOADS));
                sync.raise(W::C_VALUES + before);
            }
        }
        if (mine) {
            const uint32_t at = (L + (mine - 1) * W::LOADERS) % W::PLACES;
            __builtin_amdgcn_s_waitcnt(vmcnt_only(W::LOADS));
            sync.raise(W::C_KEYS + at);
            __builtin_amdgcn_s_waitcnt(vmcnt_only(0));
            sync.raise(W::C_VALUES + at);
        }
    } else {
        // ---- the query operands: 16 * scale * log2(e) * q as f16 hi and lo parts ----
        if constexpr (PREP) {
            // (before anything waits for the query values) the tile's two rows' angles: an angle a lane; the pairs of dims (r, r + 32) are k-steps 0 and 1 of the same lane
            float2 *rope = reinterpret_cast<float2 *>(lds_raw + W::ROPE_OFF + wave * 512);
            {
                float s, c;
                rope_angle(position + 2 * tile + (lane >> 5), rope_frequency(lane & 31, 32, prep->p.log2_theta), s, c);
                rope[lane] = float2{s, c};
            }
            wave_sync();
            norm_query(q, *prep, [&](int s) { return 32 * s + 8 * j; });
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const float2 sc = rope[((pair >> 3) - 2 * tile) * 32 + 8 * j + e];
                const float first = q[0][e], second = q[1][e];
                q[0][e] = rope_first(first, second, sc.x, sc.y), q[1][e] = rope_second(first, second, sc.x, sc.y);
            }
        }
        half8 qhi[8], qlo[8];
        const float qmul = a.scale * 1.4426950408889634f * Q_UP;
#pragma unroll
        for (int s = 0; s < 8; s++) {
#pragma unroll
            for (int e = 0; e < 8; e++) {
                _Float16 h, lw;
                split_product(q[s][e], qmul, h, lw);
                qhi[s][e] = h, qlo[s][e] = lw;
            }
        }
#pragma unroll
        for (int T = 0; T < 16; T++) acc[T] = floatx4{0, 0, 0, 0};
        const uint32_t seen = PREP ? limit : min(position + (pair >> 3) + 1, limit);  // the pair's tokens end here
        const uint32_t seen_by_all = PREP ? limit : min(position + 1, limit);

        typedef __attribute__((address_space(3))) const half8 *LdsHalf8;
        typedef _Float16 half2 __attribute__((ext_vector_type(2)));
        typedef short short4 __attribute__((ext_vector_type(4)));
        typedef __attribute__((address_space(3))) short4 *LdsShort4;
        const uint32_t k_lane = lds0 + n * W::ROW + ((j ^ n) << 4);  // (16 n' + n: the same turn)
        const uint32_t v_row = 4 * j + (n >> 2), v_lane = lds0 + W::PART + v_row * W::ROW + (v_row << 5) + (n & 3) * 8;
        for (uint32_t u = 0; u < slots; u++) {
            const uint32_t at = u % W::PLACES, use = u / W::PLACES, t0 = start_of(u);
            // ---- S^T = K Q^T of the slot's two blocks, hi and lo parts side by side ----
            sync.await(W::C_KEYS + at, use + 1);
            floatx4 hi[4][2], lo[2];  // [64 dims][block]: two products to a sum of hi parts, as in attention_partial_body
#pragma unroll
            for (int b = 0; b < 2; b++) hi[0][b] = hi[1][b] = hi[2][b] = hi[3][b] = lo[b] = floatx4{0, 0, 0, 0};
            const uint32_t k_at = k_lane + at * W::SLOT;
            // (four operands a lot, the next lot asked for before this one's products)
            half8 kop[2][4];
            auto read_keys = [&](int lot) {
#pragma unroll
                for (int i = 0; i < 4; i++) kop[lot & 1][i] = *reinterpret_cast<LdsHalf8>((k_at ^ ((2 * lot + (i >> 1)) << 6)) + (i & 1) * BLOCK * W::ROW);
            };
            read_keys(0);
#pragma unroll
            for (int lot = 0; lot < 4; lot++) {
                if (lot < 3) read_keys(lot + 1);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const int s = 2 * lot + (i >> 1), b = i & 1;
                    hi[lot][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kop[lot & 1][i], qhi[s], hi[lot][b], 0, 0, 0);
                    lo[b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kop[lot & 1][i], qlo[s], lo[b], 0, 0, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            float x[8];  // tokens 4 j .. + 3 of block 0, then of block 1
#pragma unroll
            for (int e = 0; e < 8; e++) x[e] = ((hi[0][e >> 2][e & 3] + hi[1][e >> 2][e & 3]) + (hi[2][e >> 2][e & 3] + hi[3][e >> 2][e & 3])) + lo[e >> 2][e & 3];
            sync.raise(W::C_KFREE + at);
            if (t0 + W::SLOT_TOKENS > seen_by_all) {
#pragma unroll
                for (int e = 0; e < 8; e++) x[e] = t0 + 16 * (e >> 2) + 4 * j + (e & 3) < seen ? x[e] : NEVER;
            }
            // ---- online softmax of the lane's pair ----
            float top = fmaxf(fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3])), fmaxf(fmaxf(x[4], x[5]), fmaxf(x[6], x[7])));
            top = across_rows<16, 64>(top, MaxOp()) * (1.0f / Q_UP);
            const bool grown = top > m_run + MAX_SLACK;
            if (__ballot(grown)) {
                const float to = grown ? ceilf(top) : m_run, keep = __builtin_amdgcn_exp2f(m_run - to);
                m_run = to, l_run *= keep;
#pragma unroll
                for (int T = 0; T < 16; T++) acc[T] *= keep;
            }
            // (times P_UP afterwards and not in the exponent: the arguments of the tokens that count stay near 0, where they are
            // rounded least)
#pragma unroll
            for (int e = 0; e < 8; e++) x[e] = __builtin_amdgcn_exp2f(fmaf(x[e], 1.0f / Q_UP, -m_run)) * P_UP;
            l_run += ((x[0] + x[1]) + (x[2] + x[3])) + ((x[4] + x[5]) + (x[6] + x[7]));
            uint32_t ph[4], pl[4];
#pragma unroll
            for (int e = 0; e < 8; e += 2) {
                // toward zero: the hi part is x with the low mantissa bits cut off.  The lo part is what that leaves, to the
                // nearest: cut off as well, every probability would be short of what the sum has.
                ph[e / 2] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(x[e], x[e + 1]));
                const float r0 = x[e] - __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, x[e]) & 0xffffe000u);
                const float r1 = x[e + 1] - __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, x[e + 1]) & 0xffffe000u);
                pl[e / 2] = __builtin_bit_cast(uint32_t, half2{(_Float16)r0, (_Float16)r1});
            }
            const half8 phi = as_half8(ph[0], ph[1], ph[2], ph[3]), plo = as_half8(pl[0], pl[1], pl[2], pl[3]);
            // ---- O^T += V^T P^T ----
            sync.await(W::C_VALUES + at, use + 1);
            const uint32_t v_at = v_lane + at * W::SLOT;
            half8 vop[2][4];
            auto read_values = [&](int lot) {
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const uint32_t from = v_at ^ ((4 * lot + i) << 5);
                    const u32x2 w0 = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<LdsShort4>(from)));
                    const u32x2 w1 = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<LdsShort4>(from + BLOCK * W::ROW)));
                    vop[lot & 1][i] = as_half8(w0.x, w0.y, w1.x, w1.y);
                }
            };
            read_values(0);
#pragma unroll
            for (int lot = 0; lot < 4; lot++) {
                if (lot < 3) read_values(lot + 1);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int i = 0; i < 4; i++) acc[4 * lot + i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vop[lot & 1][i], phi, acc[4 * lot + i], 0, 0, 0);
#pragma unroll
                for (int i = 0; i < 4; i++) acc[4 * lot + i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vop[lot & 1][i], plo, acc[4 * lot + i], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
            sync.raise(W::C_VFREE + at);
        }
        l_run = across_rows<16, 64>(l_run, SumOp());
    }

    // ---- the partial of every pair ----
    if (wave < uint32_t(W::COMPUTE) && 16 * tile + n < real_rows) {
        const size_t slot = (size_t(pair >> 3) * a.nsplits + split) * a.heads + kv * 8 + (pair & 7);
        if (j == 0) *reinterpret_cast<floatx2 *>(a.part_ml + 2 * slot) = floatx2{m_run, sync.lost ? __builtin_nanf("") : l_run * (1.0f / P_UP)};
        float *dst = a.part_o + slot * DIM + 4 * j;
#pragma unroll
        for (int T = 0; T < 16; T++) {
            // (many rows' partials past the caches, see attention_partial_body)
            const floatx4 value = acc[T] * (1.0f / P_UP);
            if constexpr (TILES >= 3) __builtin_nontemporal_store(value, reinterpret_cast<floatx4 *>(dst + 16 * T));
            else *reinterpret_cast<floatx4 *>(dst + 16 * T) = value;
        }
    }
    if (__builtin_expect(sync.lost != 0, 0)) wait_gave_up(a.status, a.part_ml, sync.lost, a.rows, a.nsplits, split, a.heads, kv);
}

// (two waves per SIMD: with four waves in all the compiler would take more than 256 registers, half of them through copies)
template <int TILES>
__global__ __launch_bounds__((HalfRows<TILES>::THREADS_)) __attribute__((amdgpu_waves_per_eu(2))) void attention_partial_kernel_h(PartialArgs a) {
    attention_half_rows_body<TILES, false>(a, nullptr);
}
template <int TILES>
__global__ __launch_bounds__((HalfRows<TILES>::THREADS_)) __attribute__((amdgpu_waves_per_eu(2))) void attention_token_kernel_h(TokenArgs t) {
    attention_half_rows_body<TILES, true>(t.a, &t.prep);
}
