// Rows over codes (which: code_rows in decode.hip): computing waves that each have a tile of 16 (row, head) pairs and every
// STREAMS-th slot of 32 tokens, loader waves in front of them.  Included by decode.hip, inside its namespace, behind
// decode_half_rows.hpp, whose structure it has: transposed products, probabilities that stay in registers, counters in LDS, a
// ring of slots.
//
// What bounds it: vector instructions.  A tile's 32 tokens are some 350 of them over 8-bit codes (bytes widened by v_perm, a
// scale per group into the scores and into the probabilities, which are split into hi and lo parts once per group, the biases'
// sums) and 460 over 4-bit ones, beside 68 matrix instructions; with one computing wave on a SIMD these are issued 0.77 of the
// time (counters of 8 rows at 150000 tokens: vector 0.55, matrix 0.22 of the cycles), where the register kernels' phases wait
// for each other and the keys-first kernel's rounds end in a chain of their own.  So the probabilities' products with a scale
// and their lo parts are fused operations that take the f16 as it is (64 instructions fewer a slot), and what needs no second
// wave per SIMD gets none: four waves of two tiles (two streams) beat six or eight, three rows at 57123 tokens 27.6 us a
// layer against 30.2, because fewer places of the ring are held and fewer sums are joined.  Three tiles take two streams (6 rows
// at 150000 tokens 66 against 77 with one; at 4000, even).
// Tried: pairs of waves, one for the scores and one for the values, with the probabilities handed on through LDS (6 rows,
// 8-bit, at 150000 tokens 77 against 70 at that time; below 24k tokens ahead, 12000: 23.5 against 26.0); a group's products
// beside the next one's operands, and instructions dealt out in turn (even, and 16 to 48 bytes of spills a lane).
template <int BITS, int TILES>
struct CodeRows {
    static constexpr int STREAMS = TILES == 4 ? 1 : TILES == 1 ? 4 : 2;                   // computing waves of a tile
    static constexpr int COMPUTE = TILES * STREAMS, LOADERS = 2;                          // waves; 8 at most keep 256 registers each
    static constexpr int THREADS_ = (COMPUTE + LOADERS) * 64;
    static constexpr int ROW = BITS * 32;                                    // bytes of a (token, kv head) row of codes
    static constexpr int SLOT_TOKENS = 2 * BLOCK, PART = SLOT_TOKENS * ROW;  // keys or values of a slot
    static constexpr int SC_ARRAY = SLOT_TOKENS * 8;                         // scales or biases of keys or values: [token][group] f16
    static constexpr int V_OFF = PART, SC_OFF = 2 * PART;                    // of a slot: keys, values, [ks | kz | vs | vz]
    static constexpr int SLOT = SC_OFF + 4 * SC_ARRAY;
    static constexpr int PLACES = BITS == 8 ? 8 : 16;
    static constexpr int PART_LOADS = PART / 1024, LOADS = 2 * PART_LOADS + 4;  // load instructions of a slot
    static constexpr int DEPTH = 60 / LOADS;                                    // slots a loader has on their way at once
    static_assert(DEPTH * LOADS < 64, "vmcnt is 6 bits");
    static_assert(LOADERS * DEPTH < PLACES, "places for the slots at work");
    // LDS map, in bytes
    static constexpr int SYNC_OFF = PLACES * SLOT;               // counters, u32
    static constexpr int ROPE_OFF = SYNC_OFF + 64 * 4;           // [tile][row of the tile][32] sine, cosine
    static constexpr int XM_OFF = ROPE_OFF + TILES * 512;        // [computing wave][pair] maximum, sum
    static constexpr int LDS_BYTES = XM_OFF + COMPUTE * 128;
    static constexpr int X_OFF = 0;                              // the streams' merge, over the slots: [computing wave][16][lane] 16 bytes
    static_assert(COMPUTE * 16 * 1024 <= SYNC_OFF, "the merge fits over the slots");
    static constexpr int C_ROPE = 3 * PLACES;                    // [tile]: its angles are there
    static_assert(C_ROPE + TILES <= 64, "cleared by the first wave");
    static constexpr int C_KEYS = 0, C_VALUES = PLACES, C_FREE = 2 * PLACES;  // [place]: slots whose keys | values have landed; waves that are through
    static constexpr uint32_t SPIN_LIMIT = 1u << 20;
    static_assert(LDS_BYTES <= 160 * 1024, "LDS of a CU");
    static_assert(SAETTA_MAX_ROWS * 32 * 8 + SAETTA_MAX_ROWS * 10 * DIM * 4 <= LDS_BYTES, "the new rows' workgroup fits");
};

// As MAX_SLACK: the rescaling is 68 instructions.  A probability is up to 4 P_UP then, and times a scale of its token it has to
// fit a half: scales below LARGE_SCALE do (1024 * 63.97 = 65504).  Over a slot with a larger one the maximum is followed at
// once, so that scales fit up to 255, as in the other kernels.  A loader wave looks the slot's scales over and tells with the
// counter of its keys: a slack of 0 everywhere made 3 rows at 57123 tokens 27.3 -> 27.9 us a layer, 8 rows 45.3 -> 46.0 (4-bit).
constexpr float CODE_MAX_SLACK = 2.0f;
constexpr uint32_t LARGE_SCALE = 0x5400, LARGE_SLOT = 1u << 16;  // 64 as a half; what a counter is raised by

template <int BITS, int TILES, bool PREP>
__device__ __forceinline__ void attention_code_rows_body(const PartialArgs &a, const PrepArgs *prep) {
    using W = CodeRows<BITS, TILES>;
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds_raw[];
    const uint32_t lane = threadIdx.x & 63, n = lane & 15, j = lane >> 4;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t split = blockIdx.x, kv = blockIdx.y, kvh = a.kv_heads;
    uint32_t *sync_lds = reinterpret_cast<uint32_t *>(lds_raw + W::SYNC_OFF);
    const uint32_t lds0 = uint32_t(reinterpret_cast<uintptr_t>(lds_raw));
    const uint32_t context_splits = PREP ? a.nsplits - 1 : a.nsplits;
    if constexpr (PREP) {
        if (split >= context_splits) {
            new_rows<BITS, 2 * TILES>(a, *prep, lds_raw, W::COMPUTE + W::LOADERS, split - context_splits, 1, 0, SAETTA_GQA_GROUP);
            return;
        }
    }
    const uint32_t position = a.tp->position, kv_len = a.tp->kv_len;
    const uint32_t real_rows = a.rows * 8;
    const uint32_t tile = wave % TILES, stream = wave / TILES;
    // ---- a computing wave's query values: k-step 2 g + ab of lane (n, j) is dims 64 g + 16 j + 8 ab .. + 7 of pair 16 tile + n ----
    const uint32_t pair = min(16 * tile + n, real_rows - 1);
    float q[8][8];
    if (wave < uint32_t(W::COMPUTE)) {
        const size_t of_head = size_t(pair >> 3) * a.heads + kv * 8 + (pair & 7);
        const float *src = (PREP ? prep->q_and_gate + of_head * 2 * DIM : a.q + of_head * DIM) + 16 * j;
#pragma unroll
        for (int s = 0; s < 8; s++) {
            const float *at = src + 64 * (s >> 1) + 8 * (s & 1);
            const float4 f0 = *reinterpret_cast<const float4 *>(at), f1 = *reinterpret_cast<const float4 *>(at + 4);
            q[s][0] = f0.x, q[s][1] = f0.y, q[s][2] = f0.z, q[s][3] = f0.w, q[s][4] = f1.x, q[s][5] = f1.y, q[s][6] = f1.z, q[s][7] = f1.w;
        }
    }
    if (threadIdx.x < 64) sync_lds[threadIdx.x] = 0;
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
    LdsCounters<W::SPIN_LIMIT, 0x300u, LARGE_SLOT - 1> sync{sync_lds, lane};

    floatx4 acc[16];  // O^T of the codes: [4 g + e][i] is dim 64 g + 16 i + 4 j + e of the lane's pair
    float zsum[4] = {0.0f, 0.0f, 0.0f, 0.0f};
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
        auto dma4 = [&](uint32_t lds_addr, uint32_t voff, const void *src) {
            asm volatile("s_mov_b32 m0, %0\n"
                         "s_nop 0\n"
                         "global_load_lds_dword %1, %2\n"
                         :
                         : "s"(lds_addr), "v"(voff), "s"(src)
                         : "memory", "m0");
        };
        constexpr uint32_t UNITS = W::ROW / 16, ROWS_EACH = 64 / UNITS;  // 16-byte units of a row, rows a load brings
        const uint32_t last = limit - 1, sub_row = lane / UNITS, unit = lane % UNITS;
        auto request = [&](uint32_t u) {
            const uint32_t t0 = start_of(u), to = lds0 + (u % W::PLACES) * W::SLOT;
            const uint32_t sc = (min(t0 + (lane >> 1), last) * kvh + kv) * 8 + (lane & 1) * 4;
            dma4(to + W::SC_OFF, sc, a.kscales);
            dma4(to + W::SC_OFF + W::SC_ARRAY, sc, a.kbiases);
            dma4(to + W::SC_OFF + 2 * W::SC_ARRAY, sc, a.vscales);
            dma4(to + W::SC_OFF + 3 * W::SC_ARRAY, sc, a.vbiases);
#pragma unroll
            for (int i = 0; i < W::PART_LOADS; i++) {
                const uint32_t row = ROWS_EACH * i + sub_row, turn = BITS == 8 ? row & 15 : row >> 1 & 7;
                dma(to + i * 1024, (min(t0 + row, last) * kvh + kv) * W::ROW + ((unit ^ turn) << 4), a.kdata);
            }
#pragma unroll
            for (int i = 0; i < W::PART_LOADS; i++) {
                const uint32_t row = ROWS_EACH * i + sub_row, turn = (row >> 2 & 3) * (UNITS / 4);
                dma(to + W::V_OFF + i * 1024, (min(t0 + row, last) * kvh + kv) * W::ROW + ((unit ^ turn) << 4), a.vdata);
            }
        };
        uint32_t asked = 0, told = 0;  // of this loader's slots: requested, known to have landed
        auto place_of = [&](uint32_t mine) { return (L + mine * W::LOADERS) % W::PLACES; };
        auto tell_keys = [&]() {
            asm volatile("" ::: "memory");
            const uint32_t s = *reinterpret_cast<__attribute__((address_space(3))) const uint32_t *>(lds0 + place_of(told) * W::SLOT + W::SC_OFF + 2 * W::SC_ARRAY + 4 * lane);
            const bool large = max(s & 0x7fffu, s >> 16 & 0x7fffu) >= LARGE_SCALE;
            sync.raise(W::C_KEYS + place_of(told), __ballot(large) ? LARGE_SLOT + 1 : 1);
        };
        auto tell = [&]() {
            tell_keys(), sync.raise(W::C_VALUES + place_of(told));
            told++;
        };
        for (uint32_t u = L; u < slots; u += W::LOADERS) {
            const uint32_t at = u % W::PLACES, use = u / W::PLACES;
            if (use && sync.peek(W::C_FREE + at) < TILES * use) {
                // no place yet: what has been asked for is told of first, nobody else will
                __builtin_amdgcn_s_waitcnt(vmcnt_only(0));
                while (told < asked) tell();
                sync.await(W::C_FREE + at, TILES * use);
            }
            request(u), asked++;
            if (asked - told == uint32_t(W::DEPTH)) {
                __builtin_amdgcn_s_waitcnt(vmcnt_only((W::DEPTH - 1) * W::LOADS));
                tell();
            }
        }
        auto finish = [&](auto left_c) {
            constexpr int left = decltype(left_c)::value;  // slots behind this one
            if constexpr (left < W::DEPTH - 1) {
                if (asked - told == uint32_t(left) + 1) {
                    __builtin_amdgcn_s_waitcnt(vmcnt_only(left * W::LOADS + W::PART_LOADS));
                    tell_keys();
                    __builtin_amdgcn_s_waitcnt(vmcnt_only(left * W::LOADS));
                    sync.raise(W::C_VALUES + place_of(told));
                    told++;
                }
            }
        };
        static_assert(W::DEPTH <= 5, "all of them");
        finish(std::integral_constant<int, 3>()), finish(std::integral_constant<int, 2>()), finish(std::integral_constant<int, 1>()), finish(std::integral_constant<int, 0>());
    } else {
        // ---- the query operands ----
        if constexpr (PREP) {
            // (before anything waits for the query values) the tile's two rows' angles, an angle a lane; a pair's values are half a wavefront apart (k-steps 0 and 1)
            float2 *rope = reinterpret_cast<float2 *>(lds_raw + W::ROPE_OFF + tile * 512);
            if (stream == 0) {
                float s, c;
                rope_angle(position + 2 * tile + (lane >> 5), rope_frequency(lane & 31, 32, prep->p.log2_theta), s, c);
                rope[lane] = float2{s, c};
                wave_sync();
                if constexpr (W::STREAMS > 1) sync.raise(W::C_ROPE + tile);
            } else {
                sync.await(W::C_ROPE + tile, 1);
            }
            norm_query(q, *prep, [&](int s) { return 64 * (s >> 1) + 16 * j + 8 * (s & 1); });
#pragma unroll
            for (int s = 0; s < 2; s++) {
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    const float2 sc = rope[((pair >> 3) - 2 * tile) * 32 + 16 * (j & 1) + 8 * s + e];
                    const float x = q[s][e], other = half_swap(x, j < 2);
                    q[s][e] = j < 2 ? rope_first(x, other, sc.x, sc.y) : rope_second(other, x, sc.x, sc.y);
                }
            }
        }
        half8 qhi[8], qlo[8], qz[2];  // qz: per k-step the sum of the lane's 8 values, hi and lo (the key bias term)
        const float qmul = a.scale * 1.4426950408889634f * Q_UP;
#pragma unroll
        for (int s = 0; s < 8; s++) {
            float sum_hi = 0.0f, sum_lo = 0.0f;
#pragma unroll
            for (int e = 0; e < 8; e++) {
                _Float16 h, lw;
                split_product(q[s][key_slot_dim<BITS>(e)], qmul, h, lw);
                qhi[s][e] = h, qlo[s][e] = lw;
                sum_hi += (float)h, sum_lo += (float)lw;
            }
            _Float16 h, lw;
            split_hi_lo((sum_hi + sum_lo) * (1.0f / Q_UP), h, lw);
            qz[0][s] = h, qz[1][s] = lw;
        }
#pragma unroll
        for (int T = 0; T < 16; T++) acc[T] = floatx4{0, 0, 0, 0};
        const uint32_t seen = PREP ? limit : min(position + (pair >> 3) + 1, limit);  // the pair's tokens end here
        const uint32_t seen_by_all = PREP ? limit : min(position + 1, limit);

        typedef _Float16 half2 __attribute__((ext_vector_type(2)));
        typedef __attribute__((address_space(3))) const uint32_t *Lds1;
        typedef __attribute__((address_space(3))) const u32x2 *Lds2;
        typedef __attribute__((address_space(3))) const u32x4 *Lds4;
        // keys: piece 4 g + j of token n (16 bytes | 8 bytes)
        const uint32_t k_lane = BITS == 8 ? n * W::ROW + ((j ^ n) << 4) : n * W::ROW + ((j >> 1 ^ (n >> 1)) << 4) + (j & 1) * 8;
        // values: the dword of dims 4 pn .. + 3 (4-bit: of dims 8 (pn / 2) .. + 7) of a group, of tokens 4 j .. + 3
        const uint32_t pn = (n & 3) * 4 + (n >> 2);
        const uint32_t v_lane = W::V_OFF + 4 * j * W::ROW + j * (W::ROW / 4) + (BITS == 8 ? pn : pn >> 1) * 4;
        const uint32_t sc_lane = W::SC_OFF + 4 * j * 8;  // scales of tokens 4 j .. + 3: 32 bytes
        for (uint32_t u = stream; u < slots; u += W::STREAMS) {
            const uint32_t at = u % W::PLACES, use = u / W::PLACES, t0 = start_of(u), here = lds0 + at * W::SLOT;
            // ---- S^T = K Q^T of the slot's two blocks ----
            const float slack = sync.await(W::C_KEYS + at, use + 1) < LARGE_SLOT ? CODE_MAX_SLACK : 0.0f;
            KeyRegs<BITS> kreg[2][4];
#pragma unroll
            for (int b = 0; b < 2; b++) {
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    if constexpr (BITS == 8) {
                        const u32x4 v = *reinterpret_cast<Lds4>(here + (k_lane ^ (g << 6)) + b * BLOCK * W::ROW);
                        kreg[b][g].w[0] = v.x, kreg[b][g].w[1] = v.y, kreg[b][g].w[2] = v.z, kreg[b][g].w[3] = v.w;
                    } else {
                        const u32x2 v = *reinterpret_cast<Lds2>(here + (k_lane ^ (g << 5)) + b * BLOCK * W::ROW);
                        kreg[b][g].w[0] = v.x, kreg[b][g].w[1] = v.y;
                    }
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            float x[8];  // tokens 4 j .. + 3 of block 0, then of block 1
#pragma unroll
            for (int b = 0; b < 2; b++) {
                u32x4 ks[2];
                const u32x2 kz = *reinterpret_cast<Lds2>(here + W::SC_OFF + W::SC_ARRAY + (b * BLOCK + n) * 8);
#pragma unroll
                for (int i = 0; i < 2; i++) ks[i] = *reinterpret_cast<Lds4>(here + sc_lane + b * BLOCK * 8 + i * 16);
                // bias term: slot e of every lane group belongs to group e / 2 of token n
                const half8 zop = as_half8(perm(0, kz.x, 0x01000100u), perm(0, kz.x, 0x03020302u), perm(0, kz.y, 0x01000100u), perm(0, kz.y, 0x03020302u));
                floatx4 s = {0, 0, 0, 0}, r[4];
#pragma unroll
                for (int g = 0; g < 4; g++) r[g] = floatx4{0, 0, 0, 0};
                s = __builtin_amdgcn_mfma_f32_16x16x32_f16(zop, qz[0], s, 0, 0, 0);
#pragma unroll
                for (int ab = 0; ab < 2; ab++) {
                    half8 kop[4];
#pragma unroll
                    for (int g = 0; g < 4; g++) kop[g] = key_operand<BITS>(kreg[b][g], ab);
#pragma unroll
                    for (int g = 0; g < 4; g++) r[g] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kop[g], qhi[2 * g + ab], r[g], 0, 0, 0);
#pragma unroll
                    for (int g = 0; g < 4; g++) r[g] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kop[g], qlo[2 * g + ab], r[g], 0, 0, 0);
                }
                s = __builtin_amdgcn_mfma_f32_16x16x32_f16(zop, qz[1], s, 0, 0, 0);
                const uint32_t sw[8] = {ks[0].x, ks[0].y, ks[0].z, ks[0].w, ks[1].x, ks[1].y, ks[1].z, ks[1].w};
                constexpr float C1 = code_up<BITS>() / Q_UP;
#pragma unroll
                for (int tk = 0; tk < 4; tk++) {
                    float d = 0.0f;
#pragma unroll
                    for (int g = 0; g < 4; g++) d += half_bits_to_float(sw[2 * tk + (g >> 1)] >> (16 * (g & 1))) * r[g][tk];
                    x[4 * b + tk] = s[tk] + d * C1;
                }
            }
            if (t0 + W::SLOT_TOKENS > seen_by_all) {
#pragma unroll
                for (int e = 0; e < 8; e++) x[e] = t0 + 16 * (e >> 2) + 4 * j + (e & 3) < seen ? x[e] : NEVER;
            }
            // ---- online softmax of the lane's pair (see attention_half_rows_body) ----
            float top = fmaxf(fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3])), fmaxf(fmaxf(x[4], x[5]), fmaxf(x[6], x[7])));
            top = across_rows<16, 64>(top, MaxOp());
            const bool grown = top > m_run + slack;
            if (__ballot(grown)) {
                // (Up to four rows: the score itself, so that its token's probability is 1 and its products with the scales are
                // halves as they are. In whole numbers every product is split, and the lo parts are cut off: rel 3.84e-5 against
                // 64 bits instead of 3.50e-5 for 2 rows of 4-bit codes at 50000 tokens, 8.9e-5 instead of 8.4e-5 for 3 of 8 bits at
                // 57123, 30 times as much over equal keys. With lo parts to the nearest whole numbers are ahead, 4.74e-5
                // against 4.80e-5 for 6 rows of 8 bits there.)
                const float to = grown ? (TILES >= 3 ? ceilf(top) : top) : m_run, keep = __builtin_amdgcn_exp2f(m_run - to);
                m_run = to, l_run *= keep;
#pragma unroll
                for (int T = 0; T < 16; T++) acc[T] *= keep;
#pragma unroll
                for (int g = 0; g < 4; g++) zsum[g] *= keep;
            }
#pragma unroll
            for (int e = 0; e < 8; e++) x[e] = __builtin_amdgcn_exp2f(x[e] - m_run) * P_UP;
            l_run += ((x[0] + x[1]) + (x[2] + x[3])) + ((x[4] + x[5]) + (x[6] + x[7]));
            // (The lo parts of up to four rows are cut off like the hi parts, those of more rounded to the nearest, as in the kernels
            // that these rows took: the codes' sum and the biases' nearly cancel, so that the choice shows in the results. All to
            // the nearest, the errors against 64 bits at 32768 tokens of 8-bit codes are 3.9e-5 instead of 7e-5, and the results
            // 3e-5 away from what they were.)
            constexpr bool LO_NEAREST = TILES >= 3;
            // ---- O^T += V^T P^T, a group of dims at a time: its scale goes into the probabilities, its bias apart ----
            sync.await(W::C_VALUES + at, use + 1);
            ValRegs<BITS> vreg[2];
            u32x4 vs[2][2], vz[2][2];
#pragma unroll
            for (int b = 0; b < 2; b++) {
#pragma unroll
                for (int i = 0; i < 2; i++) {
                    vs[b][i] = *reinterpret_cast<Lds4>(here + sc_lane + 2 * W::SC_ARRAY + b * BLOCK * 8 + i * 16);
                    vz[b][i] = *reinterpret_cast<Lds4>(here + sc_lane + 3 * W::SC_ARRAY + b * BLOCK * 8 + i * 16);
                }
            }
            auto read_values = [&](int g) {
                const uint32_t from = here + (v_lane ^ (g * (W::ROW / 4)));
#pragma unroll
                for (int e = 0; e < 8; e++) vreg[g & 1].w[e] = *reinterpret_cast<Lds1>(from + ((e >> 2) * BLOCK + (e & 3)) * W::ROW);
            };
            read_values(0);
#pragma unroll
            for (int g = 0; g < 4; g++) {
                if (g < 3) read_values(g + 1);
                __builtin_amdgcn_sched_barrier(0);
                uint32_t ph[4], pl[4];
                float zs = 0.0f;
#pragma unroll
                for (int e = 0; e < 8; e += 2) {
                    const int word = 2 * (e & 3) + (g >> 1);  // of the block's 8: token e & 3, groups (0, 1) or (2, 3)
                    const uint32_t s0 = vs[e >> 2][word >> 2][word & 3] >> (16 * (g & 1)), s1 = vs[e >> 2][(word + 2) >> 2][(word + 2) & 3] >> (16 * (g & 1));
                    const uint32_t z0 = vz[e >> 2][word >> 2][word & 3] >> (16 * (g & 1)), z1 = vz[e >> 2][(word + 2) >> 2][(word + 2) & 3] >> (16 * (g & 1));
                    // (as fused operations, which take the f16 as it is)
                    const float x0 = fmaf(x[e], half_bits_to_float(s0), 0.0f), x1 = fmaf(x[e + 1], half_bits_to_float(s1), 0.0f);
                    const half2 hi = __builtin_bit_cast(half2, __builtin_amdgcn_cvt_pkrtz(x0, x1));
                    ph[e / 2] = __builtin_bit_cast(uint32_t, hi);
                    const float r0 = fmaf(x[e], half_bits_to_float(s0), -(float)hi[0]), r1 = fmaf(x[e + 1], half_bits_to_float(s1), -(float)hi[1]);
                    if constexpr (LO_NEAREST) pl[e / 2] = __builtin_bit_cast(uint32_t, half2{(_Float16)r0, (_Float16)r1});
                    else pl[e / 2] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(r0, r1));
                    zs = fmaf(x[e], half_bits_to_float(z0), zs), zs = fmaf(x[e + 1], half_bits_to_float(z1), zs);
                }
                zsum[g] += zs;
                const half8 phi = as_half8(ph[0], ph[1], ph[2], ph[3]), plo = as_half8(pl[0], pl[1], pl[2], pl[3]);
                half8 vop[4];
#pragma unroll
                for (int e = 0; e < 4; e++) vop[e] = val_operand<BITS>(vreg[g & 1], e, pn);
#pragma unroll
                for (int e = 0; e < 4; e++) acc[4 * g + e] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vop[e], phi, acc[4 * g + e], 0, 0, 0);
#pragma unroll
                for (int e = 0; e < 4; e++) acc[4 * g + e] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vop[e], plo, acc[4 * g + e], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
            sync.raise(W::C_FREE + at);
        }
        l_run = across_rows<16, 64>(l_run, SumOp());
#pragma unroll
        for (int g = 0; g < 4; g++) zsum[g] = across_rows<16, 64>(zsum[g], SumOp());
    }

    // ---- the streams of a tile joined, and the partial of every pair ----
    constexpr float UNSCALE = code_up<BITS>() / P_UP;
    auto piece = [&](int i) {  // dims 16 i + 4 j .. + 3
        const int g = i >> 2, c = i & 3;
        floatx4 o = {acc[4 * g][c], acc[4 * g + 1][c], acc[4 * g + 2][c], acc[4 * g + 3][c]};
        return o * UNSCALE + zsum[g] * (1.0f / P_UP);
    };
    const bool real = wave < uint32_t(W::COMPUTE) && 16 * tile + n < real_rows;
    const size_t slot = (size_t(pair >> 3) * a.nsplits + split) * a.heads + kv * 8 + (pair & 7);
    float *dst = a.part_o + slot * DIM + 4 * j;
    auto put = [&](int i, floatx4 value) {
        // (many rows' partials past the caches, see attention_partial_body)
        if constexpr (TILES >= 3) __builtin_nontemporal_store(value, reinterpret_cast<floatx4 *>(dst + 16 * i));
        else *reinterpret_cast<floatx4 *>(dst + 16 * i) = value;
    };
    const uint32_t streams = min(slots, uint32_t(W::STREAMS));  // that had a slot
    if (W::STREAMS == 1 || streams == 1) {
        if (wave < uint32_t(W::COMPUTE) && stream == 0) {
            if (real && j == 0) *reinterpret_cast<floatx2 *>(a.part_ml + 2 * slot) = floatx2{m_run, sync.lost ? __builtin_nanf("") : l_run * (1.0f / P_UP)};
#pragma unroll
            for (int i = 0; i < 16; i++) {
                if (real) put(i, piece(i));
            }
        }
    } else {
        floatx4 *xo = reinterpret_cast<floatx4 *>(lds_raw + W::X_OFF);
        floatx2 *xm = reinterpret_cast<floatx2 *>(lds_raw + W::XM_OFF);
        __syncthreads();  // nobody reads a slot any more
        if (wave < uint32_t(W::COMPUTE) && stream < streams) {
            if (j == 0) xm[wave * 16 + n] = floatx2{m_run, sync.lost ? __builtin_nanf("") : l_run * (1.0f / P_UP)};
#pragma unroll
            for (int i = 0; i < 16; i++) xo[(wave * 16 + i) * 64 + lane] = piece(i);
        }
        __syncthreads();
        if (wave < uint32_t(W::COMPUTE)) {
            float m = NO_SCORE, l = 0.0f, f[W::STREAMS];
            floatx2 ml[W::STREAMS];
#pragma unroll
            for (int s = 0; s < W::STREAMS; s++) {
                ml[s] = uint32_t(s) < streams ? xm[(s * TILES + tile) * 16 + n] : floatx2{NO_SCORE, 0.0f};
                m = fmaxf(m, ml[s][0]);
            }
#pragma unroll
            for (int s = 0; s < W::STREAMS; s++) {
                f[s] = __builtin_amdgcn_exp2f(ml[s][0] - m);
                l += f[s] * ml[s][1];
            }
            if (real && j == 0 && stream == 0) *reinterpret_cast<floatx2 *>(a.part_ml + 2 * slot) = floatx2{m, l};
            for (uint32_t i = stream; i < 16; i += W::STREAMS) {
                floatx4 o = {0, 0, 0, 0};
#pragma unroll
                for (int s = 0; s < W::STREAMS; s++) {
                    if (uint32_t(s) < streams) o += xo[((s * TILES + tile) * 16 + i) * 64 + lane] * f[s];
                }
                if (real) put(int(i), o);
            }
        }
    }
    if (__builtin_expect(sync.lost != 0, 0)) wait_gave_up(a.status, a.part_ml, sync.lost, a.rows, a.nsplits, split, a.heads, kv);
}

template <int BITS, int TILES>
__global__ __launch_bounds__((CodeRows<BITS, TILES>::THREADS_)) __attribute__((amdgpu_waves_per_eu(2))) void attention_partial_kernel_c(PartialArgs a) {
    attention_code_rows_body<BITS, TILES, false>(a, nullptr);
}
template <int BITS, int TILES>
__global__ __launch_bounds__((CodeRows<BITS, TILES>::THREADS_)) __attribute__((amdgpu_waves_per_eu(2))) void attention_token_kernel_c(TokenArgs t) {
    attention_code_rows_body<BITS, TILES, true>(t.a, &t.prep);
}
