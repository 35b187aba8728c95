// Fused template attention over one position's T tokens (64 squares, then T - 64 metadata tokens).
// Computes what model/fused_blocks.py:35-97 (template_bias_kernel + template_attention_kernel) and
// model/attention_cuda.py:97-304 compute, for any head counts and widths, with the reference's fp16 rounding points:
//   q' = f16((q * (1 / sqrt(mean(q^2) + eps))) * q_gain),  k' = f16((k * (1 / sqrt(mean(k^2) + eps))) * k_gain)
//   s[i, j] = (q'_i . k'_j) * scale + [i, j < 64] f16(sum_t c[b, i, h, t] templates[t, i, j])
//   out_i = sum_j f16(exp(s_ij - max_i)) v_j / sum_j exp(s_ij - max_i)
// in f32 (MFMA products of the fp16 operands are exact; sums are f32).
// projected[B, T, H*dq | KV*dq | KV*dv | H*tc] in, out[B, T, H*dv] (fp16). The templates come key-major,
// keyed[i][j][t] (8 templates a key, zero past templates_count), so that a lane reads its query's
// templates for 4 keys as 4 16-byte loads (the reference pairs its templates likewise,
// model/attention_cuda.py:410-440).
//
// Two kernels: attention_wave.h's, for query and value widths up to 64 and up to 80 tokens (every network's), and this file's,
// for wider heads and more tokens. Here a workgroup takes a run of groups_per_block (position, key/value group) pairs, in
// order, which may run on from one position into the next; it has one wavefront per slab of 16 queries. A group's raw key,
// value and query rows arrive by DMA into LDS, double-buffered: the next group's rows load while this group's heads run. The
// keys are normalised in place in LDS (four threads a key), the queries in registers; a wavefront then runs each head of
// the group on v_mfma_f32_16x16x32_f16: the scores come out transposed, S^T = K' Q'^T, so a lane holds one query's scores for
// 4 keys of each 16-key tile -- exactly the fragment O^T = V^T P^T needs as its B operand, so the probabilities never leave
// registers. V^T's fragments are read from the raw value rows by transposing LDS reads (ds_read_b64_tr_b16: in each 16
// lanes, lane j receives element j % 4 of the 8 bytes lanes j / 4 + 4 r address, r = 0..3), so the values are never
// transposed in LDS. The template bias is an MFMA too, from the templates held in registers.
// Attention is held to a tolerance, not to bits: its f32 sums run in the MFMA's and the lanes' order (sums of
// squares are v_dot2_f32_f16 of the fp16 pairs), the norms take IEEE divides and square roots, and the softmax's
// exponent is one fma into the hardware exp2.
#include "attention_wave.h"

namespace {

// TILES: key tiles of 16 the instantiation holds (T <= 16 TILES)
template <int DQP, int DV, int TILES>
struct Layout {
    static constexpr int STEPS = (TILES + 1) / 2;     // 32-key steps of P V
    static constexpr int KEYS = TILES * 16;           // keys (and queries) staged
    static constexpr int KC = DQP / 8, VC = DV / 8;   // 16-byte chunks a raw key (query) row, a raw value row
    // value keys staged, whole DMA instructions of them (64 chunks): a half step of P V past them reads zeros
    static constexpr int VKEYS = (KEYS * VC + 63) / 64 * 64 / VC;
    static constexpr int WAVES = TILES;               // one a slab of 16 queries
    // LDS in bytes: two buffers of keys (raw as they land, normalised in place), two of raw values, then
    // two of raw queries and template coefficients
    static constexpr int RAW_K_BYTES = KEYS * DQP * 2;   // a buffer's
    static constexpr int RAW_V_BYTES = VKEYS * DV * 2;   // a buffer's
    static constexpr int RAW_Q_BYTES = KEYS * DQP * 2;   // a head's
    static constexpr int COEF_BYTES = 64 * MAX_TEMPLATES * 2;   // a head's template coefficients, a square query a row
    static constexpr int FIXED_BYTES = 2 * RAW_K_BYTES + 2 * RAW_V_BYTES;
    static int bytes(int per_kv) { return FIXED_BYTES + 2 * per_kv * (RAW_Q_BYTES + COEF_BYTES); }
};

// Every wavefront's LDS writes are done and visible; unlike __syncthreads, the DMA loads in flight go on.
DEVICE void lds_barrier() {
    __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0), vmcnt and expcnt left alone
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// A wavefront's share of the DMA of a raw block of ROWS rows x CH 16-byte chunks, 64 chunks an instruction:
// instruction i = wave + j WAVES writes slots i * 64 + lane, slot s holding chunk (s % CH) ^ swizzle(row) of row
// s / CH. The lane's source offsets (halves from the block's first column) are planned once: rows past last read
// row last again (their values are masked or multiplied by zero later), so every address is inside the rows. The
// offsets are in bytes, so that a load's address is the block's (uniform) start plus the lane's 32-bit offset: the
// scalar-base form of the DMA, with no 64-bit address arithmetic in the lanes.
template <int ROWS, int CH, int WAVES>
struct DmaPlan {
    static constexpr int INSTRUCTIONS = ROWS * CH / 64;
    static constexpr int PER_WAVE = (INSTRUCTIONS + WAVES - 1) / WAVES;
    static_assert(ROWS * CH % 64 == 0, "whole DMA instructions");
    uint32_t offset[PER_WAVE];
    DEVICE void plan(int last, int stride, int wave, int lane) {
#pragma unroll
        for (int j = 0; j < PER_WAVE; j++) {
            const int slot = (wave + j * WAVES) * 64 + lane, row = min(slot / CH, ROWS - 1), chunk = (slot % CH) ^ swizzle<CH>(row);
            offset[j] = (uint32_t)(min(row, last) * stride + chunk * 8) * 2u;
        }
    }
    DEVICE void issue(LDS_SPACE int8_t* raw, const half_t* source, int wave) const {
        const int8_t* bytes = reinterpret_cast<const int8_t*>(source);
#pragma unroll
        for (int j = 0; j < PER_WAVE; j++) {
            const int i = wave + j * WAVES;
            // non-temporal (cache policy 2): the projection's rows are read once, and streaming them past the caches
            // leaves the output rows cached for the combine GEMM (a forward 17.33-17.36 against 17.48-17.49 ms at batch
            // 1024, alternated on one MI355X)
            if (INSTRUCTIONS % WAVES == 0 || i < INSTRUCTIONS)
                __builtin_amdgcn_global_load_lds((const void*)(bytes + offset[j]), (LDS_SPACE void*)(raw + i * 1024), 16, 0, 2);
        }
    }
};

// TILES = ceil(T / 16) exactly: the launch picks the instantiation, so every count below is fixed at compile time.
// Registers are held to two wavefronts a SIMD, within which the query and value widths up to 64 need no scratch (a
// scratch reload would wait for the DMA in flight too); query widths of 128, and value widths of 128 past 96 tokens,
// spill some. (Fewer registers for more workgroups a CU cost more instructions than they gain: the kernel is bound by its
// VALU work.)
template <int DQP, int DV, int TILES, bool BF16>
__global__ __launch_bounds__(64 * TILES) __attribute__((amdgpu_waves_per_eu(2))) void template_attention_kernel(
    const half_t* __restrict__ projected, const half_t* __restrict__ keyed, const half_t* __restrict__ q_gain,
    const half_t* __restrict__ k_gain, half_t* __restrict__ out, int T, int heads, int kv_heads, int dq, int templates_count,
    int groups_per_block, float eps, float scale)
{
    typedef Layout<DQP, DV, TILES> L;
    constexpr bool BY_STEP = TILES == 5;   // with five tiles the softmax sum and P V outputs are added by 32-key step, in step order
    constexpr int KC = L::KC, VC = L::VC, WAVES = L::WAVES, THREADS = 64 * WAVES, STEPS = L::STEPS, KEYS = L::KEYS;
    extern __shared__ __align__(16) int8_t lds[];
    LDS_SPACE int8_t* raw_k = (LDS_SPACE int8_t*)lds;                        // [2][KEYS * DQP halves]
    LDS_SPACE int8_t* raw_v = raw_k + 2 * L::RAW_K_BYTES;                    // [2][VKEYS * DV halves]
    LDS_SPACE int8_t* raw_q = raw_v + 2 * L::RAW_V_BYTES;    // [2][per_kv][KEYS * DQP halves]
    LDS_SPACE int8_t* raw_c = raw_q + 2 * (heads / kv_heads) * L::RAW_Q_BYTES;   // [2][per_kv][64][8 halves]

    const int tid = threadIdx.x, lane = tid & 63, slab = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int width = heads * dq + kv_heads * dq + kv_heads * DV + heads * templates_count;
    const int k_offset = heads * dq, v_offset = k_offset + kv_heads * dq, c_offset = v_offset + kv_heads * DV;
    const int per_kv = heads / kv_heads;
    // pair p of the launch is key/value group p % kv_heads of position p / kv_heads
    auto board_of = [&](int pair) { return projected + (size_t)(pair / kv_heads) * T * width; };
    const int first_pair = blockIdx.x * groups_per_block;
    const int head_bytes = L::RAW_Q_BYTES;

    const int col = lane & 15, quad = lane >> 4;
    const int query = slab * 16 + col;
    const bool query_ok = query < T;
    const bool square_query = query < 64;

    // the DMA plans: keys and queries share one (same rows, same chunks), values have their own
    DmaPlan<KEYS, KC, WAVES> key_plan;
    DmaPlan<L::VKEYS, VC, WAVES> value_plan;
    key_plan.plan(T - 1, width, slab, lane);
    value_plan.plan(T - 1, width, slab, lane);
    const uint32_t coefficient_row = (uint32_t)(lane * width + c_offset) * 2u;   // a square query's row (bytes), for the coefficients' DMA

    // a pair's keys and values (kv), its queries and coefficients (q), into a buffer
    auto dma_group = [&](int pair, int buffer, bool kv, bool q) {
        const half_t* board = board_of(pair);
        const int group = pair % kv_heads;
        if (kv) {
            value_plan.issue(raw_v + buffer * L::RAW_V_BYTES, board + v_offset + group * DV, slab);
            key_plan.issue(raw_k + buffer * L::RAW_K_BYTES, board + k_offset + group * dq, slab);
        }
        if (q) {
            for (int hi = 0; hi < per_kv; hi++)
                key_plan.issue(raw_q + (buffer * per_kv + hi) * head_bytes, board + (group * per_kv + hi) * dq, slab);
            if (templates_count == MAX_TEMPLATES) {
                for (int hi = slab; hi < per_kv; hi += WAVES)
                    __builtin_amdgcn_global_load_lds((const void*)(reinterpret_cast<const int8_t*>(board + (group * per_kv + hi) * MAX_TEMPLATES) + coefficient_row),
                                                     (LDS_SPACE void*)(raw_c + (buffer * per_kv + hi) * L::COEF_BYTES), 16, 0, 2);
            }
        }
    };
    dma_group(first_pair, 0, true, true);

    // The template bias of a 16-key tile is an MFMA too: bias^T[k][q] = sum over (q', t) of templates[t][q'][k] *
    // [q' == q] c[q][t], an inner dimension of the wavefront's 16 queries x 8 templates, 32 a step. In step j the A
    // operand lane (key 16 kt + lane % 16, quad) holds keyed[q' = 16 slab + 4 j + quad][key][0..7] -- its query's 8
    // templates for the key -- and the B operand lane (query col, quad) holds c[col][0..7] when 4 j + quad == col,
    // else zeros. The A operands stay in registers for every group (zero for the queries past the squares; loaded
    // from clamped places, then zeroed, so that the loads issue together).
    uint4 templates[4][4];
#pragma unroll
    for (int kt = 0; kt < 4; kt++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int template_query = slab * 16 + 4 * j + quad;
            templates[kt][j] = *reinterpret_cast<const uint4*>(keyed + ((size_t)min(template_query, 63) * 64 + kt * 16 + (lane & 15)) * MAX_TEMPLATES);
            if (template_query >= 64) templates[kt][j] = uint4{0, 0, 0, 0};
        }

    // The query gains of this lane's query columns (zero past dq), and the key gains of this thread's key columns: the keys
    // are normalised in LDS by four adjacent threads a key, KC / 4 chunks each.
    float gains[DQP / 32][8];
#pragma unroll
    for (int ks = 0; ks < DQP / 32; ks++)
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const int d = ks * 32 + quad * 8 + e;
            gains[ks][e] = d < dq ? (float)q_gain[min(d, dq - 1)] : 0.0f;
        }
    constexpr int PART_CHUNKS = KC / 4;
    constexpr int KEY_PASSES = (KEYS * 4 + THREADS - 1) / THREADS;   // the keys normalised THREADS / 4 at a time
    static_assert(KC % 4 == 0, "four threads a key");
    const int first_chunk = (tid % 4) * PART_CHUNKS;
    float key_gains[PART_CHUNKS][8];
#pragma unroll
    for (int c = 0; c < PART_CHUNKS; c++)
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const int d = (first_chunk + c) * 8 + e;
            key_gains[c][e] = d < dq ? (float)k_gain[min(d, dq - 1)] : 0.0f;
        }
    // the staged outputs this thread writes out: row item / VC, chunk item % VC of each head
    constexpr int O_TOTAL = KEYS * VC, O_ITEMS = (O_TOTAL + THREADS - 1) / THREADS;
    const float columns = (float)dq;
    // 1 / sqrt(mean of squares + eps): the mean is the product by the exact reciprocal when dq is a power of two, the
    // same bits as the quotient without an IEEE divide
    const bool power_of_two = (dq & (dq - 1)) == 0;
    const float reciprocal_columns = 1.0f / columns;
    auto inverse_norm = [&](float squares) {
        const float mean = power_of_two ? squares * reciprocal_columns : squares / columns;
        return 1.0f / __builtin_sqrtf(mean + eps);
    };

    // A key normalised in place: k' = f16((k * (1 / sqrt(mean of squares + eps))) * k_gain) over the key's dq columns, the
    // four threads of a key adding their partial sums as (a + b) + (c + d). Past dq a raw key chunk holds another head's
    // columns: zeroed, as a zero query column would not cancel an infinite one.
    auto normalise_key = [&](LDS_SPACE int8_t* keys, int scale_key) {
        uint4 raw[PART_CHUNKS];
        float squares = 0.0f;
#pragma unroll
        for (int c = 0; c < PART_CHUNKS; c++) {
            raw[c] = lds_chunk(keys + raw_slot<KC>(scale_key, first_chunk + c) * 16);
            if ((first_chunk + c) * 8 >= dq) raw[c] = uint4{0, 0, 0, 0};
            squares = squares8<BF16>(raw[c], squares);
        }
        squares += lane_xor1(squares);
        squares += lane_xor2(squares);
        const float inverse = inverse_norm(squares);
#pragma unroll
        for (int c = 0; c < PART_CHUNKS; c++) {
            v8h normed;
            float wide[8];
            widen8<BF16>(raw[c], wide);
#pragma unroll
            for (int e = 0; e < 8; e++) normed[e] = (half_t)((wide[e] * inverse) * key_gains[c][e]);
            *reinterpret_cast<LDS_SPACE v8h*>(keys + raw_slot<KC>(scale_key, first_chunk + c) * 16) = normed;
        }
    };

    // The templates and gains have landed before the loop (with the first group's rows): counting loads across the
    // loop's iterations, the compiler would otherwise wait for every load in flight -- the next group's rows too --
    // at each use of them in the loop.
    __builtin_amdgcn_s_waitcnt(0);

    // A group's outputs are staged in its query buffer, each wavefront writing its own query rows of each head over
    // the queries it has read (the value width is at most the query width), and written out during the next group, once
    // its keys are normalised -- 16 bytes a lane along the rows, where the wait at the start of the group after finds them
    // long done.
    // Stored straight from the MFMA layout, 8 bytes a lane scattered over 16 rows, they would be waited for at once.
    constexpr bool STAGED = DV <= DQP;
    auto write_out = [&](int pair, int buffer) {
        for (int hi = 0; hi < per_kv; hi++) {
            const LDS_SPACE int8_t* staged = raw_q + (buffer * per_kv + hi) * head_bytes;
            half_t* to = out + (size_t)(pair / kv_heads) * T * (heads * DV) + (pair % kv_heads * per_kv + hi) * DV;
            // plain LDS reads, the compiler waiting for them: no DMA is in flight here (the next group's goes out after the
            // barrier that follows)
#pragma unroll
            for (int k = 0; k < O_ITEMS; k++) {
                const int item = tid + k * THREADS, q = item / VC, c = item % VC;
                if ((O_TOTAL % THREADS == 0 || item < O_TOTAL) && q < T)
                    *reinterpret_cast<uint4*>(to + (size_t)q * (heads * DV) + c * 8) = lds_chunk(staged + raw_slot<KC>(q, c) * 16);
            }
        }
    };

    for (int gi = 0; gi < groups_per_block; gi++) {
        const int pair = first_pair + gi, group = pair % kv_heads;
        const size_t b = pair / kv_heads;
        const half_t* board = board_of(pair);
        const int buffer = gi & 1;
        // this group's raw rows have landed (this wavefront's DMA), and every wavefront is past the previous group
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();

        LDS_SPACE int8_t* group_keys = raw_k + buffer * L::RAW_K_BYTES;
#pragma unroll
        for (int pass = 0; pass < KEY_PASSES; pass++) {
            const int scale_key = pass * (THREADS / 4) + tid / 4;
            if (KEYS * 4 % THREADS != 0 && scale_key >= KEYS) break;
            normalise_key(group_keys, scale_key);
        }
        // The previous group's outputs leave its query buffer once the keys are normalised; after the barrier every
        // wavefront has read its share, and the next group's keys, values and queries load into the other buffers. (Issued
        // at the group's start instead, the DMA and the stores cost 2 and 2 us more at batch 1024: they then ran beside the
        // key normalisation's LDS traffic and its reads.)
        if (STAGED && gi > 0) write_out(pair - 1, buffer ^ 1);
        lds_barrier();   // the normalised keys are in place, and every wavefront's outputs are read
        if (gi + 1 < groups_per_block) dma_group(pair + 1, buffer ^ 1, true, true);

        for (int hi = 0; hi < per_kv; hi++) {
            const int head = group * per_kv + hi;
            // this query's template coefficients for the head, as f16 pairs (zero past templates_count, and for the
            // queries that are not squares, whose bias is then zero)
            uint4 coefficients;
            {
                const half_t* from = board + (size_t)min(query, 63) * width + c_offset + head * templates_count;
                if (templates_count == MAX_TEMPLATES) {
                    coefficients = lds_read16_settled(raw_c + (buffer * per_kv + hi) * L::COEF_BYTES + min(query, 63) * 16);
                } else {
                    uint16_t c[MAX_TEMPLATES];
#pragma unroll
                    for (int t = 0; t < MAX_TEMPLATES; t++) {
                        const uint16_t value = __builtin_bit_cast(uint16_t, from[min(t, max(templates_count - 1, 0))]);
                        c[t] = t < templates_count ? value : (uint16_t)0;
                    }
                    coefficients = uint4{c[0] | ((uint32_t)c[1] << 16), c[2] | ((uint32_t)c[3] << 16), c[4] | ((uint32_t)c[5] << 16),
                                         c[6] | ((uint32_t)c[7] << 16)};
                }
                if constexpr (BF16) coefficients = bf16_to_f16x8(coefficients);
                if (!square_query) coefficients = uint4{0, 0, 0, 0};
            }
            // the query row's fragment of B: lane holds dq columns ks * 32 + 8 quad .. + 8
            const LDS_SPACE int8_t* queries = raw_q + (buffer * per_kv + hi) * head_bytes;
            const LDS_SPACE int8_t* keys = raw_k + buffer * L::RAW_K_BYTES;
            uint4 qv[DQP / 32];
            float squares = 0.0f;
#pragma unroll
            for (int ks = 0; ks < DQP / 32; ks++) {
                const int c = ks * 4 + quad;
                qv[ks] = lds_chunk(queries + raw_slot<KC>(query, c) * 16);
                if (c * 8 >= dq) qv[ks] = uint4{0, 0, 0, 0};
                squares = squares8<BF16>(qv[ks], squares);
            }
            squares = sum_across_rows(squares);
            const float q_inverse = inverse_norm(squares);
            v8h qf[DQP / 32];
#pragma unroll
            for (int ks = 0; ks < DQP / 32; ks++) {
                float wide[8];
                widen8<BF16>(qv[ks], wide);
#pragma unroll
                for (int e = 0; e < 8; e++) qf[ks][e] = (half_t)((wide[e] * q_inverse) * gains[ks][e]);
            }

            // the bias MFMAs' B operands: this query's coefficients in the one step j with 4 j + quad == col
            v8h mix[4];
#pragma unroll
            for (int j = 0; j < 4; j++)
                mix[j] = __builtin_bit_cast(v8h, 4 * j + quad == col ? coefficients : uint4{0, 0, 0, 0});

            // S^T tiles: lane holds s[query][16 kt + 4 quad + r]; square keys take the template bias (zero for the
            // queries past the squares), keys past T are masked
            float s[2 * STEPS][4];
            float top = -__builtin_inff();
#pragma unroll
            for (int kt = 0; kt < 2 * STEPS; kt++) {
                if (kt >= TILES) {
#pragma unroll
                    for (int r = 0; r < 4; r++) s[kt][r] = -__builtin_inff();
                    continue;
                }
                // one tile's keys at a time: loads hoisted over the tiles would hold all their registers at once
                __builtin_amdgcn_sched_barrier(0);
                v4f acc = v4f{0, 0, 0, 0};
#pragma unroll
                for (int ks = 0; ks < DQP / 32; ks++) {
                    const v8h kf = *reinterpret_cast<const LDS_SPACE v8h*>(keys + raw_slot<KC>(kt * 16 + col, ks * 4 + quad) * 16);
                    acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf, qf[ks], acc, 0, 0, 0);
                }
                v4f bias = v4f{0, 0, 0, 0};
                if (kt < 4) {
#pragma unroll
                    for (int j = 0; j < 4; j++)
                        bias = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, templates[kt][j]), mix[j], bias, 0, 0, 0);
                }
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    float value = acc[r] * scale;
                    if (kt < 4) {
                        value += (float)(half_t)bias[r];
                    } else if (kt * 16 + quad * 4 + r >= T) {
                        value = -__builtin_inff();
                    }
                    s[kt][r] = value;
                    top = fmaxf(top, value);
                }
            }
            top = max_across_rows(top);
            float total = 0.0f;
            const float offset = -top * LOG2E;
            if constexpr (BY_STEP) {
                // each 32-key step's sum across the wavefront, then the steps' sums in order
#pragma unroll
                for (int st = 0; st < STEPS; st++) {
                    float step_total = 0.0f;
#pragma unroll
                    for (int kt = 2 * st; kt < 2 * st + 2; kt++)
#pragma unroll
                        for (int r = 0; r < 4; r++) {
                            const float p = kt < TILES ? __builtin_amdgcn_exp2f(__builtin_fmaf(s[kt][r], LOG2E, offset)) : 0.0f;
                            s[kt][r] = p;
                            step_total += p;
                        }
                    step_total = sum_across_rows(step_total);
                    total = st == 0 ? step_total : total + step_total;
                }
            } else {
#pragma unroll
                for (int kt = 0; kt < 2 * STEPS; kt++)
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const float p = kt < TILES ? __builtin_amdgcn_exp2f(__builtin_fmaf(s[kt][r], LOG2E, offset)) : 0.0f;
                        s[kt][r] = p;
                        total += p;
                    }
                total = sum_across_rows(total);
            }
            const float inverse_total = __builtin_amdgcn_rcpf(total);

            // O^T = V^T P^T over 32-key steps: position e of both operands is key 32 st + 16 (e / 4) + 4 quad + e % 4.
            // V^T's half h (positions 4 h ..) of lane (col, quad) is V[32 st + 16 h + 4 quad + r][16 dt + col], r = 0..3:
            // a transposing read in which lane 4 r' + g of the 16 addresses the 4 values of key 32 st + 16 h + 4 quad + r',
            // columns 16 dt + 4 g .. + 3 (half g % 2 of chunk 2 dt + g / 2).
            // the swizzle of a row repeats every 16 rows, so the rows 16 h + 32 st on are the lane's first at a fixed offset
            const LDS_SPACE int8_t* values = raw_v + buffer * L::RAW_V_BYTES;
            const int value_row = 4 * quad + col / 4, value_group = col % 4;
            const LDS_SPACE int8_t* value_base[DV / 16];
            uint32_t value_words[DV / 16];   // the same LDS addresses, as the asm reads take them
#pragma unroll
            for (int dt = 0; dt < DV / 16; dt++) {
                value_base[dt] = values + raw_slot<VC>(value_row, 2 * dt + value_group / 2) * 16 + (value_group % 2) * 8;
                value_words[dt] = (uint32_t)(uintptr_t)value_base[dt];
            }
            v4f o[DV / 16];
#pragma unroll
            for (int dt = 0; dt < DV / 16; dt++) o[dt] = v4f{0, 0, 0, 0};
            each_step<0, STEPS>([&](auto st_index) {
                constexpr int st = decltype(st_index)::value, ROW_BYTES = VC * 16;
                __builtin_amdgcn_sched_barrier(0);
                uint32_t pw[4];
#pragma unroll
                for (int r = 0; r < 2; r++) {
                    pw[r] = narrow16x2<BF16>(s[2 * st][2 * r], s[2 * st][2 * r + 1]);
                    pw[2 + r] = narrow16x2<BF16>(s[2 * st + 1][2 * r], s[2 * st + 1][2 * r + 1]);
                }
                const uint4 pf = uint4{pw[0], pw[1], pw[2], pw[3]};
                const uint4 pf_lo = low_parts<BF16>(pw, s[2 * st], s[2 * st + 1]);
                // the step's reads go out together, with one wait for them all
                v2u lower[DV / 16], upper[DV / 16];
                StepReads<DV / 16, (32 * st + 16 < L::VKEYS)>::template read<32 * st * ROW_BYTES, (32 * st + 16) * ROW_BYTES>(value_words, lower, upper);
#pragma unroll
                for (int dt = 0; dt < DV / 16; dt++) {
                    const uint4 vf = uint4{lower[dt][0], lower[dt][1], upper[dt][0], upper[dt][1]};
                    if constexpr (BY_STEP && st > 0) {
                        o[dt] = o[dt] + pv_steps<BF16>(vf, pf, pf_lo, v4f{0, 0, 0, 0});
                    } else {
                        o[dt] = pv_steps<BF16>(vf, pf, pf_lo, o[dt]);
                    }
                }
            });
            if constexpr (STAGED) {
                // over this query's own row of the head's queries: columns 16 dt + 4 quad .. + 4 are chunk 2 dt + quad / 2
                LDS_SPACE int8_t* row = raw_q + (buffer * per_kv + hi) * head_bytes;
#pragma unroll
                for (int dt = 0; dt < DV / 16; dt++) {
                    const uint2 result = uint2{narrow16x2<BF16>(o[dt][0] * inverse_total, o[dt][1] * inverse_total),
                                               narrow16x2<BF16>(o[dt][2] * inverse_total, o[dt][3] * inverse_total)};
                    lds_write8(row + raw_slot<KC>(query, 2 * dt + quad / 2) * 16 + (quad & 1) * 8, result);
                }
            } else if (query_ok) {
                half_t* to = out + (b * T + query) * (heads * DV) + head * DV + quad * 4;
#pragma unroll
                for (int dt = 0; dt < DV / 16; dt++) {
                    const uint2 result = uint2{narrow16x2<BF16>(o[dt][0] * inverse_total, o[dt][1] * inverse_total),
                                               narrow16x2<BF16>(o[dt][2] * inverse_total, o[dt][3] * inverse_total)};
                    *reinterpret_cast<uint2*>(to + dt * 16) = result;
                }
            }
        }
    }
    if constexpr (STAGED) {
        __builtin_amdgcn_s_waitcnt(0);   // this wavefront's staging writes are done (the compiler does not see them)
        __syncthreads();
        write_out(first_pair + groups_per_block - 1, (groups_per_block - 1) & 1);
    }
}

template <int DQP, int DV, int TILES, bool BF16>
int launch(const void* projected, const void* keyed, const void* q_gain, const void* k_gain, void* out, int B, int T, int heads,
           int kv_heads, int dq, int templates_count, int groups_per_block, float eps, float scale, hipStream_t stream)
{
    typedef Layout<DQP, DV, TILES> L;
    // (refused whichever kernel runs, so that what the operator takes does not depend on the tokens)
    const int bytes = L::bytes(heads / kv_heads);
    if (bytes > 160 * 1024)
        return chess_fail(CHESS_UNSUPPORTED, "template_attention would stage %d bytes of LDS for %d heads a key/value head", bytes, heads / kv_heads);
    // widths up to 64 and up to 80 tokens: attention_wave.h's kernel, which shares the pairs out by itself
    if constexpr (DQP <= 64 && DV <= 64 && TILES <= 5) {
        return launch_waves<DQP, DV, TILES, BF16>(projected, keyed, q_gain, k_gain, out, B, T, heads, kv_heads, dq, templates_count, eps, scale, stream);
    } else {
        auto kernel = template_attention_kernel<DQP, DV, TILES, BF16>;
        if (bytes > 65536) {
            const hipError_t allowed = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
            if (allowed != hipSuccess) return (int)allowed;
        }
        const dim3 grid((unsigned)((long)B * kv_heads / groups_per_block)), block(64 * L::WAVES);   // TILES == ceil(T / 16): the caller picked it so
        // (bf16 rows travel as 16-bit elements behind the same pointers: the kernel reads them only through widen16<BF16>)
        hipLaunchKernelGGL(kernel, grid, block, bytes, stream, (const half_t*)projected, (const half_t*)keyed, (const half_t*)q_gain,
                           (const half_t*)k_gain, (half_t*)out, T, heads, kv_heads, dq, templates_count, groups_per_block, eps, scale);
        return launch_status();
    }
}

template <int DQP, int DV, bool BF16>
int by_tokens(const void* projected, const void* keyed, const void* q_gain, const void* k_gain, void* out, int B, int T, int heads,
              int kv_heads, int dq, int templates_count, int groups_per_block, float eps, float scale, hipStream_t stream)
{
    auto launched = [&](auto tiles) {
        return launch<DQP, DV, decltype(tiles)::value, BF16>(projected, keyed, q_gain, k_gain, out, B, T, heads, kv_heads, dq, templates_count,
                                                             groups_per_block, eps, scale, stream);
    };
    switch ((T + 15) / 16) {
        case 4: return launched(std::integral_constant<int, 4>{});
        case 5: return launched(std::integral_constant<int, 5>{});
        case 6: return launched(std::integral_constant<int, 6>{});
        case 7: return launched(std::integral_constant<int, 7>{});
        default: return launched(std::integral_constant<int, 8>{});
    }
}

template <int DQP, bool BF16>
int by_dv(const void* projected, const void* keyed, const void* q_gain, const void* k_gain, void* out, int B, int T, int heads,
          int kv_heads, int dq, int dv, int templates_count, int groups_per_block, float eps, float scale, hipStream_t stream)
{
    switch (dv) {
        case 16: return by_tokens<DQP, 16, BF16>(projected, keyed, q_gain, k_gain, out, B, T, heads, kv_heads, dq, templates_count, groups_per_block, eps, scale, stream);
        case 32: return by_tokens<DQP, 32, BF16>(projected, keyed, q_gain, k_gain, out, B, T, heads, kv_heads, dq, templates_count, groups_per_block, eps, scale, stream);
        case 64: return by_tokens<DQP, 64, BF16>(projected, keyed, q_gain, k_gain, out, B, T, heads, kv_heads, dq, templates_count, groups_per_block, eps, scale, stream);
        default:
            if constexpr (BF16) return chess_fail(CHESS_UNSUPPORTED, "template_attention takes bf16 rows of value widths up to 64");
            else return by_tokens<DQP, 128, BF16>(projected, keyed, q_gain, k_gain, out, B, T, heads, kv_heads, dq, templates_count, groups_per_block, eps, scale, stream);
    }
}

}  // namespace

namespace {

template <bool BF16>
int template_attention(const void* projected, const void* keyed_templates, const void* q_gain, const void* k_gain, void* out, int B, int T,
                       int heads, int kv_heads, int dq, int dv, int templates_count, int groups_per_block, float eps, float scale, void* stream)
{
    if (B < 0 || T < 64 || T > 128)
        return chess_fail(CHESS_UNSUPPORTED, "template_attention takes 64 to 128 tokens a position, not %d", T);
    if (heads <= 0 || kv_heads <= 0 || heads % kv_heads != 0)
        return chess_fail(CHESS_INVALID_SHAPE, "%d heads cannot be split into groups for %d key/value heads", heads, kv_heads);
    if (dq <= 0 || dq > 128 || dq % 8 != 0) return chess_fail(CHESS_UNSUPPORTED, "template_attention takes query widths of 8 to 128 in steps of 8, not %d", dq);
    if (dv != 16 && dv != 32 && dv != 64 && dv != 128) return chess_fail(CHESS_UNSUPPORTED, "template_attention takes value widths 16, 32, 64 or 128, not %d", dv);
    if (BF16 && (dq > 64 || dv > 64)) return chess_fail(CHESS_UNSUPPORTED, "template_attention takes bf16 rows of query and value widths up to 64, not %d and %d", dq, dv);
    if (templates_count < 0 || templates_count > MAX_TEMPLATES)
        return chess_fail(CHESS_UNSUPPORTED, "template_attention takes at most %d templates, not %d", MAX_TEMPLATES, templates_count);
    if (groups_per_block <= 0 || ((long)B * kv_heads) % groups_per_block != 0)
        return chess_fail(CHESS_INVALID_SHAPE, "%d key/value groups a workgroup do not divide the %d positions' %d", groups_per_block, B, kv_heads);
    const int width = heads * dq + kv_heads * dq + kv_heads * dv + heads * templates_count;
    if (width % 8 != 0) return chess_fail(CHESS_MISALIGNED, "template_attention's vector loads need 16-byte aligned rows (row width %d halves)", width);
    if (B == 0) return CHESS_OK;   // no positions: nothing read or written, so the pointers may be null
    if (!projected || !keyed_templates || !q_gain || !k_gain || !out) return chess_fail(CHESS_INVALID_SHAPE, "template_attention: a required pointer is null");
    if (!aligned16(projected) || !aligned16(out) || !aligned16(keyed_templates))
        return chess_fail(CHESS_MISALIGNED, "template_attention's vector loads need 16-byte aligned rows (row width %d halves)", width);
    hipStream_t s = (hipStream_t)stream;
    if (dq <= 32) return by_dv<32, BF16>(projected, keyed_templates, q_gain, k_gain, out, B, T, heads, kv_heads, dq, dv, templates_count, groups_per_block, eps, scale, s);
    if constexpr (!BF16)
        if (dq > 64) return by_dv<128, BF16>(projected, keyed_templates, q_gain, k_gain, out, B, T, heads, kv_heads, dq, dv, templates_count, groups_per_block, eps, scale, s);
    return by_dv<64, BF16>(projected, keyed_templates, q_gain, k_gain, out, B, T, heads, kv_heads, dq, dv, templates_count, groups_per_block, eps, scale, s);
}

}  // namespace

extern "C" int chess_template_attention(const void* projected, const void* keyed_templates, const void* q_gain, const void* k_gain, void* out,
                                        int B, int T, int heads, int kv_heads, int dq, int dv, int templates_count, int groups_per_block,
                                        float eps, float scale, void* stream)
{
    return template_attention<false>(projected, keyed_templates, q_gain, k_gain, out, B, T, heads, kv_heads, dq, dv, templates_count,
                                     groups_per_block, eps, scale, stream);
}

extern "C" int chess_template_attention_bf16(const void* projected, const void* keyed_templates, const void* q_gain, const void* k_gain,
                                             void* out, int B, int T, int heads, int kv_heads, int dq, int dv, int templates_count,
                                             int groups_per_block, float eps, float scale, void* stream)
{
    return template_attention<true>(projected, keyed_templates, q_gain, k_gain, out, B, T, heads, kv_heads, dq, dv, templates_count,
                                    groups_per_block, eps, scale, stream);
}
