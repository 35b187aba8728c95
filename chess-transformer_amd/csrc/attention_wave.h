// The template attention's kernel for query and value widths up to 64 and up to 80 tokens (the networks' 70): each
// wavefront works by itself, from the projected rows to the stored outputs, and shares nothing but the templates with
// the others, so that after the start there is no barrier and a wavefront's waits are covered by the other wavefronts
// of its SIMD. (Before it, the slabs of 16 queries of a (position, key/value group) pair met at three barriers a head, to
// share the normalised keys; a compute unit held 8 such wavefronts, which waited for about half of their cycles.)
//
// Two ways of sharing out the pairs, with the same bits:
//   WHOLE   a wavefront takes whole pairs, slab after slab; the templates (64 KB) are in LDS. For launches of many
//           pairs: keys and values are read and normalised once a pair, 8 (widths up to 32: 12) pairs at once a compute unit.
//   FOURS   four wavefronts a pair, one a slab of 16 squares, the slab past the squares taken by one of them in turn, each
//           normalising the keys for itself; the templates come from global memory. The shorter chain, for small launches.
// Timed on an MI355X, as the launches of a graph (us, before and after): 70 tokens, 8 x 64 heads: batch 1024 98.6 and 67.1,
// 256 31.3 and 21.6, 64 13.1 and 11.0, 1 8.3 and 7.5; 24 on 12 heads, query width 16, value width 32: batch 700 201 and 80, 51
// 26.9 and 14.3; 8 x 32 heads: batch 999 84 and 41; 64 tokens, 8 x 64 heads in bf16: batch 4096 264 and 231. Bound by its VALU
// work beside waits that two wavefronts a SIMD do not cover: at batch 1024 the VALU is busy for half of the kernel's cycles;
// the rows alone would take 44 us at the rate of a large copy.
#pragma once

#include "attention_common.h"

namespace {

enum AttentionMode { WHOLE, FOURS };

template <int DQP, int DV, int TILES, AttentionMode MODE>
struct WaveLayout {
    static constexpr int STEPS = (TILES + 1) / 2;     // 32-key steps of P V
    static constexpr int KEYS = TILES * 16;
    static constexpr int KS = DQP / 32;               // MFMA steps of Q K
    static constexpr int VC = DV / 8;                 // 16-byte chunks a raw value row
    // value keys staged, whole DMA instructions of them (64 chunks): a half step of P V past them reads zeros
    static constexpr int VKEYS = (KEYS * VC + 63) / 64 * 64 / VC;
    static constexpr int V_DMA = VKEYS * VC / 64;
    static constexpr int V_BYTES = VKEYS * DV * 2;    // a wavefront's
    static constexpr bool NARROW = DQP <= 32 && DV <= 32;
    static constexpr int WAVES = MODE == WHOLE ? (NARROW ? 12 : 8) : 4;
    static constexpr int TEMPLATE_WORDS = MODE == WHOLE ? 64 * 64 : 1;   // 16-byte words in LDS
    // V^T's fragments held in registers over a pair's slabs (else read from LDS at each), and the next pair's raw keys loaded
    // while this one is taken: where the widths leave the registers (the narrow ones' 12 wavefronts have 168 each)
    static constexpr bool HELD_VALUES = DV <= 32, NEXT_KEYS = MODE == WHOLE && !NARROW;
    // With five tiles a slab's softmax sum and P V outputs are added by 32-key step, in step order
    static constexpr bool BY_STEP = TILES == 5;
    static_assert(TILES == 4 || TILES == 5, "four slabs of squares, and one past them");
};

// A transposing LDS read (ds_read_b64_tr_b16): in each 16 lanes, lane j receives element j % 4 of the 8 bytes lanes
// j / 4 + 4 r address, r = 0 .. 3
typedef short v4s __attribute__((ext_vector_type(4)));
DEVICE v2u read_transposed(const LDS_SPACE int8_t* p) {
    return __builtin_bit_cast(v2u, __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_SPACE v4s*)p));
}

// One half of a word of two fp16 values times b, and that half plus c, in one instruction each (v_fma_mix_f32 reads the
// half as it is): the f32 product's and sum's bits (a zero product is +0)
template <bool HIGH> DEVICE float half_times(uint32_t word, float b) {
    float out;
    if constexpr (HIGH) asm("v_fma_mix_f32 %0, %1, %2, 0 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(out) : "v"(word), "v"(b));
    else asm("v_fma_mix_f32 %0, %1, %2, 0 op_sel_hi:[1,0,0]" : "=v"(out) : "v"(word), "v"(b));
    return out;
}
template <bool HIGH> DEVICE float half_plus(uint32_t word, float c) {
    float out;
    if constexpr (HIGH) asm("v_fma_mix_f32 %0, %1, 1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(out) : "v"(word), "v"(c));
    else asm("v_fma_mix_f32 %0, %1, 1.0, %2 op_sel_hi:[1,0,0]" : "=v"(out) : "v"(word), "v"(c));
    return out;
}
// two f32 values as a word of fp16 (results of MFMAs: no product that the rounding could be fused into)
DEVICE uint32_t two_halves(float a, float b) { return __builtin_bit_cast(uint32_t, h2{(__fp16)a, (__fp16)b}); }

template <int DQP, int DV, int TILES, bool BF16, AttentionMode MODE>
__global__ __launch_bounds__((64 * WaveLayout<DQP, DV, TILES, MODE>::WAVES)) __attribute__((amdgpu_waves_per_eu(2)))
void template_attention_wave_kernel(
    const half_t* __restrict__ projected, const half_t* __restrict__ keyed, const half_t* __restrict__ q_gain,
    const half_t* __restrict__ k_gain, half_t* __restrict__ out, int T, int heads, int kv_heads, int dq, int templates_count,
    int pairs, float eps, float scale)
{
    typedef WaveLayout<DQP, DV, TILES, MODE> L;
    constexpr int KS = L::KS, VC = L::VC, STEPS = L::STEPS, DT = DV / 16;
    // (two arrays, so that the compiler can tell a read of the templates from the values' DMA in flight)
    __shared__ v4u template_words[L::TEMPLATE_WORDS];
    __shared__ __align__(16) int8_t value_rows[L::WAVES * L::V_BYTES];

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 15, quad = lane >> 4;
    const int width = heads * dq + kv_heads * dq + kv_heads * DV + heads * templates_count;
    const int k_offset = heads * dq, v_offset = k_offset + kv_heads * dq, c_offset = v_offset + kv_heads * DV;
    const int per_kv = heads / kv_heads;
    LDS_SPACE int8_t* values = (LDS_SPACE int8_t*)value_rows + wave * L::V_BYTES;

    // The template bias of a 16-key tile is an MFMA too: bias^T[k][q] = sum over (q', t) of templates[t][q'][k] *
    // [q' == q] c[q][t], an inner dimension of the slab's 16 queries x 8 templates, 32 a step. In step j the A operand lane
    // (key 16 kt + lane % 16, quad) holds keyed[q' = 16 slab + 4 j + quad][key][0..7] -- its query's 8 templates for the
    // key -- and the B operand lane (query col, quad) holds c[col][0..7] when 4 j + quad == col, else zeros.
    if constexpr (MODE == WHOLE) {
        // all the squares' templates, in LDS in the order the steps read them: [slab][key tile][step][lane]
        for (int i = tid; i < 64 * 64; i += 64 * L::WAVES) {
            const int q = i / 64, k = i % 64;
            const int place = ((q / 16 * 4 + k / 16) * 4 + q % 16 / 4) * 64 + q % 4 * 16 + k % 16;
            template_words[place] = reinterpret_cast<const v4u*>(keyed)[i];
        }
    }
    const LDS_SPACE int8_t* template_lane = (const LDS_SPACE int8_t*)template_words + lane * 16;

    // The lane's 16-byte chunks of a query or key row: columns ks * 32 + 8 quad .. + 8. Past dq a row's chunk holds another
    // head's columns (or lies past the row): read the row's first chunk there, as zeros
    bool live[KS];
    int chunk[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
        live[ks] = (ks * 4 + quad) * 8 < dq;
        chunk[ks] = live[ks] ? (ks * 4 + quad) * 8 : 0;
    }
    auto masked = [&](uint4 raw, bool keep) { return keep ? raw : uint4{0, 0, 0, 0}; };
    // their gains (2-byte aligned), each chunk one load: loaded element by element under a test of dq, every load would be
    // waited for by itself
    uint4 q_gains[KS], k_gains[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
        uint4 raw_q, raw_k;
        __builtin_memcpy(&raw_q, q_gain + chunk[ks], 16);
        __builtin_memcpy(&raw_k, k_gain + chunk[ks], 16);
        q_gains[ks] = masked(raw_q, live[ks]);
        k_gains[ks] = masked(raw_k, live[ks]);
    }
    // 1 / sqrt(mean of squares + eps). The mean is the quotient's bits without an IEEE divide: the product by the reciprocal
    // (rounded to nearest), corrected once by its remainder (an infinite sum keeps its infinite mean).
    const float columns = (float)dq, reciprocal_columns = 1.0f / columns;
    auto inverse_norm = [&](float squares) {
        const float near = squares * reciprocal_columns;
        const float corrected = __builtin_fmaf(__builtin_fmaf(-near, columns, squares), reciprocal_columns, near);
        const float mean = near < __builtin_inff() ? corrected : near;
        return 1.0f / __builtin_sqrtf(mean + eps);
    };
    auto normalised = [&](const uint4& raw, float inverse, const uint4& gains) {   // f16((x * inverse) * gain)
        const uint32_t x[4] = {raw.x, raw.y, raw.z, raw.w}, g[4] = {gains.x, gains.y, gains.z, gains.w};
        uint32_t normed[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            float low, high;
            if constexpr (BF16) {
                low = widen16<true>(x[i] & 0xFFFFu) * inverse;
                high = widen16<true>(x[i] >> 16) * inverse;
            } else {
                low = half_times<false>(x[i], inverse);
                high = half_times<true>(x[i], inverse);
            }
            normed[i] = narrow16x2<false>(half_times<false>(g[i], low), half_times<true>(g[i], high));
        }
        return __builtin_bit_cast(v8h, uint4{normed[0], normed[1], normed[2], normed[3]});
    };
    // A position's rows as a buffer: a load takes the lane's part of its address from a register and the rest from a scalar
    // one. Of the tile past the squares, whose rows may pass T, the whole row is in the lane's part, held to row T - 1 (such a
    // row's scores are masked, its outputs not stored): every load is inside the rows, whatever of an address a buffer's bounds
    // check counts.
    const uint32_t row_bytes = (uint32_t)width * 2;
    auto rows_of = [&](int pair) {
        return buffer_resource(projected + (size_t)(pair / kv_heads) * T * width, (uint32_t)T * row_bytes);
    };
    uint32_t lane_row[KS];   // the lane's chunks of row col
#pragma unroll
    for (int ks = 0; ks < KS; ks++) lane_row[ks] = (uint32_t)col * row_bytes + (uint32_t)chunk[ks] * 2;
    const uint32_t to_tail = (uint32_t)(min(64 + col, T - 1) - col) * row_bytes;   // from there to row 64 + col's
    uint4 raw_keys[TILES][KS];
    auto load_keys = [&](int pair) {
        const BufferResource rows = rows_of(pair);
        const uint32_t at = (uint32_t)(k_offset + pair % kv_heads * dq) * 2;
#pragma unroll
        for (int kt = 0; kt < TILES; kt++)
#pragma unroll
            for (int ks = 0; ks < KS; ks++)
                raw_keys[kt][ks] = kt < 4 ? buffer_load16(rows, lane_row[ks], at + kt * 16 * row_bytes) : buffer_load16(rows, lane_row[ks] + to_tail, at);
    };
    // a slab's query rows and template coefficients of head hi of a pair's
    uint4 raw_query[KS], raw_mix;
    auto load_query = [&](int pair, int hi, int slab) {
        const BufferResource rows = rows_of(pair);
        const int head = pair % kv_heads * per_kv + hi;
        const bool past = TILES > 4 && slab == 4;
        const uint32_t at = past ? 0 : (uint32_t)slab * 16 * row_bytes, shift = past ? to_tail : 0;
#pragma unroll
        for (int ks = 0; ks < KS; ks++) raw_query[ks] = buffer_load16(rows, lane_row[ks] + shift, at + (uint32_t)(head * dq) * 2);
        if (templates_count == MAX_TEMPLATES) {
            raw_mix = buffer_load16(rows, (uint32_t)col * row_bytes + shift, at + (uint32_t)(c_offset + head * MAX_TEMPLATES) * 2);
        } else {   // fewer than 8 coefficients start at any 2-byte place (past the squares a square's are read, and not used)
            const half_t* from = projected + ((size_t)(pair / kv_heads) * T + min(slab * 16 + col, 63)) * width + c_offset + head * templates_count;
            uint16_t c[MAX_TEMPLATES];
#pragma unroll
            for (int t = 0; t < MAX_TEMPLATES; t++) c[t] = t < templates_count ? __builtin_bit_cast(uint16_t, from[t]) : (uint16_t)0;
            raw_mix = uint4{c[0] | ((uint32_t)c[1] << 16), c[2] | ((uint32_t)c[3] << 16), c[4] | ((uint32_t)c[5] << 16),
                            c[6] | ((uint32_t)c[7] << 16)};
        }
    };
    auto load_values = [&](int pair) {   // the raw values, into LDS (rows past T: row T - 1 again)
        const BufferResource rows = rows_of(pair);
        const uint32_t at = (uint32_t)(v_offset + pair % kv_heads * DV) * 2;
        constexpr int DMA_ROWS = 64 / VC;
#pragma unroll
        for (int i = 0; i < L::V_DMA; i++) {
            const int lane_slot = lane / VC, row = i * DMA_ROWS + lane_slot, c = (lane % VC) ^ swizzle<VC>(row);
            // streamed (WHOLE): the values are read once, and past the caches they leave the output rows there for the combine
            // GEMM (67.1 against 70.4 us at batch 1024; the keys' and queries' rows, whose lines other heads read too, streamed
            // as well: 77.3)
            const bool squares = (i + 1) * DMA_ROWS <= 64;
            const uint32_t lane_at = (uint32_t)(squares ? lane_slot : min(row, T - 1)) * row_bytes + c * 16, row_at = squares ? i * DMA_ROWS * row_bytes : 0;
            if constexpr (MODE == WHOLE) buffer_dma16_streamed(rows, (LDS_SPACE void*)(values + i * 1024), lane_at, at + row_at);
            else buffer_dma16(rows, (LDS_SPACE void*)(values + i * 1024), lane_at, at + row_at);
        }
    };
    // the templates of the wavefront's own slab, in the steps' order (FOURS)
    v4u slab_templates[MODE == WHOLE ? 1 : 4][4];
    auto load_templates = [&] {
        if constexpr (MODE != WHOLE) {
            const half_t* from = keyed;
            asm volatile("" : "+s"(from));   // loaded for each pair (they are near): kept for all, their 64 registers would spill others
            const BufferResource all = buffer_resource(from, 64 * 64 * MAX_TEMPLATES * 2);
#pragma unroll
            for (int kt = 0; kt < 4; kt++)
#pragma unroll
                for (int j = 0; j < 4; j++)
                    slab_templates[kt][j] = __builtin_bit_cast(v4u, buffer_load16(all, (uint32_t)(quad * 64 + col) * 16, (uint32_t)((wave * 16 + 4 * j) * 64 + kt * 16) * 16));
        }
    };
    // the bias MFMAs' B operands: this query's coefficients in the one step j with 4 j + quad == col
    auto coefficients = [&](v8h (&mix)[4]) {
        uint4 c = raw_mix;
        if constexpr (BF16) c = bf16_to_f16x8(c);
#pragma unroll
        for (int j = 0; j < 4; j++) mix[j] = __builtin_bit_cast(v8h, masked(c, 4 * j + quad == col));
    };
    auto rounded_bias = [&](const v4u (&operands)[4], const v8h (&mix)[4]) {   // of the lane's 4 keys of a tile, in fp16
        v4f bias = v4f{0, 0, 0, 0};
#pragma unroll
        for (int j = 0; j < 4; j++) bias = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, operands[j]), mix[j], bias, 0, 0, 0);
        return uint2{two_halves(bias[0], bias[1]), two_halves(bias[2], bias[3])};
    };
    uint2 slab_bias[4];
    auto take_slab_bias = [&] {   // the wavefront's own slab's (FOURS)
        if constexpr (MODE != WHOLE) {
            v8h mix[4];
            coefficients(mix);
#pragma unroll
            for (int kt = 0; kt < 4; kt++) slab_bias[kt] = rounded_bias(slab_templates[kt], mix);
        }
    };

    // the workgroup's share of the pairs: its wavefronts take them in turn (WHOLE), or each takes its slab of all of them
    const int share = pairs / (int)gridDim.x, more = pairs % (int)gridDim.x, block = blockIdx.x;
    const int first = share * block + min(block, more) + (MODE == WHOLE ? wave : 0);
    const int last = share * (block + 1) + min(block + 1, more);
    constexpr int STRIDE = MODE == WHOLE ? L::WAVES : 1;
    if constexpr (MODE == WHOLE) __syncthreads();   // the templates are in place
    if (first >= last) return;

    if constexpr (MODE == WHOLE) {
        load_keys(first);
        load_query(first, 0, 0);
    }
    int turn = wave / 4;
    for (int pair = first; pair < last; pair += STRIDE) {
        const int group = pair % kv_heads;
        const bool more_pairs = pair + STRIDE < last;
        if constexpr (MODE == WHOLE) {
            // The wavefronts of a SIMD take the higher priorities in turn, a pair each: left to the hardware's order the oldest
            // finishes its pairs long before the others, which then run with nothing to cover their waits (74.8 against 79.4 us
            // at batch 1024 of 8 x 64 heads).
            switch (turn++ % (L::WAVES / 4)) {
                case 0: __builtin_amdgcn_s_setprio(0); break;
                case 1: __builtin_amdgcn_s_setprio(1); break;
                default: __builtin_amdgcn_s_setprio(2);
            }
            __builtin_amdgcn_s_waitcnt(0);   // this pair's keys and first queries, loaded while the one before was taken
            load_values(pair);
        } else {
            // everything the pair needs, in flight together
            load_query(pair, 0, wave);
            load_keys(pair);
            load_templates();
            load_values(pair);
            take_slab_bias();
            __builtin_amdgcn_sched_barrier(0);   // the templates' registers are free before the keys are normalised
        }

        // the keys: k' = f16((k * (1 / sqrt(mean of squares + eps))) * k_gain). The sum of squares runs over each quarter of
        // the row's chunks in order, the quarters added as (a + b) + (c + d): with one chunk a quad, the quads' sums; with two
        // (chunks 2 p and 2 p + 1, held by neighbouring quads), the odd quad going on from its neighbour's sum.
        v8h keys[TILES][KS];
        float key_squares[TILES];
#pragma unroll
        for (int kt = 0; kt < TILES; kt++) {
            if constexpr (KS == 1) {
                raw_keys[kt][0] = masked(raw_keys[kt][0], live[0]);
                key_squares[kt] = sum_across_rows(squares8<BF16>(raw_keys[kt][0], 0.0f));
            } else {
                float quarter[KS];
#pragma unroll
                for (int ks = 0; ks < KS; ks++) {
                    raw_keys[kt][ks] = masked(raw_keys[kt][ks], live[ks]);
                    const float own = squares8<BF16>(raw_keys[kt][ks], 0.0f);
                    const auto from = __builtin_amdgcn_permlane16_swap(__float_as_uint(own), __float_as_uint(own), false, false);
                    const float both = squares8<BF16>(raw_keys[kt][ks], __uint_as_float(from[0]));
                    const auto odd = __builtin_amdgcn_permlane16_swap(__float_as_uint(both), __float_as_uint(both), false, false);
                    quarter[ks] = sum_halves32(__uint_as_float(odd[1]));
                }
                key_squares[kt] = quarter[0] + quarter[1];
            }
        }
        // the first four tiles' divide and root are taken once, a tile a quad, and handed to every quad by lane swaps
        float key_inverse[TILES];
        {
            const float mine = quad == 0 ? key_squares[0] : quad == 1 ? key_squares[1] : quad == 2 ? key_squares[2] : key_squares[3];
            const uint32_t inverse = __float_as_uint(inverse_norm(mine));
            const auto even_odd = __builtin_amdgcn_permlane16_swap(inverse, inverse, false, false);   // quads 0, 0, 2, 2 and 1, 1, 3, 3
            const auto even = __builtin_amdgcn_permlane32_swap(even_odd[0], even_odd[0], false, false);
            const auto odd = __builtin_amdgcn_permlane32_swap(even_odd[1], even_odd[1], false, false);
            key_inverse[0] = __uint_as_float(even[0]), key_inverse[1] = __uint_as_float(odd[0]);
            key_inverse[2] = __uint_as_float(even[1]), key_inverse[3] = __uint_as_float(odd[1]);
        }
        if constexpr (TILES > 4) key_inverse[4] = inverse_norm(key_squares[4]);
#pragma unroll
        for (int kt = 0; kt < TILES; kt++)
#pragma unroll
            for (int ks = 0; ks < KS; ks++) keys[kt][ks] = normalised(raw_keys[kt][ks], key_inverse[kt], k_gains[ks]);

        __builtin_amdgcn_s_waitcnt(0);   // the values have landed (with no DMA in flight, no read of them waits again)
        if (L::NEXT_KEYS && more_pairs) load_keys(pair + STRIDE);

        // V^T's fragments: half h (positions 4 h ..) of lane (col, quad) is V[32 st + 16 h + 4 quad + r][16 dt + col], r =
        // 0..3: a transposing read in which lane 4 r' + g of the 16 addresses the 4 values of key 32 st + 16 h + 4 quad + r',
        // columns 16 dt + 4 g .. + 3 (half g % 2 of chunk 2 dt + g / 2). The swizzle of a row repeats every 16 rows.
        const int value_row = 4 * quad + col / 4, value_group = col % 4;
        const LDS_SPACE int8_t* value_base[DT];
#pragma unroll
        for (int dt = 0; dt < DT; dt++) value_base[dt] = values + raw_slot<VC>(value_row, 2 * dt + value_group / 2) * 16 + (value_group % 2) * 8;
        auto read_values = [&](int st, v2u (&lo)[DT], v2u (&hi)[DT]) {
            constexpr int ROW_BYTES = VC * 16;
#pragma unroll
            for (int dt = 0; dt < DT; dt++) {
                lo[dt] = read_transposed(value_base[dt] + 32 * st * ROW_BYTES);
                hi[dt] = 32 * st + 16 < L::VKEYS ? read_transposed(value_base[dt] + (32 * st + 16) * ROW_BYTES) : v2u{0, 0};
            }
        };
        v2u lower[L::HELD_VALUES ? STEPS : 1][DT], upper[L::HELD_VALUES ? STEPS : 1][DT];
        if constexpr (L::HELD_VALUES) {
#pragma unroll
            for (int st = 0; st < STEPS; st++) read_values(st, lower[st], upper[st]);
        }

        // A slab of a head's queries, raw in raw_query; SQUARES: they are squares, with the template bias. Once they are
        // normalised, the rows of the slab taken next are loaded (next_pair < 0: none).
        auto take_slab = [&](int hi, int slab, int next_pair, int next_hi, int next_slab, auto squares_here) {
            constexpr bool SQUARES = decltype(squares_here)::value;
            const int head = group * per_kv + hi;
            // q' = f16((q * (1 / sqrt(mean of squares + eps))) * q_gain): the fragment of B, columns ks * 32 + 8 quad .. + 8
            v8h qf[KS], mix[4];
            float squares = 0.0f;
#pragma unroll
            for (int ks = 0; ks < KS; ks++) {
                raw_query[ks] = masked(raw_query[ks], live[ks]);
                squares = squares8<BF16>(raw_query[ks], squares);
            }
            const float q_inverse = inverse_norm(sum_across_rows(squares));
#pragma unroll
            for (int ks = 0; ks < KS; ks++) qf[ks] = normalised(raw_query[ks], q_inverse, q_gains[ks]);
            if constexpr (MODE == WHOLE && SQUARES) coefficients(mix);
            if (next_pair >= 0) load_query(next_pair, next_hi, next_slab);

            // S^T tiles: lane holds s[query][16 kt + 4 quad + r]; square keys take the template bias, keys past T are masked
            float s[2 * STEPS][4];
            float top = -__builtin_inff();
#pragma unroll
            for (int kt = 0; kt < 2 * STEPS; kt++) {
                if (kt >= TILES) {
#pragma unroll
                    for (int r = 0; r < 4; r++) s[kt][r] = -__builtin_inff();
                    continue;
                }
                v4f acc = v4f{0, 0, 0, 0};
#pragma unroll
                for (int ks = 0; ks < KS; ks++) acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(keys[kt][ks], qf[ks], acc, 0, 0, 0);
                uint2 rounded = uint2{0, 0};
                if constexpr (SQUARES) {
                    if (kt < 4) {
                        if constexpr (MODE == WHOLE) {
                            v4u operands[4];
#pragma unroll
                            for (int j = 0; j < 4; j++)
                                operands[j] = *reinterpret_cast<const LDS_SPACE v4u*>(template_lane + slab * 16384 + (kt * 4 + j) * 1024);
                            rounded = rounded_bias(operands, mix);
                        } else {
                            rounded = slab_bias[kt];
                        }
                    }
                }
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    float value = acc[r] * scale;
                    if (kt < 4) {
                        if constexpr (SQUARES) value = r % 2 ? half_plus<true>(r / 2 ? rounded.y : rounded.x, value) : half_plus<false>(r / 2 ? rounded.y : rounded.x, value);
                    } else if (kt * 16 + quad * 4 + r >= T) {
                        value = -__builtin_inff();
                    }
                    s[kt][r] = value;
                    top = fmaxf(top, value);
                }
            }
            const float offset = -max_across_rows(top) * LOG2E;
            float total = 0.0f;
#pragma unroll
            for (int st = 0; st < STEPS; st++) {
                float step_total = 0.0f;
#pragma unroll
                for (int kt = 2 * st; kt < 2 * st + 2; kt++)
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const float p = kt < TILES ? __builtin_amdgcn_exp2f(__builtin_fmaf(s[kt][r], LOG2E, offset)) : 0.0f;
                        s[kt][r] = p;
                        if constexpr (L::BY_STEP) step_total = kt == 2 * st && r == 0 ? p : kt < TILES ? step_total + p : step_total;
                        else total = kt == 0 && r == 0 ? p : total + p;
                    }
                // with five tiles each step's sum across the wavefront, then the steps' sums in order
                if constexpr (L::BY_STEP) {
                    step_total = sum_across_rows(step_total);
                    total = st == 0 ? step_total : total + step_total;
                }
            }
            if constexpr (!L::BY_STEP) total = sum_across_rows(total);
            const float inverse_total = __builtin_amdgcn_rcpf(total);

            // O^T = V^T P^T over 32-key steps: position e of both operands is key 32 st + 16 (e / 4) + 4 quad + e % 4
            v4f o[DT];
#pragma unroll
            for (int dt = 0; dt < DT; dt++) o[dt] = v4f{0, 0, 0, 0};
#pragma unroll
            for (int st = 0; st < STEPS; st++) {
                const int at = L::HELD_VALUES ? st : 0;
                uint32_t pw[4];
#pragma unroll
                for (int r = 0; r < 2; r++) {
                    pw[r] = narrow16x2<BF16>(s[2 * st][2 * r], s[2 * st][2 * r + 1]);
                    pw[2 + r] = narrow16x2<BF16>(s[2 * st + 1][2 * r], s[2 * st + 1][2 * r + 1]);
                }
                const uint4 pf = uint4{pw[0], pw[1], pw[2], pw[3]};
                const uint4 pf_lo = low_parts<BF16>(pw, s[2 * st], s[2 * st + 1]);
                if constexpr (!L::HELD_VALUES) read_values(st, lower[at], upper[at]);
#pragma unroll
                for (int dt = 0; dt < DT; dt++) {
                    const uint4 vf = uint4{lower[at][dt][0], lower[at][dt][1], upper[at][dt][0], upper[at][dt][1]};
                    if (L::BY_STEP && st > 0) {
                        o[dt] = o[dt] + pv_steps<BF16>(vf, pf, pf_lo, v4f{0, 0, 0, 0});
                    } else {
                        o[dt] = pv_steps<BF16>(vf, pf, pf_lo, o[dt]);
                    }
                }
            }
            // the lane's outputs of its query: columns 16 dt + 4 quad .. + 3; neighbouring quads trade (v_permlane16_swap) the
            // even column group's words of one for the odd group's of the other, so that each lane stores 16 bytes
            uint2 words[DT];
#pragma unroll
            for (int dt = 0; dt < DT; dt++)
                words[dt] = uint2{narrow16x2<BF16>(o[dt][0] * inverse_total, o[dt][1] * inverse_total),
                                  narrow16x2<BF16>(o[dt][2] * inverse_total, o[dt][3] * inverse_total)};
            const BufferResource outs = buffer_resource(out + (size_t)(pair / kv_heads) * T * (heads * DV), (uint32_t)(T * heads * DV) * 2);
            // (past the squares as the loads: the whole row in the lane's part, and for rows past T a part past any buffer,
            // which stores nothing)
            const uint32_t out_bytes = (uint32_t)(heads * DV) * 2, at = (SQUARES ? (uint32_t)slab * 16 * out_bytes : 0) + (uint32_t)(head * DV) * 2;
            const uint32_t lane_at = SQUARES ? col * out_bytes : 64 + col < T ? (64 + col) * out_bytes : 0x80000000u;
            if constexpr (DT == 1) {
                buffer_store8(outs, words[0], lane_at + quad * 8, at);
            } else {
#pragma unroll
                for (int dp = 0; dp < DT / 2; dp++) {
                    const auto x = __builtin_amdgcn_permlane16_swap(words[2 * dp].x, words[2 * dp + 1].x, false, false);
                    const auto y = __builtin_amdgcn_permlane16_swap(words[2 * dp].y, words[2 * dp + 1].y, false, false);
                    buffer_store16(outs, v4u{x[0], y[0], x[1], y[1]}, lane_at + 32 * (quad & 1) + 16 * (quad >> 1), at + 64 * dp);
                }
            }
        };
        constexpr auto SQUARES = std::true_type{};
        constexpr auto OTHERS = std::false_type{};
        for (int hi = 0; hi < per_kv; hi++) {
            const bool more_heads = hi + 1 < per_kv;
            if constexpr (MODE == WHOLE) {
                // what follows the head's last slab: the next head's first, or the next pair's
                const int next_pair = more_heads ? pair : more_pairs ? pair + STRIDE : -1, next_hi = more_heads ? hi + 1 : 0;
#pragma unroll 1
                for (int slab = 0; slab < 4; slab++) {
                    const bool on = slab + 1 < TILES;
                    take_slab(hi, slab, on ? pair : next_pair, on ? hi : next_hi, on ? slab + 1 : 0, SQUARES);
                }
                if constexpr (TILES > 4) take_slab(hi, 4, next_pair, next_hi, 0, OTHERS);
            } else {
                const int next_pair = more_heads ? pair : -1;
                if (hi > 0) {
                    load_templates();
                    take_slab_bias();
                }
                const bool tail = TILES > 4 && (block + hi) % 4 == wave;   // this head's slab past the squares is this wavefront's too
                take_slab(hi, wave, tail ? pair : next_pair, tail ? hi : hi + 1, tail ? 4 : wave, SQUARES);
                if constexpr (TILES > 4)
                    if (tail) take_slab(hi, 4, next_pair, hi + 1, wave, OTHERS);
            }
        }
        if (MODE == WHOLE && !L::NEXT_KEYS && more_pairs) load_keys(pair + STRIDE);
    }
}

// The launch's mode by n, its pairs a compute unit (rounded up). FOURS's workgroups of four wavefronts, one a SIMD each,
// take a time that grows with n; WHOLE's wavefronts, one or two (narrow widths: up to three) a SIMD, much the same for n of
// 1 to 4 and of 5 to 8, and longer the more heads a pair has. So a head a pair takes WHOLE from n = 3 (4 where the values
// are wider than the queries), several heads from 4, but three or more not at 5, nor, of narrow widths over five tiles, two
// or more up to 6. Timed both ways on an MI355X (us, FOURS and WHOLE, at 512, 768, 1,024, 1,280 and 1,536 pairs): 8 x 64
// heads over 64 tokens 9.3 and 9.9, 12.4 and 11.1, 16.6 and 12.0, 18.4 and 14.7, 22.5 and 15.8, over 70 10.8 and 12.1, 14.2
// and 13.2, 18.0 and 14.2, 20.3 and 18.6, 25.0 and 19.7; 16 on 4 x 32 over 64 tokens 13.4 and 20.1, 17.8 and 21.6, 22.4 and
// 22.2, 26.1 and 29.1, 30.2 and 29.8, over 70 17.3 and 25.5, 21.8 and 26.9, 27.0 and 28.1, 31.6 and 37.4, 36.0 and 37.9; 24
// on 12, query width 16, value width 32, over 70 11.3 and 14.7, 14.3 and 15.6, 18.1 and 16.2, 19.7 and 22.2, 22.4 and 23.0;
// past 1,536 pairs WHOLE wins everywhere. Its workgroups, one a compute unit, share the pairs out evenly however few they
// are: filled with a pair for each wavefront instead, 1,024 pairs of 16 on 4 x 32 heads over 64 tokens had 86 workgroups
// and took 36.0 us, where the kernel before this one took 23.9 (70 tokens, 8 x 64 heads, 1,032 pairs: 18.5 against 16.6
// now).
template <int DQP, int DV, int TILES, bool BF16>
int launch_waves(const void* projected, const void* keyed, const void* q_gain, const void* k_gain, void* out, int B, int T, int heads,
                 int kv_heads, int dq, int templates_count, float eps, float scale, hipStream_t stream)
{
    int device = 0, units = 0;
    if (hipError_t status = hipGetDevice(&device); status != hipSuccess) return (int)status;
    if (hipError_t status = hipDeviceGetAttribute(&units, hipDeviceAttributeMultiprocessorCount, device); status != hipSuccess) return (int)status;
    const int pairs = B * kv_heads;
    auto launch = [&](auto chosen, int workgroups) {   // sharing the pairs out evenly
        constexpr AttentionMode MODE = decltype(chosen)::value;
        hipLaunchKernelGGL((template_attention_wave_kernel<DQP, DV, TILES, BF16, MODE>), dim3(workgroups),
                           dim3(64 * WaveLayout<DQP, DV, TILES, MODE>::WAVES), 0, stream, (const half_t*)projected, (const half_t*)keyed,
                           (const half_t*)q_gain, (const half_t*)k_gain, (half_t*)out, T, heads, kv_heads, dq, templates_count, pairs, eps, scale);
        return launch_status();
    };
    typedef WaveLayout<DQP, DV, TILES, WHOLE> L;
    const int n = (pairs + units - 1) / units;
    const bool fours = heads == kv_heads ? n <= (DV > DQP ? 3 : 2) : L::NARROW && TILES == 5 ? n <= 6 : n <= 3 || (n == 5 && heads > 2 * kv_heads);
    if (fours) return launch(std::integral_constant<AttentionMode, FOURS>{}, min((L::NARROW ? 4 : 2) * units, pairs));
    return launch(std::integral_constant<AttentionMode, WHOLE>{}, min(units, pairs));
}

}  // namespace
