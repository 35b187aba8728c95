// The GEMM with the weights held in registers: out[M, N] = epilogue(x[M, K] @ w[N, K]^T), for int8 operands (int32 sums, K =
// 256, 512, 768 or 1,024) and for fp16 ones (f32 sums, K = 256 or 512), with gemm_tiles.h's epilogues and op order
// (dequantise, bias, SiLU * up, residual, the next block's mix, round), so that it gives the other tiles' bits. Depth 512 is
// tile 15; the others are launched by tile 0 alone.
//
// A wavefront owns 32 output columns and holds their weights for the whole depth in up to 128 VGPRs: int8 up to depth 512, two
// fragments of 32 weight rows (gated: the gate's 32 rows and up's 32; else 64 columns); int8 past it and fp16, one (gated:
// 16 of the gate's rows and 16 of up's, whose sums meet in a lane too). A workgroup of eight wavefronts (two a
// SIMD, one workgroup a compute unit) owns a column group of 256 (or 512) columns and walks a stream of 32-row blocks of
// x, each block (16 KB of int8, 32 KB of fp16) arriving by DMA into a ring of four LDS stages: per block, every wavefront
// reads the block's operands from LDS and runs its MFMAs into one of two sets of sums, while the epilogue of the block
// before runs between them from the other set, stored straight from registers, 16 bytes a lane. The K-loop of the
// whole-tile kernels moves both operands through LDS at every step; here only x moves, once a block for the workgroup,
// and the weights never leave the registers.
//
// An MFMA step is 32 bytes of K: lane l holds 16 bytes of row l % 32, bytes 32 t + 16 (l / 32) .. at step t, for the
// weights in registers and for x in LDS alike -- the whole-tile kernels' order, so that the fp16 sums round as theirs do
// (the int32 sums are exact in any order). A block's row r sits in LDS as 16-byte chunks, chunk c at slot c ^ (r % 16):
// the 16 rows an operand read takes at one step fall in 16 different 16-byte bank groups. A DMA instruction writes 1 KB
// of LDS (two int8 rows or one fp16 row), each lane loading the chunk of x that belongs in its slot.
//
// Workgroups are spread over the XCDs (the hardware deals them out round-robin, blockIdx % 8) so that each XCD takes
// contiguous streams of row blocks with every column group: the column groups of a stream read its blocks from the
// XCD's own L2, and x leaves HBM about once.
#pragma once

#include "gemm.h"
#include "lds_dma.h"

#include <algorithm>
#include <type_traits>

namespace resident {

using namespace gemm;

typedef int v16i_r __attribute__((ext_vector_type(16)));
typedef float v16f_r __attribute__((ext_vector_type(16)));

constexpr int DEPTH = 512;      // tile 15's K; tile 0 also takes the kernel's other depths (takes)
constexpr int ROWS = 32;        // rows of x a block
constexpr int WAVES = 8;
constexpr int STAGES = 4;
constexpr int XCDS = 8;

template <typename In> struct Mma;
template <> struct Mma<int8_t> {
    typedef v4i Operand;
    typedef v16i_r Sums;
    static DEVICE Sums step(Operand w, Operand x, Sums c) { return __builtin_amdgcn_mfma_i32_32x32x32_i8(w, x, c, 0, 0, 0); }
    static DEVICE float value(Sums c, int r) { return (float)c[r]; }
};
template <> struct Mma<half_t> {
    typedef v8h Operand;
    typedef v16f_r Sums;
    static DEVICE Sums step(Operand w, Operand x, Sums c) { return __builtin_amdgcn_mfma_f32_32x32x16_f16(w, x, c, 0, 0, 0); }
    static DEVICE float value(Sums c, int r) { return c[r]; }
};

template <typename In, int NB, int EPI, int DEPTH_> struct Shape {
    static constexpr bool INT8 = std::is_same<In, int8_t>::value;
    static constexpr bool BIAS = (EPI & EPI_BIAS) != 0, RESIDUAL = (EPI & EPI_RESIDUAL) != 0, MIX = (EPI & EPI_MIX) != 0;
    static constexpr int ROW_BYTES = DEPTH_ * (int)sizeof(In);     // 256 to 1,024, a multiple of 256
    static constexpr int STEPS = ROW_BYTES / 32;                    // MFMA steps
    static constexpr int CHUNKS = ROW_BYTES / 16;                   // 16-byte chunks a row
    static constexpr int BLOCK_BYTES = ROWS * ROW_BYTES;
    // weight fragments of 32 rows a wavefront holds: two while they fit in 128 VGPRs beside the sums, so that an operand read
    // from LDS serves two MFMAs; else one (gated: 16 of the gate's rows and 16 of up's)
    static constexpr int FRAGMENTS = INT8 && ROW_BYTES <= 512 ? 2 : 1;
    static constexpr int COLUMNS = 32 * FRAGMENTS / NB;             // output columns a wavefront
    static constexpr int PER_LANE = COLUMNS / 2;                    // outputs a lane
    static constexpr int GROUP = WAVES * COLUMNS;                   // a workgroup's column group
    static constexpr int ROW_DMA = BLOCK_BYTES / 1024 / WAVES;      // a wavefront's 1 KB DMA instructions a block
    static constexpr int DMA_OPS = ROW_DMA + (INT8 ? 1 : 0);        // and (int8) the block's row scales
    static constexpr int STORE_OPS = COLUMNS / 16;                  // a wavefront's 16-byte stores a block
    static constexpr int LOAD_OPS = (RESIDUAL ? COLUMNS / 16 : 0) + (MIX ? COLUMNS / 16 : 0);   // and its 16-byte residual and input loads
    // LDS: the ring's stages, (int8) each stage's row scales, a copy a wavefront, a word a lane, then each wavefront's
    // column vectors (64 weight scales, 64 biases)
    static constexpr int SCALE_BYTES = WAVES * 64 * 4;
    static constexpr int SCALES_AT = STAGES * BLOCK_BYTES;
    static constexpr int VECTORS_AT = SCALES_AT + (INT8 ? STAGES * SCALE_BYTES : 0);
    static constexpr int LDS_BYTES = VECTORS_AT + WAVES * 128 * 4;
    // Vector memory operations this wavefront has surely issued after the last one of block b's DMA when block b is to
    // be read: the prologue's later blocks, then every turn after the one that issued it (block b - STAGES + 1's) and
    // before b's, each with its DMA and (but block 0's) the stores and residual loads of the block before it. Within a
    // turn they interleave, so the issuing turn's own are not counted. Operations complete in issue order, so waiting
    // for at most that many outstanding means block b has landed.
    static constexpr int after(int b) {
        const int issuing = b - (STAGES - 1);
        int ops = issuing < 0 ? DMA_OPS * (STAGES - 2 - b) : 0;
        for (int t = issuing + 1 > 0 ? issuing + 1 : 0; t < b; t++) ops += DMA_OPS + (t >= 1 ? STORE_OPS + LOAD_OPS : 0);
        return ops;
    }
    static_assert(ROW_BYTES % 256 == 0 && ROW_BYTES <= 1024 && STORE_OPS >= 1 && (RESIDUAL || !MIX) && !(NB == 2 && RESIDUAL), "shape");
};

// A lane's 4-column groups q = 2 p and 2 p + 1 (columns 8 q + 4 (l / 32) ..), packed, traded between lanes l and l + 32
// (v_permlane32_swap: lanes 32-63 of the first with lanes 0-31 of the second): lane l then holds columns 16 p .. 16 p + 7
// of its row and lane l + 32 columns 16 p + 8 .. 16 p + 15, in order, for one 16-byte store each.
DEVICE v4u eight_columns(uint2 even, uint2 odd) {
    const auto x = __builtin_amdgcn_permlane32_swap(even.x, odd.x, false, false);
    const auto y = __builtin_amdgcn_permlane32_swap(even.y, odd.y, false, false);
    return v4u{x[0], y[0], x[1], y[1]};
}
// the same trade of f32 values: the lane's 8 columns, in order
DEVICE void eight_values(const float (&even)[4], const float (&odd)[4], float (&to)[8]) {
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const auto pair = __builtin_amdgcn_permlane32_swap(__float_as_uint(even[j]), __float_as_uint(odd[j]), false, false);
        to[j] = __uint_as_float(pair[0]);
        to[4 + j] = __uint_as_float(pair[1]);
    }
}

template <typename OutT> DEVICE uint2 pack_four(const float (&v)[4]);
template <> DEVICE uint2 pack_four<half_t>(const float (&v)[4]) {
    const v4h four = v4h{(half_t)v[0], (half_t)v[1], (half_t)v[2], (half_t)v[3]};
    return __builtin_bit_cast(uint2, four);
}
template <> DEVICE uint2 pack_four<bf16_t>(const float (&v)[4]) {
    return uint2{bf16_pair(v[0], v[1]), bf16_pair(v[2], v[3])};
}

template <typename In, int NB, typename OutT, int EPI, int DEPTH_>
__global__ __launch_bounds__(64 * WAVES, 1) void resident_kernel(
    const In* __restrict__ x, const In* __restrict__ w, OutT* __restrict__ out, Epilogue e, int M, int N, int groups, int slices,
    int last_slices)
{
    typedef Shape<In, NB, EPI, DEPTH_> S;
    typedef Mma<In> MMA;
    typedef typename MMA::Operand Operand;
    constexpr int STEPS = S::STEPS, ROW_BYTES = S::ROW_BYTES, FRAGMENTS = S::FRAGMENTS, COLUMNS = S::COLUMNS;
    extern __shared__ __align__(16) int8_t lds[];
    LDS_SPACE int8_t* ring = (LDS_SPACE int8_t*)lds;

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int in_row = lane & 31, half = lane >> 5;

    // the workgroup's column group and stream of row blocks: each XCD's workgroups take `slices` streams of every column
    // group but the last, which takes `last_slices`
    const int xcd = blockIdx.x % XCDS, local = blockIdx.x / XCDS;
    const int full_workgroups = (groups - 1) * slices;
    if (local >= full_workgroups + last_slices) return;
    const bool in_last = local >= full_workgroups;
    const int group = in_last ? groups - 1 : local % max(groups - 1, 1);
    const int group_slices = in_last ? last_slices : slices;
    const int stream = xcd * group_slices + (in_last ? local - full_workgroups : local / max(groups - 1, 1)), streams = XCDS * group_slices;
    const int blocks = (M + ROWS - 1) / ROWS;
    const int first = (int)((long)stream * blocks / streams), count = (int)((long)(stream + 1) * blocks / streams) - first;
    if (count <= 0) return;
    const int n_wave = group * S::GROUP + wave * S::COLUMNS;   // the wavefront's first output column
    // a wavefront whose columns all lie past N only moves its share of the data (not with a residual to load)
    const bool idle = !S::RESIDUAL && n_wave >= N;

    // the weights: fragment f is 32 weight rows (gated: the gate's rows, then up's; else columns 32 f ..), lane l holding
    // row l % 32's bytes 32 t + 16 (l / 32) .. at step t. Columns past N read column N - 1 (never stored).
    const BufferResource w_rsrc = buffer_resource(w, (uint32_t)NB * (uint32_t)N * ROW_BYTES);
    Operand weights[FRAGMENTS][STEPS];
#pragma unroll
    for (int f = 0; f < FRAGMENTS && !idle; f++) {
        const int at_row = 32 * f + in_row;   // of the wavefront's weight rows: gated, the gate's COLUMNS, then up's
        const int row = NB == 2 ? at_row / COLUMNS * N + min(n_wave + at_row % COLUMNS, N - 1) : min(n_wave + at_row, N - 1);
#pragma unroll
        for (int t = 0; t < STEPS; t++)
            weights[f][t] = __builtin_bit_cast(Operand, buffer_load16(w_rsrc, (uint32_t)row * ROW_BYTES + 16 * half, 32 * t));
    }

    // The ring's DMA: this wavefront's ROWS / WAVES rows of a block, 1 KB an instruction, lane l writing slot l % CHUNKS
    // of its row from that row's chunk (l % CHUNKS) ^ (row % 16); rows past M read row M - 1. Then (int8) the block's 32
    // row scales, into the wavefront's own copy.
    const BufferResource x_rsrc = buffer_resource(x, (uint32_t)M * ROW_BYTES);
    const BufferResource scale_rsrc = buffer_resource(S::INT8 ? (const void*)e.x_scale : (const void*)x, (uint32_t)M * 4);
    auto issue_one = [&](int b, int stage, int i) {   // DMA instruction i of block b into stage `stage`
        const int m0 = (first + b) * ROWS;
        if (i < S::ROW_DMA) {
            const int instruction = S::ROW_DMA * wave + i, at_slot = instruction * 64 + lane;
            const int row = at_slot / S::CHUNKS, slot = at_slot % S::CHUNKS;
            const uint32_t source = (uint32_t)min(m0 + row, M - 1) * ROW_BYTES + ((slot ^ (row & 15)) * 16);
            buffer_dma16(x_rsrc, (LDS_SPACE void*)(ring + stage * S::BLOCK_BYTES + instruction * 1024), source, 0);
        } else {   // lane l brings row l % 32's scale (no branch around the instruction)
            buffer_dma4(scale_rsrc, (LDS_SPACE void*)(ring + S::SCALES_AT + stage * S::SCALE_BYTES + 256 * wave),
                        (uint32_t)min(m0 + in_row, M - 1) * 4, 0);
        }
    };
#pragma unroll
    for (int b = 0; b < STAGES - 1; b++)
#pragma unroll
        for (int i = 0; i < S::DMA_OPS; i++) issue_one(min(b, count - 1), b, i);

    // the wavefront's column vectors: lane j takes column j of its 64 weight scales (gated: the gate's 32, then up's) and
    // biases
    LDS_SPACE float* vectors = (LDS_SPACE float*)(lds + S::VECTORS_AT) + wave * 128;
    {
        const int column = NB == 2 ? min(n_wave + lane % COLUMNS, N - 1) : min(n_wave + lane, N - 1);
        if constexpr (S::INT8) vectors[lane] = e.w_scale[NB == 2 && lane >= COLUMNS ? N + column : column];
        if constexpr (S::BIAS) vectors[64 + lane] = (float)e.bias[column];
    }

    // a lane's operand read at step t: row l % 32, slot (2 t + l / 32) ^ (l % 16), i.e. this base with 32 t xored in
    const uint32_t operand = in_row * ROW_BYTES + 16 * (half ^ (lane & 15));
    auto operand_at = [&](int t) {   // (a row of a power of two of bytes: one xor; else a chunk's low four bits by xor, the rest added)
        if constexpr ((ROW_BYTES & (ROW_BYTES - 1)) == 0) return operand ^ (32 * t);
        else return (operand ^ (32 * t & 255)) + (32 * t & ~255);
    };
    const size_t row_bytes = (size_t)N * sizeof(OutT);
    // a lane's first 16-byte store (and residual load): row l % 32 of the block, columns n_wave + 8 (l / 32) ..; columns
    // past N store nothing (and load zeros)
    const uint32_t out_lane = (uint32_t)in_row * (uint32_t)row_bytes + (uint32_t)((n_wave + 8 * half) * sizeof(OutT));
    auto at = [&](int f, int p) {   // the store of 4-column groups 2 p and 2 p + 1 of output fragment f
        return n_wave + 32 * f + 16 * p + 8 * half < N ? out_lane + (uint32_t)((32 * f + 16 * p) * sizeof(OutT)) : 0x80000000u;
    };
    // block m0's rows of out (or of the residual), in scalar registers (a resource in vector registers takes a loop over
    // lanes an access)
    auto rows_of = [&](const void* base, int m0) {
        const uint32_t bytes = __builtin_amdgcn_readfirstlane((uint32_t)min(ROWS, M - m0) * (uint32_t)row_bytes);
        return buffer_resource((const int8_t*)base + (size_t)m0 * row_bytes, bytes);
    };

    // Block b's sums go to set b % 2, and its epilogue runs in the next block's turn, between that block's MFMAs: the
    // MFMAs of one block and the VALU of the one before it are independent, so one wavefront keeps both busy.
    typename MMA::Sums sums[2][FRAGMENTS];
    float row_scale[2] = {1.0f, 1.0f};
    // A 4-column group's column vectors (weight scales, up's, biases), read ahead of its outputs into one of two slots
    struct Columns { v4f scale, up, bias; };
    auto columns = [&](int g) {   // group g: fragment g / 4, columns 8 (g % 4) + 4 (l / 32) ..
        const int col = 32 * (g / 4) + 8 * (g % 4) + 4 * half;
        Columns c{};
        if constexpr (S::INT8) c.scale = *(const LDS_SPACE v4f*)(vectors + col);
        if constexpr (NB == 2) c.up = *(const LDS_SPACE v4f*)(vectors + COLUMNS + col);
        if constexpr (S::BIAS) c.bias = *(const LDS_SPACE v4f*)(vectors + 64 + col);
        return c;
    };
    // Output k of set D (fragment k / 16, register k % 16): lane l holds row l % 32 and, in register 4 q + r, column
    // 8 q + 4 (l / 32) + r of its fragment. Gated: up's sum is in the other fragment, or in the second half of the only one.
    auto output = [&](auto set, int k, const Columns& c) {
        constexpr int D = decltype(set)::value;
        const int f = k / 16, q = k % 16 / 4, r = k % 4;
        constexpr int UP_FRAGMENT = FRAGMENTS - 1, UP_REGISTER = FRAGMENTS == 2 ? 0 : 8;
        float value;
        if constexpr (NB == 2 && !S::BIAS) {   // silu_times' constants on the row scale
            value = silu_times((MMA::value(sums[D][0], 4 * q + r) * (row_scale[D] * NEG_LOG2E)) * c.scale[r],
                               (MMA::value(sums[D][UP_FRAGMENT], UP_REGISTER + 4 * q + r) * (row_scale[D] * NEG_LN2)) * c.up[r]);
        } else {
            if constexpr (S::INT8) {
                value = (MMA::value(sums[D][f], 4 * q + r) * row_scale[D]) * c.scale[r];
            } else {
                value = MMA::value(sums[D][f], 4 * q + r);
            }
            if constexpr (S::BIAS) value = value + c.bias[r];
            if constexpr (NB == 2) {
                const float up = (MMA::value(sums[D][UP_FRAGMENT], UP_REGISTER + 4 * q + r) * row_scale[D]) * c.up[r];
                value = silu_times(value * NEG_LOG2E, up * NEG_LN2);
            }
        }
        asm volatile("" : "+v"(value));   // the f32 value is what rounds
        return value;
    };
    // the residual's and the input's 8 columns of each of the lane's stores
    struct Added { uint4 residual, original; };
    constexpr int ADDED = S::RESIDUAL ? S::STORE_OPS : 1;
    auto load_added = [&](int m0, Added (&added)[ADDED]) {
        if constexpr (S::RESIDUAL) {
            const BufferResource residual_rsrc = rows_of(e.residual, m0);
#pragma unroll
            for (int j = 0; j < S::STORE_OPS; j++) added[j].residual = buffer_load16(residual_rsrc, at(j / 2, j % 2), 0);
        }
        if constexpr (S::MIX) {
            const BufferResource original_rsrc = rows_of(e.original, m0);
#pragma unroll
            for (int j = 0; j < S::STORE_OPS; j++) added[j].original = buffer_load16(original_rsrc, at(j / 2, j % 2), 0);
        }
    };
    const float mix_residual = S::MIX ? (float)e.residual_scale[0] : 0.0f, mix_input = S::MIX ? (float)e.input_scale[0] : 0.0f;
    // the outputs of groups q = 2 p, 2 p + 1 of fragment f stored (plus the residual, its 8 columns in the lane's 16 bytes, and
    // the next block's input mix)
    auto store = [&](const BufferResource& out_rsrc, int f, int p, const float (&even)[4], const float (&odd)[4], const Added& more) {
        if constexpr (S::RESIDUAL) {
            float eight[8];
            eight_values(even, odd, eight);
            const v8h added = __builtin_bit_cast(v8h, more.residual), original = __builtin_bit_cast(v8h, more.original);
            float lower[4], upper[4];
#pragma unroll
            for (int j = 0; j < 8; j++) {
                float value = eight[j] + (float)added[j];
                if constexpr (S::MIX) value = (to_float(from_float<OutT>(value)) * mix_residual) + ((float)original[j] * mix_input);
                (j < 4 ? lower : upper)[j % 4] = value;
            }
            const uint2 lo = pack_four<OutT>(lower), hi = pack_four<OutT>(upper);
            buffer_store16(out_rsrc, v4u{lo.x, lo.y, hi.x, hi.y}, at(f, p), 0);
        } else {
            buffer_store16(out_rsrc, eight_columns(pack_four<OutT>(even), pack_four<OutT>(odd)), at(f, p), 0);
        }
    };
    // block b landed (the wait covers this wavefront's DMA; the barrier every wavefront's), and every wavefront is done
    // with the stage that block b + STAGES - 1's DMA, issued in b's turn, overwrites
    auto begin = [&](int b) {
        if (b >= STAGES) {
            stage_barrier<S::after(STAGES)>();
        } else {
            static_for<0, STAGES>([&](auto k) {
                if (b == decltype(k)::value) stage_barrier<S::after(decltype(k)::value)>();
            });
        }
    };
    // One block's turn: its MFMAs into set P and, spread between them, the epilogue of the block before it from the other
    // set (when there is one), its PER_LANE outputs a lane in order, each pair of 4-column groups stored when done, each
    // group's column vectors read ahead into a slot of their own (read just before use, a vector's wait would also wait
    // for the operand reads ahead of it). The operand of step t + LOOKAHEAD is read at step t, and the DMA of block
    // b + STAGES - 1 goes out one instruction every DMA_EVERY steps.
    constexpr int LOOKAHEAD = 2, DMA_EVERY = 3, PER_LANE = S::PER_LANE, SPAN = 4 * STEPS / PER_LANE;   // a 4-column group's steps
    static_assert(DMA_EVERY * (S::DMA_OPS - 1) < STEPS, "the turn's DMA fits its steps");
    auto turn = [&](auto set, int b, auto finishing) {
        constexpr int P = decltype(set)::value, D = 1 - P;
        constexpr bool FINISH = decltype(finishing)::value;
        const int stage = b % STAGES;
        const int next = min(b + STAGES - 1, count - 1), next_stage = (b + STAGES - 1) % STAGES;
        const LDS_SPACE int8_t* block = ring + stage * S::BLOCK_BYTES;
        const int m0 = (first + b - 1) * ROWS;   // the block before, whose epilogue this turn runs
        const BufferResource out_rsrc = rows_of(out, FINISH ? m0 : 0);
        Added added[ADDED] = {};
        if constexpr (FINISH) load_added(m0, added);
        Columns slot[2];
        if constexpr (FINISH) slot[0] = columns(0);
        Operand a[STEPS];
#pragma unroll
        for (int t = 0; t < LOOKAHEAD; t++) a[t] = *(const LDS_SPACE Operand*)(block + operand_at(t));
        float even[4], odd[4];
#pragma unroll
        for (int t = 0; t < STEPS; t++) {
            if (t % DMA_EVERY == 0 && t / DMA_EVERY < S::DMA_OPS) issue_one(next, next_stage, t / DMA_EVERY);
            if constexpr (FINISH) {
                // group g's columns, half a group's steps before its first output (its slot's previous group then done)
#pragma unroll
                for (int g = 1; g < PER_LANE / 4; g++)
                    if (t == g * SPAN - SPAN / 2) slot[g % 2] = columns(g);
            }
            if (t + LOOKAHEAD < STEPS) a[t + LOOKAHEAD] = *(const LDS_SPACE Operand*)(block + operand_at(t + LOOKAHEAD));
#pragma unroll
            for (int f = 0; f < FRAGMENTS; f++)
                sums[P][f] = MMA::step(weights[f][t], a[t], t == 0 ? typename MMA::Sums{} : sums[P][f]);
            if constexpr (FINISH) {
                // outputs t PER_LANE / STEPS .. (t + 1) PER_LANE / STEPS - 1 of the block before
#pragma unroll
                for (int k = t * PER_LANE / STEPS; k < (t + 1) * PER_LANE / STEPS; k++) {
                    const int q = k % 16 / 4, r = k % 4;
                    (q % 2 ? odd : even)[r] = output(std::integral_constant<int, D>{}, k, slot[k / 4 % 2]);
                    if (q % 2 && r == 3) store(out_rsrc, k / 16, q / 2, even, odd, added[S::RESIDUAL ? k / 16 * 2 + q / 2 : 0]);
                }
            }
        }
        if constexpr (S::INT8) row_scale[P] = ((const LDS_SPACE float*)(ring + S::SCALES_AT + stage * S::SCALE_BYTES + 256 * wave))[in_row];
    };
    // the last block's epilogue, after the loop, alone
    auto finish = [&](auto set, int b) {
        constexpr int P = decltype(set)::value;
        const int m0 = (first + b) * ROWS;
        const BufferResource out_rsrc = rows_of(out, m0);
        Added added[ADDED] = {};
        load_added(m0, added);
        float even[4], odd[4];
#pragma unroll
        for (int k = 0; k < PER_LANE; k++) {
            const int q = k % 16 / 4, r = k % 4;
            (q % 2 ? odd : even)[r] = output(std::integral_constant<int, P>{}, k, columns(k / 4));
            if (q % 2 && r == 3) store(out_rsrc, k / 16, q / 2, even, odd, added[S::RESIDUAL ? k / 16 * 2 + q / 2 : 0]);
        }
    };
    if (idle) {
        // its share of each block's DMA and as many stores (dropped) as a working wavefront's, so that its waits count
        // the same operations, and the barriers
        for (int b = 0; b < count; b++) {
            begin(b);
#pragma unroll
            for (int i = 0; i < S::DMA_OPS; i++) issue_one(min(b + STAGES - 1, count - 1), (b + STAGES - 1) % STAGES, i);
            if (b >= 1) {
                const BufferResource out_rsrc = rows_of(out, (first + b - 1) * ROWS);
#pragma unroll
                for (int j = 0; j < S::STORE_OPS; j++) buffer_store16(out_rsrc, v4u{}, 0x80000000u, 0);
            }
        }
        __builtin_amdgcn_s_waitcnt(vmcnt_only(0));
        return;
    }
    constexpr auto EVEN = std::integral_constant<int, 0>{};
    constexpr auto ODD = std::integral_constant<int, 1>{};
    begin(0);
    turn(EVEN, 0, std::false_type{});
    int b = 1;
    for (; b + 1 < count; b += 2) {
        begin(b);
        turn(ODD, b, std::true_type{});
        begin(b + 1);
        turn(EVEN, b + 1, std::true_type{});
    }
    if (b < count) {
        begin(b);
        turn(ODD, b, std::true_type{});
        finish(ODD, b);
    } else {
        finish(EVEN, b - 1);
    }
    __builtin_amdgcn_s_waitcnt(vmcnt_only(0));   // the tail's repeated DMA lands before the LDS is reused
}

// How an XCD's workgroups are shared out: `slices` streams of row blocks for every column group but the last, which has
// `last_slices`. A last group with columns for only some wavefronts (they idle, but not beside a residual) gets fewer
// workgroups and longer streams: its turns cost about (WAVES + working wavefronts) / (2 WAVES) of a full group's. Of all such
// shares the one whose longest stream is the shortest: rounding the full groups' share up instead can leave the last group
// almost none (256 to 2 x 1,408: six and two of 32, where five and seven take 0.200 of the rows' time and not 0.375). Graphs of
// launches on an MI355X, us, rounded up and so: 70,000 rows of 256 to 2 x 1,408 120.7 and 83.0, of 512 to 2 x 1,408 145.0 and
// 106.8; 35,000 of 1,024 to 1,600 80.2 and 64.4; 69,930 of 768 to 1,152 73.4 and 69.3; 512 to 1,600 (nine and five) is shared alike.
// `busy` is the part of the XCD's workgroups' time that the groups' work takes.
struct Plan { int groups, slices, last_slices; double busy; };
template <typename S> Plan plan(int N, int per_xcd) {
    Plan p{(N + S::GROUP - 1) / S::GROUP};
    p.slices = p.last_slices = per_xcd / p.groups;
    const int working = (N - (p.groups - 1) * S::GROUP + S::COLUMNS - 1) / S::COLUMNS;   // the last group's working wavefronts
    const double cost = (WAVES + working) / (2.0 * WAVES), last_cost = S::RESIDUAL ? 1.0 : cost;
    auto longest = [&](int slices, int last_slices) { return std::max(p.groups > 1 ? 1.0 / slices : 0.0, last_cost / last_slices); };
    if (p.groups > 1 && last_cost < 1.0) {
        auto last_of = [&](int slices) { return per_xcd - (p.groups - 1) * slices; };
        for (int slices = p.slices + 1; slices <= (per_xcd - 1) / (p.groups - 1); slices++)
            if (longest(slices, last_of(slices)) < longest(p.slices, last_of(p.slices))) p.slices = slices;
        p.last_slices = last_of(p.slices);
    }
    p.busy = (p.groups - 1 + cost) / per_xcd / longest(p.slices, p.last_slices);
    return p;
}

// The launch: a workgroup a compute unit, each XCD's workgroups taking streams of row blocks for every column group.
template <typename In, int NB, typename OutT, int EPI, int DEPTH_ = DEPTH>
int launch(const void* x, const void* w, void* out, const Epilogue& e, int M, int N, hipStream_t stream) {
    typedef Shape<In, NB, EPI, DEPTH_> S;
    auto kernel = resident_kernel<In, NB, OutT, EPI, DEPTH_>;
    static const hipError_t allowed = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, S::LDS_BYTES);
    if (allowed != hipSuccess) return (int)allowed;
    int device = 0, units = 0;
    if (hipError_t status = hipGetDevice(&device); status != hipSuccess) return (int)status;
    if (hipError_t status = hipDeviceGetAttribute(&units, hipDeviceAttributeMultiprocessorCount, device); status != hipSuccess) return (int)status;
    const int workgroups = units - units % XCDS;
    const int per_xcd = workgroups / XCDS, groups = (N + S::GROUP - 1) / S::GROUP;
    if (groups > per_xcd)
        return chess_fail(CHESS_UNSUPPORTED, "tile 15 takes at most %d column groups of %d on this device, not %d", per_xcd, S::GROUP, groups);
    const Plan p = plan<S>(N, per_xcd);
    hipLaunchKernelGGL(kernel, dim3(workgroups), dim3(64 * WAVES), S::LDS_BYTES, stream, (const In*)x, (const In*)w, (OutT*)out, e, M, N, p.groups,
                       p.slices, p.last_slices);
    return launch_status();
}

// What tile 15 takes: depth 512, N a multiple of 8 (a lane stores 8 columns, all of them or none past N), outputs under
// 2 GiB (32-bit store offsets); int8 in, fp16 or bf16 out, with or without the bias (gated or not); fp16 in and out, not
// gated, with the bias and the residual (the attention's output projection) or the bias alone (the fp16 block's
// projection).
template <typename In, int NB, typename OutT>
int dispatch(const void* x, const void* w, void* out, const Epilogue& e, int M, int N, int K, hipStream_t stream) {
    constexpr bool INT8 = std::is_same<In, int8_t>::value;
    if (K != DEPTH) return chess_fail(CHESS_UNSUPPORTED, "tile 15 holds weights of depth %d in registers, not %d", DEPTH, K);
    if (N % 8 != 0) return chess_fail(CHESS_UNSUPPORTED, "tile 15 takes N a multiple of 8, not %d", N);
    if ((uint64_t)M * N * sizeof(OutT) >= (1ull << 31)) return chess_fail(CHESS_UNSUPPORTED, "tile 15 writes outputs under 2 GiB");
    if constexpr (!std::is_same<OutT, half_t>::value && !(INT8 && std::is_same<OutT, bf16_t>::value)) {
        return chess_fail(CHESS_UNSUPPORTED, "tile 15 writes fp16 (or, from int8 sums, bf16)");
    } else if constexpr (INT8) {
        if (e.flags & ~EPI_BIAS) return chess_fail(CHESS_UNSUPPORTED, "tile 15 adds no residual or input mix to int8 sums");
        return e.flags & EPI_BIAS ? launch<In, NB, OutT, EPI_BIAS>(x, w, out, e, M, N, stream) : launch<In, NB, OutT, 0>(x, w, out, e, M, N, stream);
    } else {
        if (NB != 1 || (e.flags != (EPI_BIAS | EPI_RESIDUAL) && e.flags != EPI_BIAS))
            return chess_fail(CHESS_UNSUPPORTED, "tile 15 takes fp16 sums with the bias (and the residual) only, not gated");
        return e.flags & EPI_RESIDUAL ? launch<In, 1, OutT, EPI_BIAS | EPI_RESIDUAL>(x, w, out, e, M, N, stream)
                                      : launch<In, 1, OutT, EPI_BIAS>(x, w, out, e, M, N, stream);
    }
}

// What tile 0 gives to this kernel: tile 15's launches and, with the same limits, the other depths of the networks' widths.
// f(depth, epilogue), as constants, launches one; a launch that no instantiation takes is false.
template <typename In, int NB, typename OutT, typename F> bool taken(int flags, int K, F&& f) {
    constexpr bool INT8 = std::is_same<In, int8_t>::value;
    auto with = [&](auto depth, auto epilogue) {
        if (K != decltype(depth)::value || flags != decltype(epilogue)::value) return false;
        f(depth, epilogue);
        return true;
    };
    constexpr std::integral_constant<int, 0> PLAIN{};
    constexpr std::integral_constant<int, EPI_BIAS> BIAS{};
    constexpr std::integral_constant<int, EPI_RESIDUAL> RESIDUAL{};
    constexpr std::integral_constant<int, EPI_RESIDUAL | EPI_MIX> MIX{};
    constexpr std::integral_constant<int, EPI_BIAS | EPI_RESIDUAL> BIAS_RESIDUAL{};
    constexpr std::integral_constant<int, 256> D256{};
    constexpr std::integral_constant<int, 512> D512{};
    constexpr std::integral_constant<int, 768> D768{};
    constexpr std::integral_constant<int, 1024> D1024{};
    if constexpr (sizeof(OutT) != 2 || (!INT8 && NB == 2)) {
        return false;
    } else if constexpr (!INT8) {
        return with(D256, BIAS) || with(D256, BIAS_RESIDUAL) || with(D512, BIAS) || with(D512, BIAS_RESIDUAL);
    } else if constexpr (NB == 2) {
        return with(D256, PLAIN) || with(D512, PLAIN) || with(D768, PLAIN);
    } else {
        return with(D256, BIAS) || with(D512, BIAS) || with(D512, PLAIN) || with(D768, BIAS) || with(D1024, BIAS) || with(D1024, RESIDUAL)
            || with(D1024, MIX);
    }
}

// The least row blocks a workgroup's stream has to hold for the launch to pay for its weights' load and its ends. Timed on an
// MI355X as graphs of launches (us, this kernel and the best other tile): int8, 768 to 1,152 columns, 17,920 rows (11 blocks)
// 26.0 and 26.8, 35,000 40.1 and 44.4, 69,930 69.3 and 87.3; 768 to 2 x 992 gated, 7,000 (7) 19.8 and 17.2, 17,920 (17) 35.5
// and 38.3, 69,930 113 and 141; 256 to 2 x 1,024 gated, 17,920 (9) 21.5 and 20.0, 69,930 (34) 56.4 and 64.2; 256 to 832,
// 17,920 (4) 14.9 and 11.7, 69,930 (17) 31.6 and 35.4; 1,024 to 768 with the residual and the mix, 17,920 (7) 29.4 and 32.2,
// 35,000 (13) 46.8 and 54.4; 1,024 to 256 so, 35,000 (4) 25.7 and 25.0, 69,930 (9) 36.5 and 41.1; fp16, 256 to 256 with bias
// and residual, 69,930 (9) 22.4 and 24.5. (Left out, as no faster: the residual at depths 512 and 768.) A launch of one
// output a weight row that writes more than the last-level cache holds is bound by its writes, and whole lines from LDS go
// faster than these 16-byte stores (512 to 2,048 at 65,536 rows, 268 MB: 121 us and 109 on tile 4); gated, 293 MB still take
// 163 and 240. For output rows of whole KB, from short inputs and without a residual to read, that is so from 230 MiB on
// (this kernel and tile 4: 512 to 1,024, 210 MiB 90 and 92, 230 MiB 116 and 100; 512 to 1,536, 220 MiB 95 and 95, 240 MiB 115
// and 100; 512 to 2,048, 230 MiB 99 and 100, 255 MiB 120 and 110; 256 to 2,048, 240 MiB 73 and 76, 250 MiB 84 and 77), for
// others not up to 256 MiB (512 to 1,600, 230 MiB 80 and 103, 255 MiB 106 and 116; 768 to 1,152, 255 MiB 139 and 150; 1,024
// to 1,024 with the residual 163 and 239; fp16, 512 to 512 144 and 195). Below LARGE_ROWS, where the other tile is 11 and not
// the slower 4, a plan whose workgroups are too often out of work does not pay: 768 to 2 x 2,176 (17 groups for 32
// workgroups, busy 0.53) at 12,000 rows 68.5 and 59.9, 256 to 2 x 4,352 65.9 and 49.1 (at 35,000 177 and 174, at 70,000 345
// and 333; 512 to 2 x 4,352 208 and 241), 512 to 2 x 2,816 (11 groups, 0.69) 49.8 and 52.5; with the shorter MFMA chains of
// depth 256 the line lies higher, 256 to 2 x 2,816 39.6 and 34.1. Two working wavefronts of a sole group's eight do not
// either: 256 to 72 at 110,000 rows 18.4 and 14.1, 512 to 72 19.8 and 19.0 (three, 768 to 72: 20.9 and 23.4). Beside a
// residual a part-filled group costs a full one, which near the line is no loss yet: 1,024 to 264 and 384 at 25,000 rows 22.9
// and 24.1, where tile 13 takes 23.9 and 24.3; with the mix 27.0 and 29.2, and 26.9 and 27.9.
constexpr int STREAM_BLOCKS = 10, DEEP_STREAM_BLOCKS = 6, F16_STREAM_BLOCKS = 8, LARGE_ROWS = 32768;
constexpr double LEAST_BUSY = 0.6, LEAST_BUSY_256 = 0.7;
constexpr uint64_t MOST_WRITTEN = 256ull << 20, MOST_WRITTEN_WHOLE_KB = 230ull << 20;

template <typename In, int NB, typename OutT> bool takes(int flags, int M, int N, int K) {
    const uint64_t row_bytes = (uint64_t)N * sizeof(OutT);
    const bool short_inputs = (size_t)K * sizeof(In) <= 512 && !(flags & EPI_RESIDUAL);
    const uint64_t most = NB == 2 ? 1ull << 31 : short_inputs && row_bytes % 1024 == 0 ? MOST_WRITTEN_WHOLE_KB : MOST_WRITTEN;
    if (N % 8 != 0 || M * row_bytes >= most) return false;
    int device = 0, units = 0;
    if (hipGetDevice(&device) != hipSuccess || hipDeviceGetAttribute(&units, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess) return false;
    bool worth = false;
    const bool known = taken<In, NB, OutT>(flags, K, [&](auto depth, auto epilogue) {
        typedef Shape<In, NB, decltype(epilogue)::value, decltype(depth)::value> S;
        const int per_xcd = units / XCDS, least = !S::INT8 ? F16_STREAM_BLOCKS : S::RESIDUAL ? DEEP_STREAM_BLOCKS : STREAM_BLOCKS;
        if ((N + S::GROUP - 1) / S::GROUP > per_xcd || N <= 2 * S::COLUMNS) return;
        const Plan p = plan<S>(N, per_xcd);
        worth = (M >= LARGE_ROWS || p.busy >= (S::ROW_BYTES == 256 ? LEAST_BUSY_256 : LEAST_BUSY))
             && (long)(M / ROWS) * p.groups >= (long)least * units;
    });
    return known && worth;
}
template <typename In, int NB, typename OutT>
int launch_taken(const void* x, const void* w, void* out, const Epilogue& e, int M, int N, int K, hipStream_t stream) {
    int status = CHESS_OK;
    taken<In, NB, OutT>(e.flags, K, [&](auto depth, auto epilogue) {
        status = launch<In, NB, OutT, decltype(epilogue)::value, decltype(depth)::value>(x, w, out, e, M, N, stream);
    });
    return status;
}

}  // namespace resident
