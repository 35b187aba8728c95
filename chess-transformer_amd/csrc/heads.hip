// The policy head's move logits of B positions, from the final norm's rows.
// Computes what model/fused_blocks.py:863-872 (the heads without fused ends) computes after its `a` matmul:
//   narrow[t][c] = x[t] . W[c] + w_bias[c]                          c < NN: s, the promotion logits, board_down's
//   logits[i][j] = (a[i] + a_bias) . x[j] + narrow[i][0]             i, j < 64, the squares
//   out[m] = logits[from m][to m] (+ narrow[to'][column'] for a promotion move)
// and writes board_down's inputs narrow[t][down_first..NN) for the value head. x is the stream [B, T, D] fp16 (exact
// in f32), a [B, T, D] f32 (rows 0..63 read), a_bias [D], W [NN, D] and w_bias [NN] f32. The reference takes these
// products in f32 (torch's F.linear and bmm); here they are f32 MFMAs (v_mfma_f32_32x32x2_f32: exact products,
// f32 sums), so the results agree with it to f32 rounding, not to the bit.
//
// Two launches. The first takes one 32 x 32 block of products a workgroup: the 4 quadrants of the logits and the 3 blocks of
// 32 token rows of the narrow products (all NN <= 32 columns), 7 workgroups a position, so that a batch of few positions
// still spreads over the chip. Its wavefronts split D in up to 4 parts, whose partial blocks meet in LDS and are added in
// part order. A step covers 8 of D: lane l (row l % 32, half h = l / 32) loads 4 consecutive values k0 + 4h .. + 3 of its
// row of each operand and feeds them to 4 MFMAs, value m to MFMA m, so that in MFMA m both operands' k-halves stand for
// k0 + m and k0 + 4 + m; four steps' loads go out together. The blocks go to a workspace of the caller's, 7,168 floats a
// position (the 64 x 64 logits, then 96 x 32 narrow products). The second launch, a workgroup a position, adds each
// square's narrow column 0, gathers the 1,968 moves with their promotion logits, and writes board_down's inputs.
#include "chess_common.h"

#include <mutex>

namespace {

constexpr int SQUARES = 64;
constexpr int MAX_NARROW = 32;
constexpr int MAX_TOKENS = 96;                 // three blocks of 32 token rows
constexpr int THREADS = 256;

typedef float v16f __attribute__((ext_vector_type(16)));

DEVICE v16f mfma_f32(float a, float b, v16f c) { return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0); }

// nn.GELU's exact form, 0.5 v (1 + erf(v / sqrt 2)), with the device library's erf
DEVICE float gelu(float v) { return 0.5f * v * (1.0f + erff(v * 0.70710678118654752f)); }

// the 32 x 32 block sum_k A[row0 + i][k] * X[col0 + j][k] over k < length, rows stride elements apart: A's rows f32 (a_bias
// added when BIAS), X's fp16; rows past a_rows and columns past x_rows read the last one (never kept). Lane l holds, in
// register 4q + r, the sum for A row 8q + 4(l / 32) + r and X row l % 32. length is a multiple of 64: four steps a turn,
// their loads (the bias's too) issued before their MFMAs, so that a turn's loads are in flight together.
template <bool BIAS>
DEVICE v16f block_products(const float* A, int a_rows, const float* a_bias, const half_t* X, int x_rows, int length, int stride, int lane) {
    constexpr int TURN = 4;   // steps of 8 a turn
    const int r32 = lane & 31, h = lane >> 5;
    const float* a_row = A + (size_t)min(r32, a_rows - 1) * stride + 4 * h;
    const half_t* x_row = X + (size_t)min(r32, x_rows - 1) * stride + 4 * h;
    v16f acc = {};
    for (int turn = 0; turn < length; turn += 8 * TURN) {
        float4 av[TURN], bias[TURN];
        v4h xv[TURN];
#pragma unroll
        for (int s = 0; s < TURN; s++) {
            av[s] = *reinterpret_cast<const float4*>(a_row + turn + 8 * s);
            xv[s] = *reinterpret_cast<const v4h*>(x_row + turn + 8 * s);
            if constexpr (BIAS) bias[s] = *reinterpret_cast<const float4*>(a_bias + turn + 8 * s + 4 * h);
        }
#pragma unroll
        for (int s = 0; s < TURN; s++) {
            float4 a4 = av[s];
            if constexpr (BIAS) a4 = float4{a4.x + bias[s].x, a4.y + bias[s].y, a4.z + bias[s].z, a4.w + bias[s].w};
            acc = mfma_f32(a4.x, (float)xv[s][0], acc);
            acc = mfma_f32(a4.y, (float)xv[s][1], acc);
            acc = mfma_f32(a4.z, (float)xv[s][2], acc);
            acc = mfma_f32(a4.w, (float)xv[s][3], acc);
        }
    }
    return acc;
}

constexpr int BLOCKS_A_POSITION = 4 + MAX_TOKENS / 32;
constexpr int WORKSPACE_FLOATS = SQUARES * SQUARES + MAX_TOKENS * MAX_NARROW;   // a position's

__global__ __launch_bounds__(THREADS) void head_blocks_kernel(
    const half_t* __restrict__ x, const float* __restrict__ a, const float* __restrict__ a_bias, const float* __restrict__ w,
    const float* __restrict__ w_bias, float* __restrict__ workspace, int B, int T, int D, int NN, int parts)
{
    __shared__ float partial[4][32 * 32];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // The workgroups go to the 8 XCDs in turn, each with its own L2: a position's 7 blocks run on one XCD (positions
    // x, x + 8, ... on XCD x), so that its rows of a and x come from that L2 after the first read.
    constexpr int XCDS = 8;
    const int xcd = blockIdx.x % XCDS, on_xcd = blockIdx.x / XCDS;
    const int block = on_xcd % BLOCKS_A_POSITION;
    const size_t b = (size_t)(on_xcd / BLOCKS_A_POSITION) * XCDS + xcd;
    if (b >= (size_t)B) return;   // the whole workgroup: the launch rounds the positions up to a multiple of 8
    const half_t* xb = x + b * T * D;
    const int r32 = lane & 31, h = lane >> 5;
    const int t0 = (block - 4) * 32;
    if (block >= 4 && t0 >= T) return;   // the whole workgroup: a narrow block past the tokens
    const int part = D / parts, k0 = wave * part;
    if (wave < parts) {
        // quadrant: rows i0.. of a (the from side), columns j0.. of x (the to side); narrow: W's rows (columns c) and x's
        // token rows t0..
        const int i0 = (block >> 1) * 32, j0 = (block & 1) * 32;
        const v16f products = block < 4
            ? block_products<true>(a + (b * T + i0) * D + k0, 32, a_bias + k0, xb + (size_t)j0 * D + k0, 32, part, D, lane)
            : block_products<false>(w + k0, NN, nullptr, xb + (size_t)t0 * D + k0, T - t0, part, D, lane);
#pragma unroll
        for (int q = 0; q < 4; q++)
#pragma unroll
            for (int r = 0; r < 4; r++) partial[wave][(8 * q + 4 * h + r) * 32 + r32] = products[4 * q + r];
    }
    __syncthreads();
    float* out = workspace + b * WORKSPACE_FLOATS;
#pragma unroll
    for (int e = tid; e < 32 * 32; e += THREADS) {
        float sum = partial[0][e];
        for (int p = 1; p < parts; p++) sum = sum + partial[p][e];
        const int row = e / 32, column = e % 32;   // row of the first operand, column of the second
        if (block < 4) {
            out[((block >> 1) * 32 + row) * SQUARES + (block & 1) * 32 + column] = sum;
        } else if (row < NN && t0 + column < T) {
            out[SQUARES * SQUARES + (t0 + column) * MAX_NARROW + row] = sum + w_bias[row];
        }
    }
}

// The moves and the values a thread takes in one turn, each kind of load issued for all of them before any is used: the chain
// from a move's cells to its products is two trips long, and a loop over single moves paid it for each left over from its
// unrolling. With the bias's loads above, on an MI355X at 512 columns: both launches at one position 14.4 -> 11.4 us, at 64
// 19.5 -> 16.1, at 300 49.9 -> 46.8.
constexpr int GATHER_TURN = 8, DOWN_TURN = 5;

__global__ __launch_bounds__(THREADS) void head_gather_kernel(
    const float* __restrict__ workspace, const int* __restrict__ cells, const int* __restrict__ promotions, float* __restrict__ out,
    float* __restrict__ down, int T, int NN, int down_first, int moves, int out_stride, int activate)
{
    const int tid = threadIdx.x;
    const size_t b = blockIdx.x;
    const float* logits = workspace + b * WORKSPACE_FLOATS;
    const float* narrow = logits + SQUARES * SQUARES;
    // the moves: cells[m] = from * 64 + to; promotions[m] = to' * 32 + column of its promotion logit, or -1 (the places
    // are masked into the blocks, so that no table entry reads outside them); logits = the quadrant + s[from] (the from
    // square's narrow column 0)
    float* out_b = out + b * out_stride;
    for (int m0 = tid; m0 < moves; m0 += GATHER_TURN * THREADS) {
        int cell[GATHER_TURN], promotion[GATHER_TURN];
        float value[GATHER_TURN], s[GATHER_TURN], promoted[GATHER_TURN];
#pragma unroll
        for (int i = 0; i < GATHER_TURN; i++) {   // (a move past the last reads the last one's and is not written)
            const int m = min(m0 + i * THREADS, moves - 1);
            cell[i] = cells[m];
            promotion[i] = promotions[m];
        }
#pragma unroll
        for (int i = 0; i < GATHER_TURN; i++) {
            const int from = (cell[i] >> 6) & 63;
            value[i] = logits[from * SQUARES + (cell[i] & 63)];
            s[i] = narrow[from * MAX_NARROW];
            promoted[i] = promotion[i] >= 0 ? narrow[((promotion[i] >> 5) & 63) * MAX_NARROW + (promotion[i] & 31)] : 0.0f;
        }
#pragma unroll
        for (int i = 0; i < GATHER_TURN; i++) {
            float sum = value[i] + s[i];
            if (promotion[i] >= 0) sum = sum + promoted[i];
            if (m0 + i * THREADS < moves) out_b[m0 + i * THREADS] = sum;
        }
    }
    const int width = NN - down_first, values = T * width;
    float* down_b = down + b * values;
    for (int e0 = tid; e0 < values; e0 += DOWN_TURN * THREADS) {
        float value[DOWN_TURN];
#pragma unroll
        for (int i = 0; i < DOWN_TURN; i++) {
            const int e = min(e0 + i * THREADS, values - 1), token = e / width;
            value[i] = narrow[token * MAX_NARROW + down_first + e - token * width];
        }
#pragma unroll
        for (int i = 0; i < DOWN_TURN; i++)
            if (e0 + i * THREADS < values) down_b[e0 + i * THREADS] = activate ? gelu(value[i]) : value[i];
    }
}

// The value head of B positions (model/model.py's eval_head after board_down_project; what the reference's fused
// heads compute in head_value_tile and head_value_kernel, model/fused_blocks.py:649-728):
//   hidden[b][u] = gelu(sum_k c[b][k] * W1[u][k] + b1[u])          c = board_down's GELU outputs, k < K = T * 16
//   logit[b][v]  = sum_u hidden[b][u] * W2[v][u] + b2[v]            v < bins
//   score[b]     = sum_v exp(logit - max) * centre[v] / sum_v exp(logit - max)
// in f32, the expected score written to the answer row's place rows[b * row_stride + score_column].
constexpr int VALUE_TILE = 16;     // positions and hidden units a workgroup of the first layer
constexpr int VALUE_CHUNK = 16;    // a token's board_down values: the K step of a wavefront
constexpr int MAX_BINS = 128;

// hidden = gelu(c @ W1^T + b1), 16 positions x 16 units a workgroup, on v_mfma_f32_16x16x4f32 (exact products, f32
// sums). Lane l supplies row l % 16 of each operand and 4 consecutive k of that row (one 16-byte load), value m to
// MFMA m, so that in MFMA m the k-group l / 16 of both operands stands for k0 + 4 (l / 16) + m. The four wavefronts
// take the K chunks in turn (wavefront w the chunks w, w + 4, ...), and their partial tiles are added in LDS as
// (w0 + w1) + (w2 + w3): a fixed order, so that no position's units depend on the batch it is in. Lane l ends with
// positions 4 (l / 16) + r (register r) of unit l % 16.
// A wavefront's chunks go in turns of HIDDEN_TURN, a turn's loads all in flight together, the last turn's missing chunks left
// out by a branch the whole wavefront takes (17 of the 70 chunks in a loop unrolled by 6 left 5 to go one by one).
constexpr int HIDDEN_TURN = 6;

__global__ __launch_bounds__(THREADS) void value_hidden_kernel(const float* __restrict__ c, const float* __restrict__ weight,
                                                               const float* __restrict__ bias, float* __restrict__ hidden, int B, int K, int H)
{
    __shared__ float partial[4][VALUE_TILE * VALUE_TILE];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int p0 = blockIdx.x * VALUE_TILE, u0 = blockIdx.y * VALUE_TILE;
    const int row = lane & 15, group = lane >> 4;
    const float* a_row = c + (size_t)min(p0 + row, B - 1) * K + 4 * group;
    const float* b_row = weight + (size_t)(u0 + row) * K + 4 * group;
    v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};
    const int chunks = K / VALUE_CHUNK;
    for (int first = wave; first < chunks; first += 4 * HIDDEN_TURN) {   // (a chunk past K reads the last one and is left out)
        float4 a4[HIDDEN_TURN], b4[HIDDEN_TURN];
#pragma unroll
        for (int i = 0; i < HIDDEN_TURN; i++) {
            const int chunk = min(first + 4 * i, chunks - 1);
            a4[i] = *reinterpret_cast<const float4*>(a_row + chunk * VALUE_CHUNK);
            b4[i] = *reinterpret_cast<const float4*>(b_row + chunk * VALUE_CHUNK);
        }
#pragma unroll
        for (int i = 0; i < HIDDEN_TURN; i++) {
            if (first + 4 * i < chunks) {
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a4[i].x, b4[i].x, acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a4[i].y, b4[i].y, acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a4[i].z, b4[i].z, acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a4[i].w, b4[i].w, acc, 0, 0, 0);
            }
        }
    }
#pragma unroll
    for (int r = 0; r < 4; r++) partial[wave][(4 * group + r) * VALUE_TILE + row] = acc[r];
    __syncthreads();
    const int position = tid / VALUE_TILE, unit = tid % VALUE_TILE;
    const float sum = (partial[0][tid] + partial[1][tid]) + (partial[2][tid] + partial[3][tid]);
    if (p0 + position < B) hidden[(size_t)(p0 + position) * H + u0 + unit] = gelu(sum + bias[u0 + unit]);
}

// The second layer, the softmax and the expected score, a workgroup a position: thread t takes bin t % 128 over half t / 128
// of the units (its W2 row from LDS, the position's hidden row uniform across each wavefront), f32 fma along
// its units in order; the halves meet in LDS as first + second, then wavefront 0 holds bins l and l + 64 in lane l and takes
// the maximum, the exponentials' sum and the centres' weighted sum as wavefront trees. A position's chain of dependent
// loads is a quarter of one wavefront's walk over all the units, and a batch of few positions still spreads over the chip.
// W2 comes through LDS, in rows of 64 units that 16 lanes read as two whole lines: read straight into the lanes that sum it, each
// 16-byte load touched 64 lines. Both launches of the value head, on an MI355X at 512 units and 81 bins: one position 14.9 ->
// 13.4 us, 300 31.2 -> 26.6, 1,024 64.3 -> 55.6.
constexpr int SCORE_PARTS = THREADS / MAX_BINS;
constexpr int SCORE_UNITS = 64;                   // units of a part staged at a time
constexpr int SCORE_ROW = SCORE_UNITS + 4;        // and a row's floats in LDS: 64 lanes' 16-byte reads fall in all banks

__global__ __launch_bounds__(THREADS) void value_score_kernel(const float* __restrict__ hidden, const float* __restrict__ weight,
                                                              const float* __restrict__ bias, const float* __restrict__ centres,
                                                              float* __restrict__ logits, float* __restrict__ rows, int B, int H, int bins,
                                                              int row_stride, int score_column)
{
    __shared__ float partial[SCORE_PARTS][MAX_BINS];
    __shared__ __align__(16) float staged[SCORE_PARTS * MAX_BINS * SCORE_ROW];
    __shared__ __align__(16) float staged_hidden[SCORE_PARTS * SCORE_UNITS];
    const int tid = threadIdx.x, lane = tid & 63;
    const int b = blockIdx.x;
    const int v = tid % MAX_BINS, part = __builtin_amdgcn_readfirstlane(tid / MAX_BINS), units = H / SCORE_PARTS;
    // staging item i of a thread: 16 bytes of a bin's row (the last bin's again past it), and of the hidden row; the next
    // units' items are in flight while these are summed
    constexpr int QUARTS = SCORE_UNITS / 4, ITEMS = SCORE_PARTS * MAX_BINS * QUARTS / THREADS;
    v4f next[ITEMS], next_hidden;
    auto load = [&](int k0) {
#pragma unroll
        for (int i = 0; i < ITEMS; i++) {
            const int item = tid + i * THREADS, to = item / QUARTS, k = min(k0 + item % QUARTS * 4, units - 4);
            next[i] = *reinterpret_cast<const v4f*>(weight + (size_t)min(to / SCORE_PARTS, bins - 1) * H + to % SCORE_PARTS * units + k);
        }
        next_hidden = *reinterpret_cast<const v4f*>(hidden + (size_t)b * H + tid / QUARTS % SCORE_PARTS * units + min(k0 + tid % QUARTS * 4, units - 4));
    };
    float sum = 0.0f;
    load(0);
    for (int k0 = 0; k0 < units; k0 += SCORE_UNITS) {
        if (k0 > 0) __syncthreads();   // the units before are summed
#pragma unroll
        for (int i = 0; i < ITEMS; i++) {
            const int item = tid + i * THREADS, to = item / QUARTS;
            *reinterpret_cast<v4f*>(staged + (to % SCORE_PARTS * MAX_BINS + to / SCORE_PARTS) * SCORE_ROW + item % QUARTS * 4) = next[i];
        }
        if (tid < SCORE_PARTS * QUARTS) reinterpret_cast<v4f*>(staged_hidden)[tid] = next_hidden;
        __syncthreads();
        load(min(k0 + SCORE_UNITS, units - 4));   // (past the last: the same place again, not used)
        const float* row = staged + (part * MAX_BINS + v) * SCORE_ROW;
        const float* h = staged_hidden + part * SCORE_UNITS;
        const int here = min(SCORE_UNITS, units - k0);
#pragma unroll 8
        for (int k = 0; k < here; k += 4) {
            const v4f x = *reinterpret_cast<const v4f*>(h + k);
            const v4f a = *reinterpret_cast<const v4f*>(row + k);
            sum = __builtin_fmaf(x[0], a[0], sum); sum = __builtin_fmaf(x[1], a[1], sum); sum = __builtin_fmaf(x[2], a[2], sum); sum = __builtin_fmaf(x[3], a[3], sum);
        }
    }
    partial[part][v] = sum;
    __syncthreads();
    if (tid >= 64) return;   // wavefronts 1-3: nothing waits for them past the barrier
    const int v0 = lane, v1 = lane + 64;
    const bool in0 = v0 < bins, in1 = v1 < bins;
    const float l0 = in0 ? (partial[0][v0] + partial[1][v0]) + bias[v0] : -__builtin_inff();
    const float l1 = in1 ? (partial[0][v1] + partial[1][v1]) + bias[v1] : -__builtin_inff();
    const float top = wave_max(fmaxf(l0, l1));
    const float e0 = in0 ? expf(l0 - top) : 0.0f, e1 = in1 ? expf(l1 - top) : 0.0f;
    const float total = wave_sum(e0 + e1);
    const float weighted = wave_sum((in0 ? e0 * centres[v0] : 0.0f) + (in1 ? e1 * centres[v1] : 0.0f));
    if (logits) {
        if (in0) logits[(size_t)b * bins + v0] = l0;
        if (in1) logits[(size_t)b * bins + v1] = l1;
    }
    if (lane == 0) rows[(size_t)b * row_stride + score_column] = weighted / total;
}

int value_head(const void* c, const void* hidden_weight, const void* hidden_bias, const void* out_weight, const void* out_bias, const void* centres,
               void* value_logits, void* rows, float* hidden, int B, int K, int H, int bins, int row_stride, int score_column, hipStream_t stream)
{
    hipLaunchKernelGGL(value_hidden_kernel, dim3((B + VALUE_TILE - 1) / VALUE_TILE, H / VALUE_TILE), dim3(THREADS), 0, stream,
                       (const float*)c, (const float*)hidden_weight, (const float*)hidden_bias, hidden, B, K, H);
    if (int status = launch_status()) return status;
    hipLaunchKernelGGL(value_score_kernel, dim3(B), dim3(THREADS), 0, stream, (const float*)hidden, (const float*)out_weight,
                       (const float*)out_bias, (const float*)centres, (float*)value_logits, (float*)rows, B, H, bins, row_stride, score_column);
    return launch_status();
}

int check_value_head(const void* c, const void* hidden_weight, const void* hidden_bias, const void* out_weight, const void* out_bias,
                     const void* centres, const void* rows, int B, int K, int H, int bins, int row_stride, int score_column)
{
    if (B < 0 || K <= 0 || K % VALUE_CHUNK != 0 || H <= 0 || H % VALUE_TILE != 0 || H % (4 * SCORE_PARTS) != 0 || bins < 1 || bins > MAX_BINS)
        return chess_fail(CHESS_UNSUPPORTED, "value_head takes inputs and units a multiple of %d and at most %d bins, not %d, %d and %d",
                          VALUE_TILE, MAX_BINS, K, H, bins);
    if (row_stride <= 0 || score_column < 0 || score_column >= row_stride)
        return chess_fail(CHESS_INVALID_SHAPE, "value_head: the score's column %d outside rows of %d", score_column, row_stride);
    if (B == 0) return CHESS_OK;   // no positions: nothing read or written, so the pointers may be null
    if (!c || !hidden_weight || !hidden_bias || !out_weight || !out_bias || !centres || !rows)
        return chess_fail(CHESS_INVALID_SHAPE, "value_head: a required pointer is null");
    if (!aligned16(c) || !aligned16(hidden_weight) || !aligned16(out_weight))
        return chess_fail(CHESS_MISALIGNED, "value_head reads its inputs and both weights 16 bytes a lane");
    return CHESS_OK;
}

}  // namespace

extern "C" int chess_move_logits(const void* x, const void* a, const void* a_bias, const void* w, const void* w_bias, const void* cells,
                                 const void* promotions, void* out, void* down, void* workspace, long long workspace_bytes, int B, int T, int D,
                                 int NN, int down_first, int moves, int out_stride, int activate, void* stream)
{
    if (B < 0 || T < SQUARES || T > MAX_TOKENS || D <= 0 || D % 64 != 0)
        return chess_fail(CHESS_UNSUPPORTED, "move_logits takes %d to %d tokens of a width that is a multiple of 64, not %d x %d", SQUARES, MAX_TOKENS,
                          T, D);
    if (NN <= 0 || NN > MAX_NARROW || down_first < 1 || down_first > NN || moves <= 0 || out_stride < moves)
        return chess_fail(CHESS_INVALID_SHAPE, "move_logits: %d narrow columns (at most %d), board_down from %d, %d moves in rows of %d", NN,
                          MAX_NARROW, down_first, moves, out_stride);
    if (B == 0) return CHESS_OK;   // no positions: nothing read or written, so the pointers may be null
    if (!x || !a || !a_bias || !w || !w_bias || !cells || !promotions || !out || !down)
        return chess_fail(CHESS_INVALID_SHAPE, "move_logits: a required pointer is null");
    if (!workspace || workspace_bytes < (long long)B * WORKSPACE_FLOATS * (long long)sizeof(float))
        return chess_fail(CHESS_INVALID_SHAPE, "move_logits' workspace holds %d floats a position, %lld bytes, not %lld", WORKSPACE_FLOATS,
                          (long long)B * WORKSPACE_FLOATS * 4LL, workspace_bytes);
    if (!aligned16(x) || !aligned16(a) || !aligned16(a_bias) || !aligned16(w))
        return chess_fail(CHESS_MISALIGNED, "move_logits reads x, a, a_bias and W 8 and 16 bytes a lane");
    // D split in the most parts (at most 4, one a wavefront) of a multiple of 64 each
    int parts = 4;
    while (D % (64 * parts) != 0) parts--;
    hipStream_t s = (hipStream_t)stream;
    hipLaunchKernelGGL(head_blocks_kernel, dim3(BLOCKS_A_POSITION * ((B + 7) / 8 * 8)), dim3(THREADS), 0, s, (const half_t*)x, (const float*)a,
                       (const float*)a_bias, (const float*)w, (const float*)w_bias, (float*)workspace, B, T, D, NN, parts);
    if (int status = launch_status()) return status;
    hipLaunchKernelGGL(head_gather_kernel, dim3(B), dim3(THREADS), 0, s, (const float*)workspace, (const int*)cells, (const int*)promotions,
                       (float*)out, (float*)down, T, NN, down_first, moves, out_stride, activate);
    return launch_status();
}

extern "C" int chess_value_head(const void* c, const void* hidden_weight, const void* hidden_bias, const void* out_weight, const void* out_bias,
                                const void* centres, void* value_logits, void* rows, void* workspace, long long workspace_bytes, int B, int K, int H,
                                int bins, int row_stride, int score_column, void* stream)
{
    if (int status = check_value_head(c, hidden_weight, hidden_bias, out_weight, out_bias, centres, rows, B, K, H, bins, row_stride, score_column))
        return status;
    if (B == 0) return CHESS_OK;
    if (!workspace || workspace_bytes < (long long)B * H * (long long)sizeof(float))
        return chess_fail(CHESS_INVALID_SHAPE, "value_head's workspace holds the hidden layer, %lld bytes, not %lld", (long long)B * H * 4LL,
                          workspace_bytes);
    if (!aligned16(workspace)) return chess_fail(CHESS_MISALIGNED, "value_head reads its workspace 16 bytes a lane");
    return value_head(c, hidden_weight, hidden_bias, out_weight, out_bias, centres, value_logits, rows, (float*)workspace, B, K, H, bins, row_stride,
                      score_column, (hipStream_t)stream);
}

// The value head without a workspace argument, for callers that cannot allocate (code under graph capture, serving
// loops that forbid allocation): the hidden layer goes through `scratch`, a file-scope device array of
// VALUE_SCRATCH_FLOATS floats (8 MiB: the hidden layer of 4,096 positions at 512 units) that each GPU holds from the
// library's load until the process ends. Host code reaches the array only through the address hipGetSymbolAddress gives
// on each device (the array's name in host code is not a device address), looked up once per device, with that
// device current, on the first call there. Every call on a GPU shares that GPU's array: calls that overlap on one GPU
// (on two streams, say) race. Every hidden value the second kernel reads was written by the first in the same call,
// so nothing needs clearing.
constexpr long long VALUE_SCRATCH_FLOATS = 1LL << 21;
static __device__ __align__(256) float scratch[VALUE_SCRATCH_FLOATS];

namespace {

constexpr int MAX_DEVICES = 64;

// the scratch array's address on the current device, looked up on the device's first call
int scratch_address(float** address) {
    static std::mutex lock;
    static float* addresses[MAX_DEVICES] = {};
    int device = 0;
    if (hipError_t error = hipGetDevice(&device); error != hipSuccess) return (int)error;
    if (device < 0 || device >= MAX_DEVICES) return chess_fail(CHESS_UNSUPPORTED, "value_head_no_alloc: device %d past the %d it keeps", device, MAX_DEVICES);
    std::lock_guard<std::mutex> guard(lock);
    if (!addresses[device]) {
        void* found = nullptr;
        if (hipError_t error = hipGetSymbolAddress(&found, HIP_SYMBOL(scratch)); error != hipSuccess) return (int)error;
        addresses[device] = (float*)found;
    }
    *address = addresses[device];
    return CHESS_OK;
}

}  // namespace

extern "C" int chess_value_head_no_alloc(const void* c, const void* hidden_weight, const void* hidden_bias, const void* out_weight,
                                         const void* out_bias, const void* centres, void* value_logits, void* rows, int B, int K, int H, int bins,
                                         int row_stride, int score_column, void* stream)
{
    if (int status = check_value_head(c, hidden_weight, hidden_bias, out_weight, out_bias, centres, rows, B, K, H, bins, row_stride, score_column))
        return status;
    if ((long long)B * H > VALUE_SCRATCH_FLOATS)
        return chess_fail(CHESS_UNSUPPORTED, "value_head_no_alloc holds at most %lld hidden values (%d positions x %d units are %lld)",
                          VALUE_SCRATCH_FLOATS, B, H, (long long)B * H);
    if (B == 0) return CHESS_OK;
    float* hidden = nullptr;
    if (int status = scratch_address(&hidden)) return status;
    return value_head(c, hidden_weight, hidden_bias, out_weight, out_bias, centres, value_logits, rows, hidden, B, K, H, bins, row_stride,
                      score_column, (hipStream_t)stream);
}
