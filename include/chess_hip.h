/* C ABI of libchess_hip.so: the gfx950 kernels of Fry's int8 network evaluation.
 *
 * Every entry point takes plain device pointers and sizes plus the hipStream_t to launch on (as
 * void*), launches asynchronously, allocates nothing and returns 0, a hipError_t (below 1000), or
 * one of the CHESS_* codes; chess_last_error() then describes the argument that was refused.
 * Unused optional pointers are NULL. fp16 data is IEEE binary16, scales are f32. A launch of no rows (or
 * no positions) checks its sizes and returns 0 at once, before any pointer is looked at: its buffers
 * may be NULL, as an empty tensor's are.
 *
 * The reference launches its kernels through ctypes (cuLaunchKernelEx on NVRTC modules,
 * model/int8_cuda.py:288-327, model/attention_cuda.py:346-391) or Triton; these entry points take
 * that place, keeping the pointer order of the reference's kernels.
 */
#ifndef CHESS_HIP_H
#define CHESS_HIP_H

#include <stddef.h>

#ifdef __cplusplus
extern "C" {
#endif

#define CHESS_INVALID_SHAPE 1001 /* a size or pointer the operator cannot take (Python: ValueError) */
#define CHESS_MISALIGNED 1002    /* an operand not 16-byte aligned (Python: ValueError) */
#define CHESS_UNSUPPORTED 1003   /* a shape outside what the kernels were built for (Python: ValueError) */

#define CHESS_OUT_F16 0
#define CHESS_OUT_BF16 1
#define CHESS_OUT_F32 2

/* RMSNorm with gain, then per-row symmetric int8: q[M, D], scale[M] = absmax / 127.
 * With original != NULL it first stores mixed = fp16(x * residual_scale + original * input_scale)
 * and normalises that. Replaces model/int8_blocks.py:156-188 (norm_quant_kernel, launch_norm_quant),
 * behind the ops norm_quant (:191-198) and mix_norm_quant (:201-212). */
int chess_norm_quant(const void* x, const void* original, const void* residual_scale, const void* input_scale, const void* gain,
                     void* mixed, void* q, void* scale, int M, int D, float eps, void* stream);

/* The fp16 blocks' RMSNorm: out[M, D] = f16((x * (1 / sqrt(tree_sum(x * x) / D + eps))) * gain), the f32 order of
 * chess_norm_quant without its quantisation; with original, x is first mixed as the fp16 block's three fp16 ops round
 * it (mixed = f16(f16(x * residual_scale) + f16(original * input_scale)), written to mixed) and the mixed rows are
 * normalised. Replaces the fp16 block's input mix and ln1 (model/fused_blocks.py:346-348), its ln2 (:351) and the
 * network's final norm (:863), torch's nn.RMSNorm. */
int chess_rms_norm(const void* x, const void* original, const void* residual_scale, const void* input_scale, const void* gain, void* mixed,
                   void* out, int M, int D, float eps, void* stream);

/* h[M, N] fp16 zero-padded to width, each 32-column block times Sylvester's H32, then per-row int8:
 * q[M, width], scale[M]. rows: rows a wavefront, 1 or 2 (0 picks by size; no choice changes a bit), the role of the
 * reference's rotate_rows (model/int8_blocks.py:33-50). Replaces model/int8_blocks.py:216-246 (rotate_quant_kernel,
 * op rotate_quant). */
int chess_rotate_quant(const void* h, void* q, void* scale, int M, int N, int width, int rows, void* stream);

/* out[M, N] = epilogue(x[M, K] @ w[N(x2 if gated), K]^T) with x, w int8 and exact int32 sums;
 * epilogue: dequantise by x_scale[M] and w_scale[N(x2)], + bias[N], silu(gate) * up when gated,
 * + residual[M, N], then the next block's input mix when original != NULL; fp16 or bf16 out.
 * K % 64 == 0. tile: 0 picks by size; otherwise (rows x outputs, wavefronts along rows x along outputs, ring stages):
 *   1 64x64 (2x2, 4)   2 128x128 (2x2, 4)   3 128x64 (2x2, 4)   4 256x128 (4x2, 3)   5 128x128 (4x2, 2)
 *   6 128x128 (4x2, 3)   7 128x128 (2x2, 3)   8 128x64 (2x2, 3)   9 128x64 (2x2, 2)   10 256x64 (4x1, 2)
 *   11 128x128 (2x2, 2)   12 128x64 (2x2, 2)   13 128x128 (2x2, 2)
 * with stages of 64 bytes of K, except 5, 12 and 13: 128 bytes (K a multiple of 128 bytes); 14 is 32x32 with K split
 * over 4 wavefronts, for few rows (K = 512, 1024 or 2048 and N % 8 == 0: the role of small_int8); 15 holds each
 * wavefront's weights in registers and streams x in 32-row blocks, eight wavefronts a compute unit (K = 512, N % 8 == 0,
 * fp16 or bf16 out, no residual or mix); 16 holds K = 2048 in registers split over four wavefronts, whose int32 partials
 * meet in LDS, and streams x in 16-row blocks (down's launch: N % 128 == 0, not gated, no bias, the residual added with or
 * without the mix, fp16 or bf16 out). No tile changes a bit.
 * Pointer order of small_int8 (model/int8_cuda.py:35-39); replaces int8_linear_kernel
 * and small_int8 (model/int8_blocks.py:66-144, model/int8_cuda.py:34-183, :362-383). */
int chess_int8_linear(const void* x, const void* x_scale, const void* w, const void* w_scale, const void* bias, const void* residual,
                      const void* original, const void* residual_scale, const void* input_scale, void* out, int M, int N, int K,
                      int gated, int out_dtype, int tile, void* stream);

/* The raw int32 sums out[M, N] = x[M, K] @ w[N, K]^T of the same kernel, for checking them to the bit
 * (the reference reads them only through its epilogue: model/int8_blocks.py:85-97). */
int chess_int8_matmul_i32(const void* x, const void* w, void* out, int M, int N, int K, int tile, void* stream);

/* The gated chess_int8_linear (silu(gate) * up, fp16 out, no bias) that also writes, for each row and 32-column block of
 * its fp16 outputs, the largest magnitude of that block times Sylvester's H32 as chess_rotate_quant rotates it:
 * block_absmax[M][N / 32] f32. N % 128 == 0; tiles as chess_int8_linear's, not 14 to 16. The first half of
 * model/int8_blocks.py:284-286 (gate_up, then rotate_quant's row maxima) for chess_rotated_int8_linear. */
int chess_gated_int8_linear_absmax(const void* x, const void* x_scale, const void* w, const void* w_scale, void* out, void* block_absmax,
                                   int M, int N, int K, int tile, void* stream);

/* out[M, N] = epilogue(q[M, K] @ w[N, K]^T), q and its row scales being what chess_rotate_quant makes of h[M, K] (fp16,
 * K == the rotated width: no padding columns), from h and its block maxima (chess_gated_int8_linear_absmax) in one launch:
 * the same bits as chess_rotate_quant followed by chess_int8_linear. Epilogue as chess_int8_linear's (bias, residual,
 * next block's input mix), fp16 out. K % 64 == 0. tile: 0 or 1 128 x 512, 2 64 x 512, 3 128 x 256, 4 64 x 256 (rows x
 * outputs, eight wavefronts). model/int8_blocks.py:285-288 (rotate_quant, then the down int8_linear). */
int chess_rotated_int8_linear(const void* h, const void* block_absmax, const void* w, const void* w_scale, const void* bias,
                              const void* residual, const void* original, const void* residual_scale, const void* input_scale, void* out,
                              int M, int N, int K, int tile, void* stream);

/* Template attention of B positions of T tokens (64 <= T <= 128): projected[B, T, H*dq | KV*dq | KV*dv | H*tc]
 * fp16, keyed_templates[64, 64, 8] fp16 (keyed[i][j][t] = templates[t][i][j] for t < tc, zero beyond; 16-byte
 * aligned), q_gain/k_gain[dq] fp16 -> out[B, T, H*dv] fp16; scale = 1/sqrt(dq).
 * A workgroup takes groups_per_block (position, key/value group) pairs in a row, which may run across positions
 * (any divisor of B * KV; it changes no bit). Up to 80 tokens with dq and dv up to 64 the launch shares its pairs out by
 * itself, and groups_per_block is only checked.
 * Replaces template_attention_cuda (model/attention_cuda.py:97-304, launch :379-391, pointer order
 * projected, paired templates, q_gain, k_gain, out; templates paired once, :410-440) and the Triton pair
 * template_bias_kernel + template_attention_kernel (model/fused_blocks.py:35-171). */
int chess_template_attention(const void* projected, const void* keyed_templates, const void* q_gain, const void* k_gain, void* out, int B,
                             int T, int heads, int kv_heads, int dq, int dv, int templates_count, int groups_per_block, float eps,
                             float scale, void* stream);

/* chess_template_attention with projected and out in bf16 (query and value widths up to 64): the same arguments,
 * keyed_templates and the gains still fp16. The normalised queries and keys, the template bias and the scores stay
 * fp16 as in the fp16 entry point; P V runs on the bf16 MFMA with P rounded to bf16.
 * No counterpart in the reference, whose attention is fp16 only (model/attention_cuda.py:97-304): the benchmark's config 2
 * (4,096 positions x 8 heads x 64, 64 tokens) asks for bf16 Q/K/V and a bf16 output. */
int chess_template_attention_bf16(const void* projected, const void* keyed_templates, const void* q_gain, const void* k_gain, void* out,
                                  int B, int T, int heads, int kv_heads, int dq, int dv, int templates_count, int groups_per_block,
                                  float eps, float scale, void* stream);

/* out[M, N] = epilogue(x[M, K] @ W[K, N(x2 if gated)]), x and W fp16 (W in_features x out_features), f32 sums,
 * taken as w = W^T, row-major [N(x2), K] (the gate's rows, then up's); epilogue + bias, silu(gate) * up,
 * + residual, input mix as chess_int8_linear; fp16 or f32 (accumulate_fp32) out. K % 32 == 0; tile as
 * chess_int8_linear, 14 excepted; 15 takes K = 512, not gated, bias and residual without mix, fp16 out (the attention's
 * output projection). Replaces linear_kernel / launch_linear (model/fused_blocks.py:229-304) behind the op
 * linear (:308-318), whose K x N weight the Python layer transposes once. */
int chess_linear(const void* x, const void* w, const void* bias, const void* residual, const void* original, const void* residual_scale,
                 const void* input_scale, void* out, int M, int N, int K, int gated, int out_dtype, int tile, void* stream);

/* The network's input out[B, T, D] fp16 from boards[B, T] of token codes (code_bytes 1, 4 or 8 each; 64 <= T <= 128):
 * embed[code] + position[t] (+ the 64 squares' 23 feature rows of table, summed in f32 in slot order and rounded to
 * fp16), summed in f32. The rows are found from the boards: rays[64][8][8] (each square's squares along the 8 directions,
 * nearest first, 64 past the edge), jumps[64][8] (its knight jumps, 64 off the board), offsets[23] (each feature's first
 * row), all int32, and the piece codes given. Rows and codes are clamped into the tables (embed_rows, table_rows).
 * Replaces board_embedding_kernel / the op board_embedding (model/fused_blocks.py:412-491) and input_embedding
 * (:376-409) with SquareFeatures.indices (model/model.py:128-174). */
int chess_board_embedding(const void* boards, int code_bytes, const void* rays, const void* jumps, const void* offsets, const void* embed,
                          const void* position, const void* table, void* out, int B, int T, int D, int embed_rows, int table_rows, int pawn,
                          int knight, int queen, int king, int theirs, int edge, int no_piece, void* stream);

/* The policy head's move logits of B positions after its `a` matmul (model/fused_blocks.py:863-872, the heads without
 * fused ends): x[B, T, D] the final norm's rows (fp16), a[B, T, D] = x @ a_weight (f32, rows 0..63 read), a_bias[D],
 * w[NN, D] and w_bias[NN] the narrow projections (f32: s, the promotion logits, board_down's inputs from down_first),
 * cells[moves] = from * 64 + to and promotions[moves] = to' * 32 + column of the move's promotion logit or -1 (int32).
 * out[b * out_stride + m] f32 = ((a[from] + a_bias) . x[to]) + narrow[from][0] (+ narrow[to'][column]), m < moves
 * (out_stride = moves + 1 writes the answer rows' logits in place); down[B, T, NN - down_first] f32 =
 * narrow[t][down_first..NN), through nn.GELU when activate (board_down_project's activation, the value head's input).
 * 64 <= T <= 96, D % 64 == 0, NN <= 32. The products go through workspace (at least B * 7,168 * 4 bytes: a position's 64 x 64
 * logits and 96 x 32 narrow products), which the call allocates nothing for. Replaces the torch ops of :866-871 (the f32
 * linear, the transposed bmm, the gathers and the promotion sum). */
int chess_move_logits(const void* x, const void* a, const void* a_bias, const void* w, const void* w_bias, const void* cells,
                      const void* promotions, void* out, void* down, void* workspace, long long workspace_bytes, int B, int T, int D, int NN,
                      int down_first, int moves, int out_stride, int activate, void* stream);

/* The value head of B positions (the eval head after board_down_project, model/model.py:200-201, and the expected score,
 * :37-41; the reference's fused head_value_tile / head_value_kernel, model/fused_blocks.py:649-728): from c[B, K] f32,
 * board_down's activated outputs (K = T * 16), hidden[b][u] = gelu(c[b] . hidden_weight[u] + hidden_bias[u]) (u < H,
 * hidden_weight [H, K] f32), logit[b][v] = hidden[b] . out_weight[v] + out_bias[v] (v < bins <= 128, out_weight
 * [bins, H] f32), and rows[b * row_stride + score_column] = sum_v softmax(logit[b])[v] * centres[v]; value_logits[B, bins]
 * f32 as well unless NULL. All f32, nn.GELU's erf form. The hidden layer goes through workspace (at least B * H * 4
 * bytes, 16-byte aligned), which the call allocates nothing for. K % 16 == 0, H % 16 == 0. */
int chess_value_head(const void* c, const void* hidden_weight, const void* hidden_bias, const void* out_weight, const void* out_bias,
                     const void* centres, void* value_logits, void* rows, void* workspace, long long workspace_bytes, int B, int K, int H,
                     int bins, int row_stride, int score_column, void* stream);

/* chess_value_head without a workspace: the hidden layer goes through the library's own file-scope device array of
 * 2,097,152 floats (8 MiB a GPU, held from the library's load to the process's end), so that the call allocates
 * nothing and takes no workspace. B * H above 2,097,152 (4,096 positions at 512 units) is refused (CHESS_UNSUPPORTED).
 * Every call on one GPU shares that GPU's array: calls that overlap on one GPU race. No counterpart in the reference:
 * it is for callers that cannot allocate (code under graph capture, serving loops that forbid allocation). */
int chess_value_head_no_alloc(const void* c, const void* hidden_weight, const void* hidden_bias, const void* out_weight, const void* out_bias,
                              const void* centres, void* value_logits, void* rows, int B, int K, int H, int bins, int row_stride,
                              int score_column, void* stream);

/* The lean lanes' answers (engine/inference.py:131-137, Lane.answer's gather on a lean lane): rows[B][row_bytes] hold at
 * byte columns_at `columns` little-endian int16 indices into a board's answer row (answer_rows[B][width] f32: the moves'
 * logits then the expected score, :19-23; the row layout of engine/selfplay_rs/src/lib.rs:331-333). answers[B][columns]
 * f32 = answer_rows[b][index]; an index outside [0, width) gives NaN. Replaces the torch.gather from the answer rows.
 * rows, row_bytes and columns_at even. */
int chess_lean_answers(const void* answer_rows, const void* rows, void* answers, int B, int width, int row_bytes, int columns_at, int columns,
                       void* stream);

/* Fills table[0..6] with hipSetDevice, hipMemcpyAsync, hipGraphLaunch, hipEventRecord, hipEventSynchronize,
 * hipStreamSynchronize, hipGetErrorString: the address table of engine/cuda_runtime.py:17-49 (CudaRuntime.CALLS
 * and addresses()), whose HIP functions have the CUDA ones' signatures; the native round loop
 * (engine/selfplay_rs/src/rounds.rs:19-56) calls them by address. */
int chess_runtime_addresses(void** table, int count);

/* A graph lane's batch in: with `device` current, bytes of input copied from pinned input_host to input on stream, the
 * recorded graph (a hipGraphExec_t) launched on stream, and the event done recorded behind it. The four runtime calls
 * that the reference's GraphedBatches.launch_filled makes one at a time (engine/inference.py:183-195). A failed step
 * returns its HIP error, and chess_last_error names the step. */
int chess_lane_submit(int device, void* stream, void* input, const void* input_host, size_t bytes, void* graph, void* done);

/* A graph lane's batch out: with `device` current, a wait on done when sleep is non-zero, then bytes of output copied
 * to pinned output_host on stream and the stream awaited: GraphedBatches.collect (engine/inference.py:199-214). It
 * blocks; Python binds it so that it releases the GIL while it waits. */
int chess_lane_fetch(int device, void* stream, void* done, int sleep, void* output_host, const void* output, size_t bytes);

/* A description of a code, and the message of the last refused call on this thread. */
const char* chess_error_string(int code);
const char* chess_last_error(void);

/* The GPU target the library was built for ("gfx950"). */
const char* chess_target(void);

#ifdef __cplusplus
}
#endif

#endif
