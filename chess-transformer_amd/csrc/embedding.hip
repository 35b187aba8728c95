// The network's input: boards of T token codes in, out[B, T, D] fp16 =
//   f16( (f32(embed[code]) + f32(position[t])) + f32(f16(sum over the 23 square features of table[row])) )
// the last term for the 64 square tokens only, its rows found from the board itself, as
// model/fused_blocks.py:412-469 (board_embedding_kernel) and model/model.py:128-174 (SquareFeatures.indices)
// find them: where the kings and queens are from the square, the codes of its 8 neighbours, the first piece
// along each of 8 lines and how far out, the knights attacking it, the nearest pawn up and down its file.
// The features are summed in f32 in their slot order (0..22), then rounded to fp16 (model/fused_blocks.py:383-393).
//
// A workgroup takes one board's run of TOKENS_A_GROUP tokens (9 workgroups a board of 70), so that a batch of one board
// still spreads over the chip: it reads the whole board's codes and finds its kings and queens, then its squares' 23
// rows with one thread a (square, direction), then gathers the rows of its (token, 8 columns) items, 16 bytes a lane,
// two items a thread. The gather is bound by its 23 KB of table rows a square (512 columns: 1.5 GB from L2 in a launch of
// 1,024 boards, 21 TB/s), and by its instructions: a value takes one, a mixed fma that reads the fp16 half as f32 (times 1, so
// that it rounds as the sum alone), and a row one address, from its place in 16-byte chunks; a conversion, an addition and
// 64-bit products of rows and widths took 80.7 us where these take 70.1 (1,024 boards of 512 columns on an MI355X; one board
// 7.5 and 6.2: the rays and jumps are read with the board). Runs of up to 32 tokens a workgroup, finding rows with all
// its threads, were no faster (69.8 us). Row numbers are clamped into the table (and codes into the embedding), so that a board
// with codes the encoding never makes reads no memory outside the tables.
#include "chess_common.h"

namespace {

constexpr int SQUARES = 64;
constexpr int FEATURES = 23;
constexpr int STEPS = 8;          // a ray's squares, nearest first: 7 and a pad, 64 past the edge

typedef int Words __attribute__((ext_vector_type(4), aligned(4)));

struct Codes {
    int pawn, knight, queen, king, theirs, edge, no_piece;
};

constexpr int TOKENS_A_GROUP = 8;
constexpr int THREADS = 256;

// Place: what holds a row's place in the table, in 16-byte chunks: 32 bits, or 64 for tables of 64 GiB or more
template <typename Code, typename Place>
__global__ __launch_bounds__(THREADS) void board_embedding_kernel(
    const Code* __restrict__ boards, const int* __restrict__ rays, const int* __restrict__ jumps, const int* __restrict__ offsets,
    const half_t* __restrict__ embed, const half_t* __restrict__ position, const half_t* __restrict__ table, half_t* __restrict__ out,
    int T, int D, int embed_rows, int table_rows, Codes codes)
{
    __shared__ int square_codes[SQUARES + 1];     // the 65th is the code past the edge
    __shared__ int token_codes[TOKENS_A_GROUP];
    __shared__ int first[4];
    __shared__ __align__(16) Place rows[TOKENS_A_GROUP][FEATURES + 1];

    const int tid = threadIdx.x;
    const int groups = (T + TOKENS_A_GROUP - 1) / TOKENS_A_GROUP, chunks = D / 8;
    const size_t b = blockIdx.x / groups;
    const int t0 = (blockIdx.x % groups) * TOKENS_A_GROUP, tokens = min(TOKENS_A_GROUP, T - t0);
    const Code* board = boards + b * T;
    // thread (square of the run, direction d); its ray and jump are read before the board's codes are there
    const int local = tid / 8, d = tid % 8, s = t0 + local;
    const bool finds = local < tokens && s < SQUARES;
    const int at_ray = (finds ? s * 8 + d : 0) * STEPS;
    const Words near = *reinterpret_cast<const Words*>(rays + at_ray), far = *reinterpret_cast<const Words*>(rays + at_ray + 4);
    const int jump = jumps[finds ? s * 8 + d : 0];
    if (tid < SQUARES) square_codes[tid] = (int)board[tid];
    if (tid < TOKENS_A_GROUP) token_codes[tid] = tid < tokens ? min(max((int)board[t0 + tid], 0), embed_rows - 1) : 0;
    if (tid == SQUARES) square_codes[SQUARES] = codes.edge;
    if (tid < 4) first[tid] = SQUARES;
    __syncthreads();
    const int pieces[4] = {codes.king, codes.king + codes.theirs, codes.queen, codes.queen + codes.theirs};
    if (tid < SQUARES) {
#pragma unroll
        for (int i = 0; i < 4; i++)
            if (square_codes[tid] == pieces[i]) atomicMin(&first[i], tid);
    }
    __syncthreads();

    // the neighbour's code and the line's first piece along d, and for d < 2 the nearest pawn along the file; direction 0's
    // thread also the kings' and queens' places and the knights, which it counts over the square's eight threads
    const int jump_code = square_codes[min(max(jump, 0), SQUARES)];
    const uint64_t ours_at = __ballot(finds && jump_code == codes.knight), theirs_at = __ballot(finds && jump_code == codes.knight + codes.theirs);
    auto place = [&](int row) { return (Place)min(max(row, 0), table_rows - 1) * (Place)chunks; };
    if (finds) {
        const int file = s % 8, rank = s / 8;
        Place* row = rows[local];
        const int steps[STEPS] = {near[0], near[1], near[2], near[3], far[0], far[1], far[2], far[3]};
        const int pawn_theirs = codes.pawn + codes.theirs;
        int line = 0, pawn = 0;
        bool line_found = false, pawn_found = false;
#pragma unroll
        for (int k = 0; k < STEPS; k++) {
            const int code = square_codes[min(max(steps[k], 0), SQUARES)];
            if (k == 0) row[4 + d] = place(code + offsets[4 + d]);
            if (!line_found && code != 0 && code != codes.edge) {
                line = 1 + (code - 1) * 7 + k;
                line_found = true;
            }
            if (d < 2 && !pawn_found && (code == codes.pawn || code == pawn_theirs)) {
                pawn = 1 + (code == pawn_theirs ? 7 : 0) + k;
                pawn_found = true;
            }
        }
        row[12 + d] = place(line + offsets[12 + d]);
        if (d < 2) row[21 + d] = place(pawn + offsets[21 + d]);
        if (d == 0) {
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int p = first[i];
                const int value = p < SQUARES ? (rank - p / 8 + 7) * 15 + file - p % 8 + 7 : codes.no_piece;
                row[i] = place(value + offsets[i]);
            }
            const int shift = (tid & 63) - d;
            const int ours = __popcll(ours_at >> shift & 0xFF), theirs = __popcll(theirs_at >> shift & 0xFF);
            row[20] = place(min(ours, 2) * 3 + min(theirs, 2) + offsets[20]);
        }
    }
    __syncthreads();

    float one = 1.0f;
    asm volatile("" : "+s"(one));   // unknown to the compiler, which would split the fma by 1 into a conversion and a sum
    for (int item = tid; item < tokens * chunks; item += THREADS) {
        const int local_token = item / chunks, token = t0 + local_token, chunk = item % chunks, d0 = chunk * 8;
        const v8h e = *reinterpret_cast<const v8h*>(embed + (size_t)token_codes[local_token] * D + d0);
        const v8h p = *reinterpret_cast<const v8h*>(position + (size_t)token * D + d0);
        float total[8];
#pragma unroll
        for (int c = 0; c < 8; c++) total[c] = (float)e[c] + (float)p[c];
        if (token < SQUARES) {
            float features[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
            for (int f = 0; f < FEATURES; f++) {
                const v8h t = reinterpret_cast<const v8h*>(table)[(size_t)(rows[local_token][f] + chunk)];
#pragma unroll
                for (int c = 0; c < 8; c++) features[c] = __builtin_fmaf((float)t[c], one, features[c]);
            }
#pragma unroll
            for (int c = 0; c < 8; c++) total[c] = total[c] + (float)(half_t)features[c];
        }
        v8h result;
#pragma unroll
        for (int c = 0; c < 8; c++) result[c] = (half_t)total[c];
        *reinterpret_cast<v8h*>(out + (b * T + token) * D + d0) = result;
    }
}

}  // namespace

extern "C" int chess_board_embedding(const void* boards, int code_bytes, const void* rays, const void* jumps, const void* offsets,
                                     const void* embed, const void* position, const void* table, void* out, int B, int T, int D,
                                     int embed_rows, int table_rows, int pawn, int knight, int queen, int king, int theirs, int edge,
                                     int no_piece, void* stream)
{
    if (B < 0 || T < SQUARES || T > 128 || D <= 0 || D % 8 != 0 || embed_rows <= 0 || table_rows <= 0)
        return chess_fail(CHESS_INVALID_SHAPE, "board_embedding takes 64 to 128 tokens and a width a multiple of 8 (T %d, D %d)", T, D);
    if (code_bytes != 1 && code_bytes != 4 && code_bytes != 8)
        return chess_fail(CHESS_UNSUPPORTED, "board_embedding reads codes of 1, 4 or 8 bytes, not %d", code_bytes);
    if (B == 0) return CHESS_OK;   // no positions: nothing read or written, so the pointers may be null
    if (!boards || !rays || !jumps || !offsets || !embed || !position || !table || !out)
        return chess_fail(CHESS_INVALID_SHAPE, "board_embedding: a required pointer is null");
    if (!aligned16(embed) || !aligned16(position) || !aligned16(table) || !aligned16(out))
        return chess_fail(CHESS_MISALIGNED, "board_embedding's 16-byte loads need aligned tables and output");
    const Codes codes{pawn, knight, queen, king, theirs, edge, no_piece};
    const long grid = (long)B * ((T + TOKENS_A_GROUP - 1) / TOKENS_A_GROUP);
    const bool wide = (uint64_t)table_rows * (D / 8) >= (1ull << 32);
    auto launch = [&](auto code) {
        typedef decltype(code) Code;
        auto kernel = wide ? board_embedding_kernel<Code, uint64_t> : board_embedding_kernel<Code, uint32_t>;
        hipLaunchKernelGGL(kernel, dim3(grid), dim3(THREADS), 0, (hipStream_t)stream, (const Code*)boards,
                           (const int*)rays, (const int*)jumps, (const int*)offsets, (const half_t*)embed, (const half_t*)position,
                           (const half_t*)table, (half_t*)out, T, D, embed_rows, table_rows, codes);
    };
    if (code_bytes == 1) launch(uint8_t{});
    else if (code_bytes == 4) launch(int{});
    else launch((long long)0);
    return launch_status();
}
