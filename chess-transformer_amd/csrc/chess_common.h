// Shared device helpers for the gfx950 kernels of the int8 network evaluation.
//
// Arithmetic contract: the library is built with -ffp-contract=off and IEEE
// (correctly rounded) f32 divide and sqrt, so every f32 expression below is the
// sequence of single IEEE operations it spells -- the CPU restatement under
// oracle/ computes the same sequence with numpy and gets the same bits.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

typedef _Float16 half_t;
typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v4h __attribute__((ext_vector_type(4)));

#define DEVICE __device__ __forceinline__

// Error codes beyond HIP's own (hipError_t values stay below 1000).
enum {
    CHESS_OK = 0,
    CHESS_INVALID_SHAPE = 1001,
    CHESS_MISALIGNED = 1002,
    CHESS_UNSUPPORTED = 1003,
};

// Output element types of the GEMM epilogues.
enum { OUT_F16 = 0, OUT_BF16 = 1, OUT_F32 = 2 };

struct bf16_t { uint16_t bits; };

DEVICE float to_float(half_t v) { return (float)v; }
DEVICE float to_float(bf16_t v) { return __uint_as_float(((uint32_t)v.bits) << 16); }
DEVICE float to_float(float v) { return v; }

// f32 -> bf16, round to nearest even; a NaN stays a quiet NaN: v_cvt_pk_bf16_f32, whose bits are those of the integer form
// ((bits + 0x7FFF + the kept part's last bit) >> 16) for every f32, compared over all of them. That form took six
// instructions a value where two values now take one.
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
DEVICE uint32_t bf16_pair(float low, float high) { return __builtin_bit_cast(uint32_t, bf16x2{(__bf16)low, (__bf16)high}); }
DEVICE bf16_t bf16_from_float(float f) { return bf16_t{__builtin_bit_cast(uint16_t, (__bf16)f)}; }

template <typename T> DEVICE T from_float(float f);
template <> DEVICE half_t from_float<half_t>(float f) { return (half_t)f; }
template <> DEVICE bf16_t from_float<bf16_t>(float f) { return bf16_from_float(f); }
template <> DEVICE float from_float<float>(float f) { return f; }

// silu(g) = g / (1 + 2^(-g log2 e)) from the hardware's exp2 (v_exp_f32) and reciprocal (v_rcp_f32):
// a few VALU ops, so the gated epilogue stays hidden under the MFMA work of a K=512 GEMM.
DEVICE float silu_fast(float g) {
    return g * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(g * -1.44269504f));
}

// The int8 gated epilogue's silu(g) * up from t = -g log2 e and u = -up ln 2 (whose product is g * up): t u / (1 + 2^t).
// The two constants ride on the row's scale (t = (acc * (x_scale * NEG_LOG2E)) * w_scale, and u likewise), so that an output
// takes two multiplies fewer than silu_fast(g) * up; every int8 tile computes it so, and the float64 oracle checks it at
// the reference's tolerance, as it does silu_fast.
constexpr float NEG_LOG2E = -1.44269504f;
constexpr float NEG_LN2 = -0.693147181f;
DEVICE float silu_times(float t, float u) {
    return (t * u) * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(t));
}

// lane ^ 1 and lane ^ 2 by DPP quad permutes (no LDS round trip): quad_perm [1, 0, 3, 2] and [2, 3, 0, 1]. These and
// the mirrors below read a lane of the same row that always exists, so bound_ctrl (zero for a lane that does not) never
// applies; set, it lets the compiler fold the move into the add or max that uses it (v_add_f32_dpp).
DEVICE float lane_xor1(float v) { return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xF, 0xF, true)); }
DEVICE float lane_xor2(float v) { return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x4E, 0xF, 0xF, true)); }

// lane 7 - i and lane 15 - i of each 8 and 16 lanes by DPP mirrors (row_half_mirror, row_mirror)
DEVICE float lane_mirror8(float v) { return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x141, 0xF, 0xF, true)); }
DEVICE float lane_mirror16(float v) { return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x140, 0xF, 0xF, true)); }

// Lanes l and l ^ 16 (rows of 16 lanes paired 0-1, 2-3), and l and l ^ 32, exchanged by VALU lane swaps
// (v_permlane16_swap, v_permlane32_swap) instead of an LDS permute: with the value as both operands, the swap leaves
// the pair's first value in one result and its second in the other, in every lane of the pair, so that
// first + second (or their max) is the same bits in both lanes, and the same bits as v + v[l ^ 16] (a + b == b + a).
DEVICE float sum_rows16(float v) {
    const auto pair = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(pair[0]) + __uint_as_float(pair[1]);
}
DEVICE float sum_halves32(float v) {
    const auto pair = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(pair[0]) + __uint_as_float(pair[1]);
}
DEVICE float max_rows16(float v) {
    const auto pair = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(pair[0]), __uint_as_float(pair[1]));
}
DEVICE float max_halves32(float v) {
    const auto pair = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(pair[0]), __uint_as_float(pair[1]));
}
// over the four lanes l, l ^ 16, l ^ 32, l ^ 48: the pairs of 16 first, then of 32
DEVICE float sum_across_rows(float v) { return sum_halves32(sum_rows16(v)); }
DEVICE float max_across_rows(float v) { return max_halves32(max_rows16(v)); }

// The balanced tree of adjacent lane pairs over each group of LANES lanes (16, 32 or the wavefront's 64), every lane
// of a group ending with the same bits (a + b == b + a bitwise): pairs of lanes, of 2, 4 and 8 lanes, then of 16-lane
// rows. Once a group's lanes all hold its partial, pairing lane i with 7 - i or 15 - i (DPP mirrors) adds the same two
// partials as lane i ^ 4 or i ^ 8; two rows' sums are then added by a lane-16 swap, four as (r0 + r1) + (r2 + r3) by
// the 16- and 32-lane swaps. VALU only: no LDS permutes.
template <int LANES> DEVICE float group_sum(float v) {
    static_assert(LANES == 16 || LANES == 32 || LANES == 64, "groups of 16, 32 or 64 lanes");
    v = v + lane_xor1(v);
    v = v + lane_xor2(v);
    v = v + lane_mirror8(v);
    v = v + lane_mirror16(v);
    if constexpr (LANES == 32) v = sum_rows16(v);
    if constexpr (LANES == 64) v = sum_across_rows(v);   // (r0 + r1) + (r2 + r3)
    return v;
}

template <int LANES> DEVICE float group_max(float v) {
    static_assert(LANES == 16 || LANES == 32 || LANES == 64, "groups of 16, 32 or 64 lanes");
    v = fmaxf(v, lane_xor1(v));
    v = fmaxf(v, lane_xor2(v));
    v = fmaxf(v, lane_mirror8(v));
    v = fmaxf(v, lane_mirror16(v));
    if constexpr (LANES == 32) v = max_rows16(v);
    if constexpr (LANES == 64) v = max_across_rows(v);
    return v;
}

DEVICE float wave_sum(float v) { return group_sum<64>(v); }
DEVICE float wave_max(float v) { return group_max<64>(v); }

// Maps a workgroup id so that consecutive tiles land on one XCD: the hardware deals
// workgroups to the 8 XCDs round-robin, and each XCD has its own L2.
DEVICE int xcd_local_tile(int wg, int tiles) {
    constexpr int XCDS = 8;
    // workgroups go to the XCDs in turn: XCD x gets the contiguous tiles [x q + min(x, r), ...), q + (x < r) of them
    const int q = tiles / XCDS, r = tiles % XCDS, x = wg % XCDS;
    return x * q + min(x, r) + wg / XCDS;
}

// Host-side launch-result check shared by the entry points.
static inline int launch_status() {
    hipError_t error = hipGetLastError();
    return error == hipSuccess ? CHESS_OK : (int)error;
}

// Records a message for chess_last_error() and returns code.
int chess_fail(int code, const char* format, ...);

__host__ __device__ static inline bool aligned16(const void* p) { return ((uintptr_t)p & 15u) == 0; }

// rint(y) for |y| < 2^22 as the low bits of an f32 add: y + 1.5 * 2^23 lands in [2^23, 2^24), where the f32 spacing is 1,
// so the IEEE add rounds y to the nearest integer, ties to even (1.5 * 2^23 is even), and the sum's bits are
// 0x4B400000 + rint(y): its low byte is rint(y) as a two's-complement int8 for |rint(y)| <= 127. Two VALU ops where
// v_rndne_f32 and v_cvt_i32_f32 and a byte extraction take four; the same integer as (int8_t)rintf(y) for every such y
// (a NaN gives 0 either way).
DEVICE uint32_t rounded_bits(float y) { return __float_as_uint(y + 12582912.0f); }
// the low bytes of a, b, c and d, in that order (v_perm_b32 byte selects: 0x0C selects zero)
DEVICE uint32_t low_bytes(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
    return __builtin_amdgcn_perm(b, a, 0x0C0C0400u) | __builtin_amdgcn_perm(d, c, 0x04000C0Cu);
}
