// What the template attention's kernels share (attention.hip, attention_wave.h): LDS reads that wait for themselves, the
// widening and rounding of fp16 and bf16 rows, and the P V steps.
#pragma once

#include "lds_dma.h"


namespace {

constexpr int MAX_TEMPLATES = 8;
constexpr float LOG2E = 1.44269504f;

typedef __fp16 h2 __attribute__((ext_vector_type(2)));

DEVICE float dot2(uint32_t a, uint32_t b, float c) {
    return __builtin_amdgcn_fdot2(__builtin_bit_cast(h2, a), __builtin_bit_cast(h2, b), c, false);
}

// A 16-byte LDS read of DMA'd data as an instruction of its own, waited for by lgkmcnt and passed through an empty
// asm so that no use moves above the wait: read through a pointer, the compiler would first wait for every DMA in
// flight (the next group's rows too), unable to tell the addresses apart.
DEVICE uint4 lds_read16_settled(const LDS_SPACE void* p) {
    v4u v;
    asm volatile("ds_read_b128 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=v"(v) : "v"((uint32_t)(uintptr_t)p) : "memory");
    return uint4{v[0], v[1], v[2], v[3]};
}

// The transposing reads of a P V step, for N = DV / 16 column groups: at base[dt] + LO and (HI) base[dt] + HI_OFF, and the
// wait for them, in one asm statement, so that the values exist only once they have landed. (Read by statements of their
// own and waited for by another, their registers could be copied by the compiler before the wait, the copy holding what
// the register held before the read landed.) Without HI the upper half is zero: keys past the staged rows, whose P is zero.
template <int N, bool HI> struct StepReads;

template <> struct StepReads<1, true> {
    template <int LO, int HI_OFF> static DEVICE void read(const uint32_t (&base)[1], v2u (&lo)[1], v2u (&hi)[1]) {
    asm volatile("ds_read_b64_tr_b16 %0, %2 offset:%3\n\t"
                 "ds_read_b64_tr_b16 %1, %2 offset:%4\n\t"
                 "s_waitcnt lgkmcnt(0)"
                 : "=&v"(lo[0]), "=&v"(hi[0])
                 : "v"(base[0]), "i"(LO), "i"(HI_OFF) : "memory");
    }
};

template <> struct StepReads<1, false> {
    template <int LO, int HI_OFF> static DEVICE void read(const uint32_t (&base)[1], v2u (&lo)[1], v2u (&hi)[1]) {
    asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2\n\t"
                 "s_waitcnt lgkmcnt(0)"
                 : "=&v"(lo[0])
                 : "v"(base[0]), "i"(LO) : "memory");
#pragma unroll
    for (int dt = 0; dt < 1; dt++) hi[dt] = v2u{0, 0};
    }
};

template <> struct StepReads<2, true> {
    template <int LO, int HI_OFF> static DEVICE void read(const uint32_t (&base)[2], v2u (&lo)[2], v2u (&hi)[2]) {
    asm volatile("ds_read_b64_tr_b16 %0, %4 offset:%6\n\t"
                 "ds_read_b64_tr_b16 %1, %4 offset:%7\n\t"
                 "ds_read_b64_tr_b16 %2, %5 offset:%6\n\t"
                 "ds_read_b64_tr_b16 %3, %5 offset:%7\n\t"
                 "s_waitcnt lgkmcnt(0)"
                 : "=&v"(lo[0]), "=&v"(hi[0]), "=&v"(lo[1]), "=&v"(hi[1])
                 : "v"(base[0]), "v"(base[1]), "i"(LO), "i"(HI_OFF) : "memory");
    }
};

template <> struct StepReads<2, false> {
    template <int LO, int HI_OFF> static DEVICE void read(const uint32_t (&base)[2], v2u (&lo)[2], v2u (&hi)[2]) {
    asm volatile("ds_read_b64_tr_b16 %0, %2 offset:%4\n\t"
                 "ds_read_b64_tr_b16 %1, %3 offset:%4\n\t"
                 "s_waitcnt lgkmcnt(0)"
                 : "=&v"(lo[0]), "=&v"(lo[1])
                 : "v"(base[0]), "v"(base[1]), "i"(LO) : "memory");
#pragma unroll
    for (int dt = 0; dt < 2; dt++) hi[dt] = v2u{0, 0};
    }
};

template <> struct StepReads<4, true> {
    template <int LO, int HI_OFF> static DEVICE void read(const uint32_t (&base)[4], v2u (&lo)[4], v2u (&hi)[4]) {
    asm volatile("ds_read_b64_tr_b16 %0, %8 offset:%12\n\t"
                 "ds_read_b64_tr_b16 %1, %8 offset:%13\n\t"
                 "ds_read_b64_tr_b16 %2, %9 offset:%12\n\t"
                 "ds_read_b64_tr_b16 %3, %9 offset:%13\n\t"
                 "ds_read_b64_tr_b16 %4, %10 offset:%12\n\t"
                 "ds_read_b64_tr_b16 %5, %10 offset:%13\n\t"
                 "ds_read_b64_tr_b16 %6, %11 offset:%12\n\t"
                 "ds_read_b64_tr_b16 %7, %11 offset:%13\n\t"
                 "s_waitcnt lgkmcnt(0)"
                 : "=&v"(lo[0]), "=&v"(hi[0]), "=&v"(lo[1]), "=&v"(hi[1]), "=&v"(lo[2]), "=&v"(hi[2]), "=&v"(lo[3]), "=&v"(hi[3])
                 : "v"(base[0]), "v"(base[1]), "v"(base[2]), "v"(base[3]), "i"(LO), "i"(HI_OFF) : "memory");
    }
};

template <> struct StepReads<4, false> {
    template <int LO, int HI_OFF> static DEVICE void read(const uint32_t (&base)[4], v2u (&lo)[4], v2u (&hi)[4]) {
    asm volatile("ds_read_b64_tr_b16 %0, %4 offset:%8\n\t"
                 "ds_read_b64_tr_b16 %1, %5 offset:%8\n\t"
                 "ds_read_b64_tr_b16 %2, %6 offset:%8\n\t"
                 "ds_read_b64_tr_b16 %3, %7 offset:%8\n\t"
                 "s_waitcnt lgkmcnt(0)"
                 : "=&v"(lo[0]), "=&v"(lo[1]), "=&v"(lo[2]), "=&v"(lo[3])
                 : "v"(base[0]), "v"(base[1]), "v"(base[2]), "v"(base[3]), "i"(LO) : "memory");
#pragma unroll
    for (int dt = 0; dt < 4; dt++) hi[dt] = v2u{0, 0};
    }
};

template <> struct StepReads<8, true> {
    template <int LO, int HI_OFF> static DEVICE void read(const uint32_t (&base)[8], v2u (&lo)[8], v2u (&hi)[8]) {
    asm volatile("ds_read_b64_tr_b16 %0, %16 offset:%24\n\t"
                 "ds_read_b64_tr_b16 %1, %16 offset:%25\n\t"
                 "ds_read_b64_tr_b16 %2, %17 offset:%24\n\t"
                 "ds_read_b64_tr_b16 %3, %17 offset:%25\n\t"
                 "ds_read_b64_tr_b16 %4, %18 offset:%24\n\t"
                 "ds_read_b64_tr_b16 %5, %18 offset:%25\n\t"
                 "ds_read_b64_tr_b16 %6, %19 offset:%24\n\t"
                 "ds_read_b64_tr_b16 %7, %19 offset:%25\n\t"
                 "ds_read_b64_tr_b16 %8, %20 offset:%24\n\t"
                 "ds_read_b64_tr_b16 %9, %20 offset:%25\n\t"
                 "ds_read_b64_tr_b16 %10, %21 offset:%24\n\t"
                 "ds_read_b64_tr_b16 %11, %21 offset:%25\n\t"
                 "ds_read_b64_tr_b16 %12, %22 offset:%24\n\t"
                 "ds_read_b64_tr_b16 %13, %22 offset:%25\n\t"
                 "ds_read_b64_tr_b16 %14, %23 offset:%24\n\t"
                 "ds_read_b64_tr_b16 %15, %23 offset:%25\n\t"
                 "s_waitcnt lgkmcnt(0)"
                 : "=&v"(lo[0]), "=&v"(hi[0]), "=&v"(lo[1]), "=&v"(hi[1]), "=&v"(lo[2]), "=&v"(hi[2]), "=&v"(lo[3]), "=&v"(hi[3]), "=&v"(lo[4]), "=&v"(hi[4]), "=&v"(lo[5]), "=&v"(hi[5]), "=&v"(lo[6]), "=&v"(hi[6]), "=&v"(lo[7]), "=&v"(hi[7])
                 : "v"(base[0]), "v"(base[1]), "v"(base[2]), "v"(base[3]), "v"(base[4]), "v"(base[5]), "v"(base[6]), "v"(base[7]), "i"(LO), "i"(HI_OFF) : "memory");
    }
};

template <> struct StepReads<8, false> {
    template <int LO, int HI_OFF> static DEVICE void read(const uint32_t (&base)[8], v2u (&lo)[8], v2u (&hi)[8]) {
    asm volatile("ds_read_b64_tr_b16 %0, %8 offset:%16\n\t"
                 "ds_read_b64_tr_b16 %1, %9 offset:%16\n\t"
                 "ds_read_b64_tr_b16 %2, %10 offset:%16\n\t"
                 "ds_read_b64_tr_b16 %3, %11 offset:%16\n\t"
                 "ds_read_b64_tr_b16 %4, %12 offset:%16\n\t"
                 "ds_read_b64_tr_b16 %5, %13 offset:%16\n\t"
                 "ds_read_b64_tr_b16 %6, %14 offset:%16\n\t"
                 "ds_read_b64_tr_b16 %7, %15 offset:%16\n\t"
                 "s_waitcnt lgkmcnt(0)"
                 : "=&v"(lo[0]), "=&v"(lo[1]), "=&v"(lo[2]), "=&v"(lo[3]), "=&v"(lo[4]), "=&v"(lo[5]), "=&v"(lo[6]), "=&v"(lo[7])
                 : "v"(base[0]), "v"(base[1]), "v"(base[2]), "v"(base[3]), "v"(base[4]), "v"(base[5]), "v"(base[6]), "v"(base[7]), "i"(LO) : "memory");
#pragma unroll
    for (int dt = 0; dt < 8; dt++) hi[dt] = v2u{0, 0};
    }
};

// f(std::integral_constant<int, I>()) for I = FIRST .. LAST - 1, in order: a loop whose index is a compile-time constant
template <int FIRST, int LAST, typename F> DEVICE void each_step(F&& f) {
    if constexpr (FIRST < LAST) {
        f(std::integral_constant<int, FIRST>());
        each_step<FIRST + 1, LAST>(f);
    }
}

DEVICE void lds_write8(LDS_SPACE void* p, uint2 v) {
    asm volatile("ds_write_b64 %0, %1" : : "v"((uint32_t)(uintptr_t)p), "v"(v) : "memory");
}

// The rows in and out are fp16, or bf16 (BF16): raw 16-bit values, widened to f32 where they are used. The normalised
// queries and keys, the template bias and the QK products stay fp16 either way (normalised values are of order one);
// with bf16 rows P V runs on the bf16 MFMA, P as a bf16 high part and low part (Probabilities), and the outputs round to
// bf16.
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
template <bool BF16> DEVICE float widen16(uint32_t bits) {
    if constexpr (BF16) return __uint_as_float(bits << 16);
    else return (float)__builtin_bit_cast(half_t, (uint16_t)bits);
}
template <bool BF16> DEVICE uint32_t narrow16(float v) {
    if constexpr (BF16) return __builtin_bit_cast(uint16_t, (__bf16)v);
    else return __builtin_bit_cast(uint16_t, (half_t)v);
}
// two f32 values rounded to 16 bits, a in the low half: the empty asm keeps them f32 values first, so that a product
// feeding one is not fused into a mixed-precision multiply-and-round (v_fma_mixlo_f16 rounds the exact product once,
// not the f32 product); the pair converts in one packed instruction
typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
template <bool BF16> DEVICE uint32_t narrow16x2(float a, float b) {
    asm volatile("" : "+v"(a), "+v"(b));
    if constexpr (BF16) return __builtin_bit_cast(uint32_t, bf2{(__bf16)a, (__bf16)b});
    else return __builtin_bit_cast(uint32_t, h2{(half_t)a, (half_t)b});
}
// a 16-byte chunk of LDS as raw 16-bit values
DEVICE uint4 lds_chunk(const LDS_SPACE int8_t* p) {
    const v4u w = *reinterpret_cast<const LDS_SPACE v4u*>(p);
    return uint4{w[0], w[1], w[2], w[3]};
}

// 8 raw values (a 16-byte chunk) as f32
template <bool BF16> DEVICE void widen8(const uint4& w, float (&out)[8]) {
    const uint32_t words[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
    for (int i = 0; i < 4; i++) {
        out[2 * i] = widen16<BF16>(words[i] & 0xFFFFu);
        out[2 * i + 1] = widen16<BF16>(words[i] >> 16);
    }
}
// 8 bf16 values as fp16 (template coefficients of order one)
DEVICE uint4 bf16_to_f16x8(const uint4& w) {
    const uint32_t words[4] = {w.x, w.y, w.z, w.w};
    uint32_t out[4];
#pragma unroll
    for (int i = 0; i < 4; i++)
        out[i] = narrow16x2<false>(widen16<true>(words[i] & 0xFFFFu), widen16<true>(words[i] >> 16));
    return uint4{out[0], out[1], out[2], out[3]};
}

// the sum of squares of 8 raw values: fp16 pairs by v_dot2_f32_f16; bf16 widened, then f32 products in order
template <bool BF16 = false> DEVICE float squares8(const uint4& w, float c) {
    if constexpr (BF16) {
        float v[8];
        widen8<true>(w, v);
#pragma unroll
        for (int i = 0; i < 8; i++) c = __builtin_fmaf(v[i], v[i], c);
        return c;
    } else {
        return dot2(w.w, w.w, dot2(w.z, w.z, dot2(w.y, w.y, dot2(w.x, w.x, c))));
    }
}
// O^T += V^T P^T for one 32-key step: the raw values (fp16 or bf16) and P (already rounded to the same type), 8 a lane
template <bool BF16> DEVICE v4f pv_step(const uint4& v, const uint4& p, v4f acc) {
    if constexpr (BF16) return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8, v), __builtin_bit_cast(bf8, p), acc, 0, 0, 0);
    else return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, v), __builtin_bit_cast(v8h, p), acc, 0, 0, 0);
}

// P V's P: fp16 rows round P to fp16, the reference's rounding point (model/attention_cuda.py:236-293); bf16 rows take P
// as a bf16 high part hi (P rounded) and low part lo = bf16(P - hi) (the subtraction exact), so that P V in bf16 carries
// about 16 bits of P, not bf16's 8, and the output's error stays that of its own bf16 rounding. low_parts gives lo's words
// for a step's 8 probabilities (two rows of 4) whose high words are hi; pv_steps adds V hi, then V lo, into acc.
template <bool BF16> DEVICE uint4 low_parts(const uint32_t (&hi)[4], const float (&first)[4], const float (&second)[4]) {
    if constexpr (BF16) {
        uint32_t lo[4];
#pragma unroll
        for (int r = 0; r < 2; r++) {
            lo[r] = narrow16x2<true>(first[2 * r] - widen16<true>(hi[r] & 0xFFFFu), first[2 * r + 1] - widen16<true>(hi[r] >> 16));
            lo[2 + r] = narrow16x2<true>(second[2 * r] - widen16<true>(hi[2 + r] & 0xFFFFu), second[2 * r + 1] - widen16<true>(hi[2 + r] >> 16));
        }
        return uint4{lo[0], lo[1], lo[2], lo[3]};
    } else {
        return uint4{0, 0, 0, 0};
    }
}
template <bool BF16> DEVICE v4f pv_steps(const uint4& v, const uint4& hi, const uint4& lo, v4f acc) {
    if constexpr (BF16) return pv_step<true>(v, lo, pv_step<true>(v, hi, acc));
    else return pv_step<false>(v, hi, acc);
}

// Raw rows are DMA'd 64 16-byte chunks an instruction, the chunks of a row in a swizzled order: chunk c of row r
// sits in slot r * CH + (c ^ swizzle(r)), which puts the 16 rows an MFMA operand group reads (one chunk each) in
// 16 different 16-byte bank groups.
template <int CH> DEVICE int swizzle(int row) { return CH >= 16 ? row % CH : (row / (16 / CH)) % CH; }
template <int CH> DEVICE int raw_slot(int row, int chunk) { return row * CH + (chunk ^ swizzle<CH>(row)); }

}  // namespace
