// Device-side helpers shared by the kernel files.
#pragma once
#include <hip/hip_fp16.h>
#include "common.hpp"

namespace cg {

__device__ __forceinline__ uint32_t fastdiv(uint32_t n, const FastDiv &f) {
    uint32_t t = __umulhi(f.m, n);
    return (t + ((n - t) >> f.s1)) >> f.s2;
}

__device__ __forceinline__ float asf(uint32_t b) { return __uint_as_float(b); }
__device__ __forceinline__ uint32_t asu(float f) { return __float_as_uint(f); }

// The f32 word of one element of a narrow format, and back (exact: a word that is stored narrow holds a value of the format).
__device__ __forceinline__ uint32_t f8_word_of_dev(uint8_t b);
__device__ __forceinline__ uint8_t f8_byte_of_dev(uint32_t u);

// VEC consecutive elements (element stride o.is) of a NARROW operand, widened to f32 words.  VEC 4 or 8 with unit stride:
// one load of 8 or 16 bytes (16-bit formats), of 4 or 8 bytes (fp8); the planner has checked the alignment.
template <int VEC>
__device__ __forceinline__ void load_narrow(const Operand &o, int64_t off, uint32_t (&r)[VEC]) {
    if (o.fmt == kFmtF8) {
        const uint8_t *p = reinterpret_cast<const uint8_t *>(o.ptr) + off;
        if (VEC >= 4 && o.is == 1) {
            uint32_t t[VEC >= 8 ? 2 : 1];
            if (VEC >= 8) {
                const uint2 q = *reinterpret_cast<const uint2 *>(p);
                t[0] = q.x;
                t[VEC >= 8 ? 1 : 0] = q.y;
            } else {
                t[0] = *reinterpret_cast<const uint32_t *>(p);
            }
#pragma unroll
            for (int j = 0; j < VEC; j++) r[j] = f8_word_of_dev((uint8_t)(t[j / 4] >> (8 * (j % 4))));
        } else if (o.is == 0) {
            const uint32_t t = f8_word_of_dev(*p);
#pragma unroll
            for (int j = 0; j < VEC; j++) r[j] = t;
        } else {
#pragma unroll
            for (int j = 0; j < VEC; j++) r[j] = f8_word_of_dev(p[(int64_t)j * o.is]);
        }
        return;
    }
    const uint16_t *p = reinterpret_cast<const uint16_t *>(o.ptr) + off;
    uint16_t h[VEC];
    if (VEC >= 4 && o.is == 1) {
        uint32_t t[VEC / 2 > 0 ? VEC / 2 : 1];
        if (VEC >= 8) {
            const uint4 q = *reinterpret_cast<const uint4 *>(p);
            t[0] = q.x;
            t[1 % (VEC / 2 > 0 ? VEC / 2 : 1)] = q.y;
            t[2 % (VEC / 2 > 0 ? VEC / 2 : 1)] = q.z;
            t[3 % (VEC / 2 > 0 ? VEC / 2 : 1)] = q.w;
        } else {
            const uint2 q = *reinterpret_cast<const uint2 *>(p);
            t[0] = q.x;
            t[1 % (VEC / 2 > 0 ? VEC / 2 : 1)] = q.y;
        }
#pragma unroll
        for (int j = 0; j < VEC; j++) h[j] = (uint16_t)(t[j / 2] >> (16 * (j % 2)));
    } else if (o.is == 0) {
        const uint16_t t = *p;
#pragma unroll
        for (int j = 0; j < VEC; j++) h[j] = t;
    } else {
#pragma unroll
        for (int j = 0; j < VEC; j++) h[j] = p[(int64_t)j * o.is];
    }
#pragma unroll
    for (int j = 0; j < VEC; j++)
        r[j] = o.fmt == kFmtBF16 ? (uint32_t)h[j] << 16 : __float_as_uint(__half2float(__ushort_as_half(h[j])));
}

// f32 words that hold values of a narrow format, stored as that format's patterns.
template <int VEC, bool STREAM = false>
__device__ __forceinline__ void store_narrow(const Operand &o, int64_t off, const uint32_t (&r)[VEC]) {
    typedef uint32_t u4 __attribute__((ext_vector_type(4)));
    typedef uint32_t u2 __attribute__((ext_vector_type(2)));
    if (o.fmt == kFmtF8) {
        uint8_t *p = reinterpret_cast<uint8_t *>(const_cast<char *>(o.ptr)) + off;
        if (VEC >= 4 && o.is == 1) {
            uint32_t t[VEC >= 8 ? 2 : 1] = {};
#pragma unroll
            for (int j = 0; j < VEC; j++) t[j / 4] |= (uint32_t)f8_byte_of_dev(r[j]) << (8 * (j % 4));
            if (VEC >= 8) {
                const u2 v = {t[0], t[VEC >= 8 ? 1 : 0]};
                if (STREAM) __builtin_nontemporal_store(v, reinterpret_cast<u2 *>(p));
                else *reinterpret_cast<u2 *>(p) = v;
            } else {
                *reinterpret_cast<uint32_t *>(p) = t[0];
            }
        } else {
#pragma unroll
            for (int j = 0; j < VEC; j++) p[(int64_t)j * o.is] = f8_byte_of_dev(r[j]);
        }
        return;
    }
    uint16_t h[VEC];
#pragma unroll
    for (int j = 0; j < VEC; j++)
        h[j] = o.fmt == kFmtBF16 ? (uint16_t)(r[j] >> 16) : __half_as_ushort(__float2half_rn(__uint_as_float(r[j])));
    uint16_t *p = reinterpret_cast<uint16_t *>(const_cast<char *>(o.ptr)) + off;
    if (VEC >= 4 && o.is == 1) {
        constexpr int W = VEC / 2 > 0 ? VEC / 2 : 1;
        uint32_t t[W];
#pragma unroll
        for (int j = 0; j < W; j++) t[j] = (uint32_t)h[(2 * j) % VEC] | ((uint32_t)h[(2 * j + 1) % VEC] << 16);
        if (VEC >= 8) {
            const u4 v = {t[0], t[1 % W], t[2 % W], t[3 % W]};
            if (STREAM) __builtin_nontemporal_store(v, reinterpret_cast<u4 *>(p));
            else *reinterpret_cast<u4 *>(p) = v;
        } else {
            const u2 v = {t[0], t[1 % W]};
            if (STREAM) __builtin_nontemporal_store(v, reinterpret_cast<u2 *>(p));
            else *reinterpret_cast<u2 *>(p) = v;
        }
    } else {
#pragma unroll
        for (int j = 0; j < VEC; j++) p[(int64_t)j * o.is] = h[j];
    }
}

// (Operands lie in device memory, which the compiler does not know of a pointer that it finds in an argument block; it would load
// through the general address space, whose loads wait for everything asked for before them, LDS included.)
// WORDS: the caller knows that the operand lies in 32-bit words (kernels compiled for launches whose operands all do:
// without the narrow formats' code between its loads a program keeps them all in flight).
// IN_MEMORY: nor is it a constant (a compiled program knows which of its leaves are).
template <int VEC, bool STREAM = false, bool WORDS = false, bool IN_MEMORY = false>
__device__ __forceinline__ void load_words(const Operand &o, int64_t off, uint32_t (&r)[VEC]) {
    if (!IN_MEMORY && o.uniform) {
#pragma unroll
        for (int j = 0; j < VEC; j++) r[j] = o.ubits;
        return;
    }
    if (!WORDS && o.fmt != kFmtWords) { // (the same for every lane: the format is a launch parameter)
        load_narrow<VEC>(o, off, r);
        return;
    }
    typedef const __attribute__((address_space(1))) uint32_t global_word;
    global_word *p = reinterpret_cast<global_word *>(reinterpret_cast<uintptr_t>(o.ptr)) + off;
    if (VEC >= 4 && o.is == 1) {
        typedef uint32_t u4 __attribute__((ext_vector_type(4)));
        typedef const __attribute__((address_space(1))) u4 global_u4;
#pragma unroll
        for (int q = 0; q < VEC / 4; q++) {
            const u4 t = STREAM ? __builtin_nontemporal_load(reinterpret_cast<global_u4 *>(p) + q) : reinterpret_cast<global_u4 *>(p)[q];
            r[(4 * q) % VEC] = t[0];
            r[(4 * q + 1) % VEC] = t[1];
            r[(4 * q + 2) % VEC] = t[2];
            r[(4 * q + 3) % VEC] = t[3];
        }
    } else if (o.is == 0) {
        uint32_t t = *p;
#pragma unroll
        for (int j = 0; j < VEC; j++) r[j] = t;
    } else {
#pragma unroll
        for (int j = 0; j < VEC; j++) r[j] = p[(int64_t)j * o.is];
    }
}

// STREAM: the output is far larger than the caches; non-temporal stores keep it from
// evicting the operands that are still being read.
template <int VEC, bool STREAM = false, bool WORDS = false>
__device__ __forceinline__ void store_words(const Operand &o, int64_t off, const uint32_t (&r)[VEC]) {
    if (!WORDS && o.fmt != kFmtWords) {
        store_narrow<VEC, STREAM>(o, off, r);
        return;
    }
    uint32_t *p = reinterpret_cast<uint32_t *>(const_cast<char *>(o.ptr)) + off;
    if (VEC >= 4 && o.is == 1) {
        typedef uint32_t u4 __attribute__((ext_vector_type(4)));
#pragma unroll
        for (int q = 0; q < VEC / 4; q++) {
            const u4 v = {r[(4 * q) % VEC], r[(4 * q + 1) % VEC], r[(4 * q + 2) % VEC], r[(4 * q + 3) % VEC]};
            if (STREAM) __builtin_nontemporal_store(v, reinterpret_cast<u4 *>(p) + q);
            else reinterpret_cast<u4 *>(p)[q] = v;
        }
    } else {
#pragma unroll
        for (int j = 0; j < VEC; j++) p[(int64_t)j * o.is] = r[j];
    }
}


// Rust `f32 as u32` (ndarray.rs:155): truncate, saturate, NaN -> 0.
__device__ __forceinline__ uint32_t f32_as_u32(float v) {
    if (!(v == v) || v <= 0.0f) return 0u;
    if (v >= 4294967296.0f) return 0xFFFFFFFFu;
    return (uint32_t)v;
}

__device__ __forceinline__ uint32_t wrapping_pow(uint32_t a, uint32_t e) {
    uint32_t acc = 1;
    while (e) {
        if (e & 1) acc *= a;
        a *= a;
        e >>= 1;
    }
    return acc;
}

// (On the device the conversion instructions round; they agree with the closed forms below on all 2^32 patterns.  SiLU gating of
// 8192 x 8192 bfloat16 values, which is bound by its arithmetic: 141 -> 111 us; adding as many fp8 values: 139 -> 93.)
typedef float float2cv __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2cv __attribute__((ext_vector_type(2)));

// f32 bits -> bits of the nearest bfloat16 value (ties to even), as f32; NaNs stay NaNs (quiet)
__host__ __device__ __forceinline__ uint32_t round_bf16_bits(uint32_t u) {
#ifdef __HIP_DEVICE_COMPILE__
    const float2cv v = {asf(u), 0.0f};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2cv)) << 16;
#endif
    if ((u & 0x7FFFFFFFu) > 0x7F800000u) return (u | 0x00400000u) & 0xFFFF0000u;
    return (u + 0x7FFFu + ((u >> 16) & 1u)) & 0xFFFF0000u;
}

// fp8 = E4M3 (float8::F8E4M3): 4 exponent bits with bias 7, 3 mantissa bits, no infinities, 0x7F the NaN, largest
// finite value 448, subnormals m * 2^-9.  f32 bits -> f32 bits of the nearest such value (ties to even); 448 and
// beyond, infinities included, give +-448 (the crate's saturating conversion); NaN stays NaN.
__host__ __device__ __forceinline__ uint32_t round_f8_bits(uint32_t u) {
    const uint32_t sign = u & 0x80000000u, a = u & 0x7FFFFFFFu;
#ifdef __HIP_DEVICE_COMPILE__
    const float x = asf((a < 0x43E00000u ? a : 0x43E00000u) | sign);
    const float y = __builtin_amdgcn_cvt_f32_fp8(__builtin_amdgcn_cvt_pk_fp8_f32(x, x, 0, false), 0);
    return a > 0x7F800000u ? sign | 0x7FC00000u : asu(y);
#endif
    if (a > 0x7F800000u) return sign | 0x7FC00000u;
    if (a >= 0x43E00000u) return sign | 0x43E00000u; // 448
    if (a < 0x3C800000u) {                           // below 2^-6: whole multiples of 2^-9
        const float units = rintf(__builtin_bit_cast(float, a) * 512.0f);
        return sign | __builtin_bit_cast(uint32_t, units * (1.0f / 512.0f));
    }
    const uint32_t r = (a + 0x7FFFFu + ((a >> 20) & 1u)) & 0xFFF00000u; // a carry runs into the exponent
    return sign | (r > 0x43E00000u ? 0x43E00000u : r);
}
// the byte of a representable value, and back
__host__ __device__ __forceinline__ uint8_t f8_byte_of(uint32_t u) {
    const uint8_t sign = (uint8_t)((u >> 24) & 0x80u);
    const uint32_t a = u & 0x7FFFFFFFu;
    if (a > 0x7F800000u) return sign | 0x7Fu;
#ifdef __HIP_DEVICE_COMPILE__
    return (uint8_t)__builtin_amdgcn_cvt_pk_fp8_f32(asf(u), asf(u), 0, false);
#endif
    if (a >= 0x3C800000u) return sign | (uint8_t)((((a >> 23) - 120u) << 3) | ((a >> 20) & 7u));
    return sign | (uint8_t)(uint32_t)(__builtin_bit_cast(float, a) * 512.0f);
}
__host__ __device__ __forceinline__ uint32_t f8_word_of(uint8_t b) {
    const uint32_t sign = (uint32_t)(b & 0x80u) << 24, e = (b >> 3) & 0xFu, m = b & 7u;
    if (e == 0xFu && m == 7u) return sign | 0x7FC00000u;
#ifdef __HIP_DEVICE_COMPILE__
    return asu(__builtin_amdgcn_cvt_f32_fp8((int)b, 0));
#endif
    if (e != 0) return sign | ((e + 120u) << 23) | (m << 20);
    return sign | __builtin_bit_cast(uint32_t, (float)m * (1.0f / 512.0f));
}

__device__ __forceinline__ uint32_t f8_word_of_dev(uint8_t b) { return f8_word_of(b); }
__device__ __forceinline__ uint8_t f8_byte_of_dev(uint32_t u) { return f8_byte_of(u); }

// One scalar application of OP on raw 32-bit words.  F = operands are f32.
template <int OP, bool F>
__device__ __forceinline__ uint32_t apply(uint32_t a, uint32_t b, uint32_t c, uint32_t *fault) {
    (void)b;
    (void)c;
    (void)fault;
    if constexpr (OP == kCopy) return a;
    if constexpr (OP == kCastF2U) return f32_as_u32(asf(a));
    if constexpr (OP == kCastU2F) return asu((float)a); // round to nearest even
    if constexpr (OP == kWhere) return F ? (asf(a) > 0.0f ? b : c) : (a != 0 ? b : c);
    if constexpr (F) {
        float x = asf(a), y = asf(b);
        if constexpr (OP == kNeg) return a ^ 0x80000000u;
        if constexpr (OP == kSin) return asu(sinf(x));
        if constexpr (OP == kCos) return asu(cosf(x));
        if constexpr (OP == kExp) return asu(expf(x));
        if constexpr (OP == kLog) return asu(logf(x));
        if constexpr (OP == kFloor) return asu(floorf(x));
        if constexpr (OP == kRound) return asu(rintf(x)); // ties to even (ndarray.rs:646-648)
        if constexpr (OP == kRoundBF16) return round_bf16_bits(a);
        if constexpr (OP == kRoundF16) return asu(__half2float(__float2half_rn(x))); // v_cvt_f16_f32: nearest even, overflow -> inf
        if constexpr (OP == kRoundF8) return round_f8_bits(a);
        if constexpr (OP == kAdd) return asu(x + y);
        if constexpr (OP == kSub) return asu(x - y);
        if constexpr (OP == kMul) return asu(x * y);
        if constexpr (OP == kDiv) return asu(x / y);
        if constexpr (OP == kPow) return asu(powf(x, y));
        if constexpr (OP == kLt) return asu(x < y ? 1.0f : 0.0f);
        if constexpr (OP == kGt) return asu(x > y ? 1.0f : 0.0f);
        if constexpr (OP == kGte) return asu(x >= y ? 1.0f : 0.0f);
        if constexpr (OP == kLte) return asu(x <= y ? 1.0f : 0.0f);
        if constexpr (OP == kEq) return asu(x == y ? 1.0f : 0.0f);
    } else {
        if constexpr (OP == kNeg) return 0u - a;
        if constexpr (OP == kAdd) return a + b;
        if constexpr (OP == kSub) return a - b;
        if constexpr (OP == kMul) return a * b;
        if constexpr (OP == kDiv) {
            if (b == 0) {
                *fault = kFaultDivZero; // reported by the next waiting call
                return 0u;
            }
            return a / b;
        }
        if constexpr (OP == kPow) return wrapping_pow(a, b);
        if constexpr (OP == kLt) return a < b;
        if constexpr (OP == kGt) return a > b;
        if constexpr (OP == kGte) return a >= b;
        if constexpr (OP == kLte) return a <= b;
        if constexpr (OP == kEq) return a == b;
    }
    return 0u;
}

// What an RMS norm divides a row by, pow(sum / n + eps, e), in the norm's own ops but for the power: a square root where e is one half, as in
// every model's norms (powf takes 0.7 us of a launch of 5; where they are not the same, at and below zero, it stays).  For every kernel that
// applies such a norm beside other work, so that a row's divisor does not depend on which of them it is.
__device__ __forceinline__ float norm_divisor(float squares, uint32_t n_bits, uint32_t eps_bits, uint32_t exp_bits) {
    const uint32_t mean = apply<kAdd, true>(apply<kDiv, true>(asu(squares), n_bits, 0, nullptr), eps_bits, 0, nullptr);
    if (exp_bits == 0x3F000000u && asf(mean) > 0.0f) return sqrtf(asf(mean));
    return asf(apply<kPow, true>(mean, exp_bits, 0, nullptr));
}

// Sum over the 64 lanes of a wave, for every lane: inside rows of 16 lanes by shifts, then from row to row, all without LDS.
template <int CTRL, int ROWS> __device__ __forceinline__ float add_shifted(float v) {
    return v + asf((uint32_t)__builtin_amdgcn_update_dpp(0, (int)asu(v), CTRL, ROWS, 0xF, true));
}
__device__ __forceinline__ float wave_total(float v) {
    v = add_shifted<0x111, 0xF>(v); // row_shr 1, 2, 4, 8
    v = add_shifted<0x112, 0xF>(v);
    v = add_shifted<0x114, 0xF>(v);
    v = add_shifted<0x118, 0xF>(v);
    v = add_shifted<0x142, 0xA>(v); // the first row's sum into the second, the third's into the fourth
    v = add_shifted<0x143, 0xC>(v); // the lower half's into the upper
    return asf((uint32_t)__builtin_amdgcn_readlane((int)asu(v), 63));
}

// f over the lanes of a wave at distances 32, 16 .. LOW, left in all of them: what a butterfly of shuffles gives, to the bit, where f
// does not mind the order of its two operands.  (Below 16 lanes by rotation: the values repeat by then.)  A shuffle is a trip through
// LDS, and a chain of six of them, 64 cycles each, is longer than the memory's latency behind which nothing else is left to do.
template <int CTRL> __device__ __forceinline__ uint32_t row_rotated(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xF, 0xF, true);
}
template <class F> __device__ __forceinline__ uint32_t fold_halves(uint32_t v, F f) { // lanes 32 apart
    const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    return f((uint32_t)r[0], (uint32_t)r[1]);
}
template <class F> __device__ __forceinline__ uint32_t fold_rows(uint32_t v, F f) { // lanes 16 apart
    const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    return f((uint32_t)r[0], (uint32_t)r[1]);
}
template <int LOW, class F> __device__ __forceinline__ uint32_t wave_fold(uint32_t v, F f) {
    static_assert(LOW == 1 || LOW == 2 || LOW == 4 || LOW == 8 || LOW == 16 || LOW == 32, "a distance between lanes");
    v = fold_halves(v, f);
    if constexpr (LOW <= 16) v = fold_rows(v, f);
    if constexpr (LOW <= 8) v = f(v, row_rotated<0x128>(v));
    if constexpr (LOW <= 4) v = f(v, row_rotated<0x124>(v));
    if constexpr (LOW <= 2) v = f(v, row_rotated<0x122>(v));
    if constexpr (LOW <= 1) v = f(v, row_rotated<0x121>(v));
    return v;
}
// Values and pointers that the compiler knows nothing of but their scalar registers: what a lane chooses among such is chosen, not branched
// for, and not fetched from the argument block lane by lane.
typedef const __attribute__((address_space(1))) float global_float;
__device__ __forceinline__ int64_t pinned(int64_t v) {
    asm volatile("" : "+s"(v));
    return v;
}
__device__ __forceinline__ global_float *pinned(const float *p) { return reinterpret_cast<global_float *>(pinned(reinterpret_cast<int64_t>(p))); }
struct AddWords {
    __device__ __forceinline__ uint32_t operator()(uint32_t a, uint32_t b) const { return asu(asf(a) + asf(b)); }
};
template <int LOW> __device__ __forceinline__ float wave_add(float v) { return asf(wave_fold<LOW>(asu(v), AddWords{})); }
// The value of the lane DIST away
template <int DIST> __device__ __forceinline__ uint32_t across(uint32_t v) {
    static_assert(DIST == 1 || DIST == 2 || DIST == 4 || DIST == 8 || DIST == 16 || DIST == 32, "a bit of the lane's number");
    if constexpr (DIST == 32) {
        const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
        return threadIdx.x & 32 ? (uint32_t)r[0] : (uint32_t)r[1];
    } else if constexpr (DIST == 16) {
        const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
        return threadIdx.x & 16 ? (uint32_t)r[0] : (uint32_t)r[1];
    } else if constexpr (DIST == 8) {
        return row_rotated<0x128>(v);
    } else if constexpr (DIST == 4) { // four up in the lower quads of a pair, four down in the upper
        const uint32_t up = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x104, 0xF, 0x5, false);
        return (uint32_t)__builtin_amdgcn_update_dpp((int)up, (int)v, 0x114, 0xF, 0xA, false);
    } else {
        return row_rotated<DIST == 2 ? 0x4E : 0xB1>(v);
    }
}
template <int DIST> __device__ __forceinline__ float add_across(float v) { return v + asf(across<DIST>(asu(v))); }
struct LargerWords {
    __device__ __forceinline__ uint32_t operator()(uint32_t a, uint32_t b) const { return asu(fmaxf(asf(a), asf(b))); }
};
// f over groups of W lanes, their nearest neighbours first (1, 2 .. W / 2): quads repeat by the time that they are mirrored
template <int W, class F> __device__ __forceinline__ uint32_t group_fold_up(uint32_t v, F f) {
    static_assert(W == 2 || W == 4 || W == 8 || W == 16 || W == 32 || W == 64, "a group of lanes");
    v = f(v, across<1>(v));
    if constexpr (W > 2) v = f(v, across<2>(v));
    if constexpr (W > 4) v = f(v, row_rotated<0x141>(v)); // (eight lanes mirrored)
    if constexpr (W > 8) v = f(v, row_rotated<0x140>(v)); // (sixteen)
    if constexpr (W > 16) v = fold_rows(v, f);
    if constexpr (W > 32) v = fold_halves(v, f);
    return v;
}
// ... and their farthest ones first (W / 2 .. 1)
template <int W, class F> __device__ __forceinline__ uint32_t group_fold(uint32_t v, F f) {
    static_assert(W == 1 || W == 2 || W == 4 || W == 8 || W == 16 || W == 32 || W == 64, "a group of lanes");
    if constexpr (W > 32) v = fold_halves(v, f);
    if constexpr (W > 16) v = fold_rows(v, f);
    if constexpr (W > 8) v = f(v, across<8>(v));
    if constexpr (W > 4) v = f(v, across<4>(v));
    if constexpr (W > 2) v = f(v, across<2>(v));
    if constexpr (W > 1) v = f(v, across<1>(v));
    return v;
}
// The sum over the lanes at distances LOW, 2 LOW .. 32, in that order
template <int LOW> __device__ __forceinline__ float wave_add_up(float v) {
    if constexpr (LOW <= 1) v = add_across<1>(v);
    if constexpr (LOW <= 2) v = add_across<2>(v);
    if constexpr (LOW <= 4) v = add_across<4>(v);
    if constexpr (LOW <= 8) v += asf(row_rotated<0x128>(asu(v)));
    if constexpr (LOW <= 16) v = asf(fold_rows(asu(v), AddWords{}));
    return asf(fold_halves(asu(v), AddWords{}));
}
// The sums of four values over the lanes at distances 32, 16, 8 and 4, in that order: of v[r] in row r (lanes 16 r .. 16 r + 15).  Two
// values share a register from the first step on, four from the second.
__device__ __forceinline__ float four_sums(float a, float b, float c, float d) {
    const auto ac = __builtin_amdgcn_permlane32_swap(asu(a), asu(c), false, false);
    const auto bd = __builtin_amdgcn_permlane32_swap(asu(b), asu(d), false, false);
    const float x = asf((uint32_t)ac[0]) + asf((uint32_t)ac[1]), y = asf((uint32_t)bd[0]) + asf((uint32_t)bd[1]);
    const auto xy = __builtin_amdgcn_permlane16_swap(asu(x), asu(y), false, false);
    float v = asf((uint32_t)xy[0]) + asf((uint32_t)xy[1]);
    v += asf(row_rotated<0x128>(asu(v)));
    return v + asf(row_rotated<0x124>(asu(v)));
}

// Offset (in elements) of row `row` of a view whose outer axes are described by
// (od, odiv, os), innermost first.
__device__ __forceinline__ int64_t row_offset(uint32_t row, uint32_t nouter, const uint32_t *od, const FastDiv *odiv,
                                              const int64_t *os) {
    int64_t off = 0;
    for (uint32_t d = 0; d < nouter; d++) {
        uint32_t q = fastdiv(row, odiv[d]);
        off += (int64_t)(row - q * od[d]) * os[d];
        row = q;
    }
    return off;
}

} // namespace cg
