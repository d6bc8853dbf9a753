// vx_bf16.hpp — f32 values as sums of bfloat16 terms, for the bf16 matrix
// cores (no reference counterpart).
//
// A bf16 value has 8 significant bits and float's exponent range, so a float
// is the sum of three bf16 terms exactly, and of two to within 2^-16 of its
// magnitude. Products of two bf16 values are exact in f32, and the matrix
// cores add them in f32: a contraction over three terms is an f32
// contraction, at a rate of 1/3 (one operand split) of ~2.5 PFLOP/s against
// the f32 matrix cores' 157 TFLOP/s.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// (a, b) rounded to nearest even, a in the low half.
__device__ __forceinline__ uint32_t vx_pk_bf16(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf16x2));
}

// The high halves of (a, b), a in the low half: both truncated to bf16.
__device__ __forceinline__ uint32_t vx_pk_hi(uint32_t a, uint32_t b) {
    return __builtin_amdgcn_perm(b, a, 0x07060302u);
}

// v[0..8) as NT terms of packed bf16, largest first. The leading terms are
// truncated (a rounded one could overflow to infinity for |v| near the
// largest float; the remainder v - trunc(v) is exact either way). NT = 3: the
// last term has at most 8 bits left, so the three add up to v exactly, except
// for bits of v below 2^-133, bf16's smallest number (there are any only where
// |v| < 2^-110). NT = 2: the last term is rounded, error <= 2^-16 |v|. An infinity
// gives {inf, NaN, ..}, a NaN {NaN, ..}.
template <int NT>
__device__ __forceinline__ void vx_split8(const float (&v)[8], u32x4 (&t)[NT]) {
    float r[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) r[i] = v[i];
#pragma unroll
    for (int k = 0; k < NT - 1; ++k) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t a = __float_as_uint(r[2 * i]), b = __float_as_uint(r[2 * i + 1]);
            t[k][i] = vx_pk_hi(a, b);
            r[2 * i] -= __uint_as_float(a & 0xFFFF0000u);
            r[2 * i + 1] -= __uint_as_float(b & 0xFFFF0000u);
        }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
        t[NT - 1][i] = NT == 3 ? vx_pk_hi(__float_as_uint(r[2 * i]), __float_as_uint(r[2 * i + 1]))
                               : vx_pk_bf16(r[2 * i], r[2 * i + 1]);
}

// v[0..8) as three terms of packed bf16 rounded to nearest, largest first, with
// |second| <= 2^-8 |v| and |third| <= 2^-16 |v| of either sign, so that in a
// product of two such sums the three smallest of the nine terms are below 2^-24
// of it and average out. |v| above 3.39e38 rounds to an infinity. The three add
// up to v exactly, except for bits of v below 2^-133, bf16's smallest number
// (there are any only where |v| < 2^-110): `lost` then gets some of its low 16
// bits set, and only then (the last remainder has 8 bits; NaNs apart).
__device__ __forceinline__ void vx_split8_rne(const float (&v)[8], u32x4 (&t)[3], uint32_t& lost) {
    float r[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) r[i] = v[i];
#pragma unroll
    for (int k = 0; k < 3; ++k)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t h = vx_pk_bf16(r[2 * i], r[2 * i + 1]);
            t[k][i] = h;
            if (k == 2) lost |= __float_as_uint(r[2 * i]) | __float_as_uint(r[2 * i + 1]);
            r[2 * i] -= __uint_as_float(h << 16);
            r[2 * i + 1] -= __uint_as_float(h & 0xFFFF0000u);
        }
    asm("" : "+v"(lost));  // (formed here: left free, the compiler kept the remainders)
}

// A second look at those of the T rows (or columns) x0.. of an operand for which
// want(x) holds, element (x, k) at base[x sx + k sk]; those past X repeat the
// last. mx[x]: the bits of the largest |element| (above 0x7F800000: it holds a
// NaN); ls[x]: whether three bf16 terms miss bits of an element (below 2^-110 and
// no multiple of 2^-133, which adding 1.5 x 2^-110 rounds it to). Lanes follow K
// where that is the dimension of stride 1 (KC), else x. All nw waves of the
// workgroup take part; mx and ls are in LDS, zeroed before.
template <bool KC, uint32_t T, class Want>
__device__ __forceinline__ void vx_scan(const float* base, int64_t sx, int64_t sk, uint32_t x0, uint32_t X, uint32_t K,
                                        uint32_t wave, uint32_t nw, uint32_t lane, uint32_t* mx, uint32_t* ls,
                                        Want want) {
    constexpr uint32_t L = T < 64u ? T : 64u;  // lanes along x
    for (uint32_t x = KC ? wave : lane % L; x < T; x += KC ? nw : L) {
        if (!want(x)) continue;
        const float* p = base + (int64_t)min(x0 + x, X - 1u) * sx;
        uint32_t m = 0u, l = 0u;
        auto take = [&](float v) {
            const uint32_t u = __float_as_uint(v) & 0x7FFFFFFFu;
            m = max(m, u);
            l |= (uint32_t)(u < 0x08800000u /* 2^-110 */) & (uint32_t)((v + 0x1.8p-110f) - 0x1.8p-110f != v);
        };
        // 16 loads in flight
        const uint32_t k0 = KC ? lane : wave * (64u / L) + lane / L, step = KC ? 64u : nw * (64u / L);
        const int64_t ks = KC ? 1 : sk;
        const float* q = p + (int64_t)k0 * ks;
        uint64_t k = 0;
        for (; k + 16u * step <= K; k += 16u * step, q += (int64_t)(16u * step) * ks) {
            float v[16];
#pragma unroll
            for (int j = 0; j < 16; ++j) v[j] = q[(int64_t)j * (KC ? 64 : (int64_t)step * sk)];
#pragma unroll
            for (int j = 0; j < 16; ++j) take(v[j]);
        }
        if (k < K) {  // (past K the last element again: no branches between the loads)
            const uint32_t rem = (uint32_t)(K - k) - 1u;
            q = p + (int64_t)k * ks;
            float v[16];
#pragma unroll
            for (uint32_t j = 0; j < 16u; ++j) v[j] = q[(int64_t)min(k0 + j * step, rem) * ks];
#pragma unroll
            for (int j = 0; j < 16; ++j) take(v[j]);
        }
        if constexpr (KC) {
#pragma unroll
            for (int o = 32; o; o >>= 1) m = max(m, (uint32_t)__shfl_xor((int)m, o, 64));
            if (lane == 0u) mx[x] = m;  // (no other wave has x)
        } else {
            atomicMax(&mx[x], m);
        }
        if (l) ls[x] = 1u;
    }
}
