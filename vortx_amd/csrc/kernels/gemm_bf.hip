// gemm_bf.hip — f32 GEMM on the bf16 matrix cores, on canonical [n, c, rows,
// cols] views (any strides; batch dims folded into grid z).
//
// Each operand element is the exact sum of three bf16 terms (vx_bf16.hpp), and
// six of the nine products of terms are formed, down to 2^-16 of the largest;
// the others are below 2^-24 of a product, the size of one f32 rounding.
// Products of bf16 values are exact in f32 and the matrix cores add them in
// f32, so the result is as close to the exact one as that of f32 MFMAs (closer:
// at K = 4096 7.1e-7 off 64 bits against 1.15e-6, with fewer additions in
// f32), at six times the MFMA work but sixteen times the rate.
//
// Measured (graph-replayed with the same operands, same box, against the f32 MFMA
// kernels): 4096^3 973 -> 647 us (212 TFLOP/s of f32 work, 1275 of bf16; a bf16
// product of that size by the vendor's library 1370 on this card), 4096 x 11008 x
// 4096 2698 -> 1813, 1024^3 22.7 -> 19.3, 1000 x 1111 x 777 with odd strides 119
// -> 26.8, 8 x 11008 x 4096 150 -> 41 (K split; with new operands each call 179 ->
// 44), 64 x 64 x 4096 392 -> 12 (K split). The large
// shapes are bound by the matrix cores and the card's power, the smaller ones
// by the stages' serial steps (load, convert, store, barrier, read, multiply)
// with one workgroup per CU.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../vx_kargs.h"
#include "vx_bf16.hpp"
#include "vx_dpp.hpp"

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));

// Operand access: "x" is the non-K dimension (M for A, N for B).
#define MODE_K 0  // stride 1 along K
#define MODE_X 1  // any strides; best with stride 1 along x

__device__ __forceinline__ void vx_epilogue(float* c, float acc, float alpha, float beta) {
    *c = beta == 0.f ? alpha * acc : alpha * acc + beta * *c;
}

// Loads of one operand's BK x T slab of a stage: pieces of 8 k-elements of one
// x, P per thread. MODE_K: BK / 8 consecutive lanes cover a row's BK elements
// (two 16-byte loads each, 4-byte aligned); else consecutive lanes are
// consecutive in x (eight 4-byte loads, one row of k each). x past the operand
// repeats its last one (those outputs are not written). NTH threads share the
// slab (the workgroup, or half of it: the others then do the same ones).
template <int MODE, int T, int BK, int NTH, int D>
struct vx_slab {
    static constexpr int KG = BK / 8, P = T * KG / NTH;
    static_assert(P * NTH == T * KG, "whole pieces");
    float r[D][P][8];  // D stages in flight
    const float* p[P];

    static __device__ __forceinline__ uint32_t px(int u) {
        const uint32_t i = threadIdx.x % NTH + (uint32_t)(NTH * u);
        return MODE == MODE_K ? i / KG : i % T;
    }
    static __device__ __forceinline__ uint32_t pk(int u) {
        const uint32_t i = threadIdx.x % NTH + (uint32_t)(NTH * u);
        return MODE == MODE_K ? i % KG : __builtin_amdgcn_readfirstlane(i / T);  // T is a multiple of 64
    }
    __device__ __forceinline__ void init(const float* base, int64_t sx, uint32_t x0, uint32_t X) {
#pragma unroll
        for (int u = 0; u < P; ++u) {
            const uint32_t x = min(x0 + px(u), X - 1u);
            p[u] = MODE == MODE_K ? base + (int64_t)x * sx + 8u * pk(u) : base + (int64_t)x * sx;
        }
    }
    // a stage inside K
    __device__ __forceinline__ void load(int d, int u, int64_t sk, uint32_t k0) {
        if constexpr (MODE == MODE_K) {
            const f32x4_a4 a = *(const f32x4_a4*)(p[u] + k0), b = *(const f32x4_a4*)(p[u] + k0 + 4);
            r[d][u][0] = a.x; r[d][u][1] = a.y; r[d][u][2] = a.z; r[d][u][3] = a.w;
            r[d][u][4] = b.x; r[d][u][5] = b.y; r[d][u][6] = b.z; r[d][u][7] = b.w;
        } else {
            const int64_t k = (int64_t)(k0 + 8u * pk(u)) * sk;  // uniform over the wave
#pragma unroll
            for (int j = 0; j < 8; ++j) r[d][u][j] = p[u][k + j * sk];
        }
    }
    // the last stage, zeros past K
    __device__ __forceinline__ void load_tail(int d, int u, int64_t sk, uint32_t k0, uint32_t K) {
        const uint32_t kp = k0 + 8u * pk(u);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            // (loads from clamped addresses, so that all are in flight at once)
            const uint32_t k = min(kp + (uint32_t)j, K - 1u);
            const float e = MODE == MODE_K ? (p[u] - 8u * pk(u))[k] : p[u][(int64_t)k * sk];
            r[d][u][j] = kp + (uint32_t)j < K ? e : 0.f;
        }
    }
    // terms of piece u to LDS: [k16][x / 32][term][64 lanes], lane (n, g) of
    // an MFMA operand (row n, k 8g..8g+7) at g 32 + (n ^ 4 kg), kg = 2 k16 + g:
    // the xor spreads the pieces that 8 consecutive lanes store over the banks
    __device__ __forceinline__ void store(int d, int u, u32x4* S, uint32_t& lost) {
        u32x4 t[3];
        vx_split8_rne(r[d][u], t, lost);
        const uint32_t x = px(u), kg = pk(u);
        u32x4* o = S + (((kg >> 1) * (T / 32) + (x >> 5)) * 3u) * 64u + (kg & 1u) * 32u + ((x & 31u) ^ (4u * kg));
#pragma unroll
        for (int k = 0; k < 3; ++k) o[64 * k] = t[k];
    }
};

// One operand's chunk of 32 elements of K of lane (n, g)'s x for the bf16 terms:
// H pieces of 8 elements (H G = 4; 32 x 32 tiles: g 0..1; 16 x 16: g 0..3). SO:
// the lane group's part of the address in the base, the rest a scalar offset,
// where both operands are read along M / N (600 x 600 x 1000 17.6 -> 16.9 us; with
// one along K the lane's offset in every address is as fast or faster, 300 x 517 x
// 600 7.11 / 6.99).
template <int MODE, int H, int G, bool SO>
struct vx_chunk {
    static constexpr uint32_t KC = 8u * G * H;
    float r[H][8];
    // what load and load_tail take for the lane's row or column p
    static __device__ __forceinline__ const float* base(const float* p, int64_t sk, uint32_t g) {
        return SO ? p + (int64_t)(8u * g) * sk : p;
    }
    __device__ __forceinline__ void load(const float* p, int64_t sk, uint32_t k0, uint32_t g) {
#pragma unroll
        for (int h = 0; h < H; ++h) {
            if constexpr (MODE == MODE_K) {
                const float* q = p + (k0 + 8u * G * h + 8u * g);
                const f32x4_a4 a = *(const f32x4_a4*)q, b = *(const f32x4_a4*)(q + 4);
                r[h][0] = a.x; r[h][1] = a.y; r[h][2] = a.z; r[h][3] = a.w;
                r[h][4] = b.x; r[h][5] = b.y; r[h][6] = b.z; r[h][7] = b.w;
            } else {
#pragma unroll
                for (int j = 0; j < 8; ++j) r[h][j] = p[(int64_t)(k0 + 8u * G * h + (SO ? 0u : 8u * g) + (uint32_t)j) * sk];
            }
        }
    }
    __device__ __forceinline__ void load_tail(const float* p, int64_t sk, uint32_t k0, uint32_t g, uint32_t K) {
#pragma unroll
        for (int h = 0; h < H; ++h)
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const uint32_t k = k0 + 8u * G * h + 8u * g + (uint32_t)j, kc = min(k, K - 1u);
                const float e = MODE == MODE_K ? p[kc] : p[((int64_t)kc - (SO ? 8u * g : 0u)) * sk];  // (clamped: no branches between the loads)
                r[h][j] = k < K ? e : 0.f;
            }
    }
};

// The same of 16 elements for f32 products in the order of K: step s of a product
// takes element G s + g.
template <int MODE, int G>
struct vx_seq {
    static constexpr uint32_t KC = 16u;
    static constexpr int NS = 16 / G, NR = MODE == MODE_K ? 16 : NS;
    float r[NR];
    static __device__ __forceinline__ const float* base(const float* p, int64_t sk, uint32_t g) { return MODE == MODE_K ? p : p + (int64_t)g * sk; }
    __device__ __forceinline__ void load(const float* p, int64_t sk, uint32_t k0, uint32_t) {
        if constexpr (MODE == MODE_K) {
#pragma unroll
            for (int j = 0; j < 16; j += 4) {
                const f32x4_a4 a = *(const f32x4_a4*)(p + k0 + j);
                r[j] = a.x; r[j + 1] = a.y; r[j + 2] = a.z; r[j + 3] = a.w;
            }
        } else {
#pragma unroll
            for (int s = 0; s < NS; ++s) r[s] = p[(int64_t)(k0 + (uint32_t)(G * s)) * sk];
        }
    }
    __device__ __forceinline__ void load_tail(const float* p, int64_t sk, uint32_t k0, uint32_t g, uint32_t K) {
#pragma unroll
        for (int j = 0; j < NR; ++j) {
            const uint32_t k = k0 + (MODE == MODE_K ? (uint32_t)j : (uint32_t)(G * j) + g), kc = min(k, K - 1u);
            const float e = MODE == MODE_K ? p[kc] : p[((int64_t)kc - g) * sk];
            r[j] = k < K ? e : 0.f;
        }
    }
    __device__ __forceinline__ float at(int s, uint32_t g) const {
        if constexpr (MODE != MODE_K) {
            return r[s];
        } else {
            // (bit masks: a choice between array elements went through scratch memory)
            float e = 0.f;
#pragma unroll
            for (uint32_t j = 0; j < (uint32_t)G; ++j) {
                const uint32_t m = g == j ? ~0u : 0u;
                e = __uint_as_float(__float_as_uint(e) | (__float_as_uint(r[G * s + j]) & m));
            }
            return e;
        }
    }
};

// K in chunks, chunks w, w + nw, ... of it to mult(a, b, odd chunk) straight
// from memory (no LDS, no barrier, one chunk ahead): pa and pb point at element 0
// of the lane's row of A and column of B.
template <class CA, class CB, class Mult>
__device__ __forceinline__ void vx_chunks(const vx_gemm_args& p, const float* pa, const float* pb, uint32_t g, uint32_t w, uint32_t nw,
                                          const Mult& mult) {
    constexpr uint32_t KC = CA::KC;
    pa = CA::base(pa, p.as[3], g);
    pb = CB::base(pb, p.bs[2], g);
    const uint32_t nck = p.K / KC;  // whole chunks
    if (w < nck) {
        CA a[2];
        CB b[2];
        const uint32_t last = (nck - 1u - w) / nw * nw + w;  // this wave's last chunk
        auto load = [&](int d, uint32_t c) {
            a[d].load(pa, p.as[3], min(c, last) * KC, g);
            b[d].load(pb, p.bs[2], min(c, last) * KC, g);
        };
        load(0, w);
        load(1, w + nw);
        uint32_t c = w;
        for (; c + nw <= last; c += 2u * nw) {
            // (each chunk's next loads go out as soon as it is split: left free,
            // the compiler issued both chunks' at the end of the round)
            __builtin_amdgcn_sched_barrier(0);
            mult(a[0], b[0], 0);
            load(0, c + 2u * nw);
            __builtin_amdgcn_sched_barrier(0);
            mult(a[1], b[1], 1);
            load(1, c + 3u * nw);
        }
        if (c <= last) mult(a[0], b[0], 0);
    }
    if (p.K % KC != 0u && w == nck % nw) {
        CA a;
        CB b;
        a.load_tail(pa, p.as[3], nck * KC, g, p.K);
        b.load_tail(pb, p.bs[2], nck * KC, g, p.K);
        mult(a, b, 1);
    }
}

// 32 x 32 or 16 x 16 outputs of a wave as f32 multiply-adds from the first k to
// the last, one rounding each: the f32 matrix cores add a step's products one
// after another in the order of the lane groups g (so measured, bit for bit).
// Where a sum overflows on the way, or infinities meet, this order decides; the
// same one in every kernel.
template <int AM, int BM>
__device__ __forceinline__ void vx_f32_tile(const vx_gemm_args& p, const float* pa, const float* pb, uint32_t g, f32x16& acc) {
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[v] = 0.f;
    vx_chunks<vx_seq<AM, 2>, vx_seq<BM, 2>>(p, pa, pb, g, 0u, 1u, [&](const auto& a, const auto& b, int) {
#pragma unroll
        for (int s = 0; s < 8; ++s) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a.at(s, g), b.at(s, g), acc, 0, 0, 0);
    });
}
template <int AM, int BM>
__device__ __forceinline__ void vx_f32_tile(const vx_gemm_args& p, const float* pa, const float* pb, uint32_t g, f32x4& acc) {
    acc = f32x4{0.f, 0.f, 0.f, 0.f};
    vx_chunks<vx_seq<AM, 4>, vx_seq<BM, 4>>(p, pa, pb, g, 0u, 1u, [&](const auto& a, const auto& b, int) {
#pragma unroll
        for (int s = 0; s < 4; ++s) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a.at(s, g), b.at(s, g), acc, 0, 0, 0);
    });
}

// Outputs of a tile that lost bits of an operand (vx_split8_rne), or that holds
// an output for which odd() is true, are looked at again. The tile's rows of A
// and columns of B are scanned (vx_scan); where one holds a NaN, so does the
// output. Any other is formed from f32 products (vx_f32_tile)
//   where it is not finite: the terms of an infinity hold a NaN;
//   where it is below 2^-120: its six sums would be rounded to 2^-149 each;
//   where an element of its row or column misses bits, up to 2^-134 each, and
//   they may count: K 2^-134 max|b| + K 2^-134 max|a| against 2^-24 of it.
// (The matrix cores keep subnormal operands, products and sums.)
// What this takes, us, without / a NaN in every row of A (the scan) / an infinity
// in every row (all outputs formed again; bound by the f32 matrix cores and, in
// the K split kernels, by one wave's loads): 4000 x 4011 x 1000 195 / 288 / 764,
// 2100 x 1900 x 1000 60 / 87 / 241, 970 x 1000 x 2000 42 / 65 / 135, 300 x 517 x
// 4096 32 / 52 / 173. One lane per output, in the same order of additions, took
// 12000 to 36000 on the first with NaNs.
__device__ __forceinline__ bool vx_gemm_bf_odd(float s) {
    const float v = __builtin_fabsf(s);
    return !(v < __builtin_inff()) || (v < 0x1p-120f && v > 0.f);
}
// ra, cb: the bits of the largest |a| of the row and |b| of the column (a NaN's are larger)
__device__ __forceinline__ bool vx_gemm_bf_again(float s, uint32_t K, uint32_t ra, bool rlost, uint32_t cb, bool clost) {
    if (ra > 0x7F800000u || cb > 0x7F800000u) return false;
    const float big = fmaxf(rlost ? __uint_as_float(cb) : 0.f, clost ? __uint_as_float(ra) : 0.f);
    return vx_gemm_bf_odd(s) || ((rlost || clost) && !(__builtin_fabsf(s) >= (float)K * 0x1p-109f * big));
}

extern __shared__ __align__(16) uint8_t vx_bf_lds[];

// A stage is 32 ST elements of K. Even and odd steps of 16 are added up apart and
// the two sums at the end, in every tile shape, so that all
// give the same bits: a wave holds both (HS 1), or, where tiles are few or
// small, twice as many waves hold one each (HS 2) and meet in LDS.
template <int AM, int BM, int TM, int TN, int WM, int WN, int HS, int ST>
__device__ __forceinline__ void vx_gemm_bf(const vx_gemm_args& p) {
    constexpr int BK = 32 * ST, KH = 2 * ST, NTH = 64 * WM * WN * HS, MI = TM / WM / 32, NJ = TN / WN / 32, NA = 2 / HS;
    constexpr int D = HS;  // stages requested ahead of the one being converted (registers allow two with HS 2)
    constexpr uint32_t SA = KH * (TM / 32) * 3u * 64u, SB = KH * (TN / 32) * 3u * 64u;  // pieces per buffer
    u32x4* SAp = (u32x4*)vx_bf_lds;
    u32x4* SBp = SAp + 2u * SA;

    // Tile order: workgroup ids are regrouped per XCD (dealt round robin over
    // 8), then walked in groups of 8 tile rows, so that an XCD's resident
    // tiles share panels of A and B in its L2.
    const uint32_t nt = p.tiles_m * p.tiles_n;
    const uint32_t bid = vx_xcd_order(blockIdx.x, nt);
    const uint32_t group = 8u * p.tiles_n;
    const uint32_t first_m = (bid / group) * 8u;
    const uint32_t gsize = min(p.tiles_m - first_m, 8u);
    const uint32_t m0 = (first_m + (bid % group) % gsize) * TM, n0 = (bid % group) / gsize * TN;
    const uint32_t z = blockIdx.z;
    const uint32_t bn = z / p.batch_c, bc = z % p.batch_c;
    const float* A = p.a + bn * p.as[0] + bc * p.as[1];
    const float* B = p.b + bn * p.bs[0] + bc * p.bs[1];
    float* C = p.c + bn * p.cs[0] + bc * p.cs[1];

    const uint32_t lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t wh = wave / (WM * WN), wm = wave / WN % WM, wn = wave % WN, n = lane & 31u, g = lane >> 5;

    f32x16 acc[NA][MI][NJ];
#pragma unroll
    for (int q = 0; q < NA; ++q)
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[q][i][j][v] = 0.f;

    // DUTY: small tiles have a piece for every thread in A and B together; the
    // first half of the waves takes A's, the second half B's
    constexpr bool DUTY = (TM + TN) * (BK / 8) == NTH;
    vx_slab<AM, TM, BK, DUTY ? NTH / 2 : NTH, D> a;
    vx_slab<BM, TN, BK, DUTY ? NTH / 2 : NTH, D> b;
    constexpr int PA = a.P, PB = b.P;
    const bool dutyb = DUTY && wave >= (uint32_t)(NTH / 128);
    a.init(A, p.as[2], m0, p.M);
    b.init(B, p.bs[3], n0, p.N);

    uint32_t lost = 0u;  // see vx_split8_rne
    const uint32_t nkf = p.K / BK;
    // accumulator q: half h of the stage in buffer buf
    auto mult = [&](uint32_t buf, int q, uint32_t h) {
        const uint32_t slot = g * 32u + (n ^ (4u * (2u * h + g)));
        const u32x4* sa = SAp + buf * SA + (h * (TM / 32) + wm * MI) * 192u + slot;
        const u32x4* sb = SBp + buf * SB + (h * (TN / 32) + wn * NJ) * 192u + slot;
        bf16x8 fa[MI][3], fb[NJ][3];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
#pragma unroll
            for (int i = 0; i < MI; ++i) fa[i][k] = __builtin_bit_cast(bf16x8, sa[i * 192 + k * 64]);
#pragma unroll
            for (int j = 0; j < NJ; ++j) fb[j][k] = __builtin_bit_cast(bf16x8, sb[j * 192 + k * 64]);
        }
        constexpr int TA[6] = {2, 0, 1, 1, 0, 0}, TB[6] = {0, 2, 1, 0, 1, 0};  // smallest products first
#pragma unroll
        for (int e = 0; e < 6; ++e)
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int j = 0; j < NJ; ++j)
                    acc[q][i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i][TA[e]], fb[j][TB[e]], acc[q][i][j], 0, 0, 0);
    };
    // stage st's elements to registers (slot d), and from there to LDS
    auto load = [&](int d, uint32_t st) {
        const uint32_t k0 = min(st, nkf - 1u) * BK;
        if (!DUTY || !dutyb) {
#pragma unroll
            for (int u = 0; u < PA; ++u) a.load(d, u, p.as[3], k0);
        }
        if (!DUTY || dutyb) {
#pragma unroll
            for (int u = 0; u < PB; ++u) b.load(d, u, p.bs[2], k0);
        }
    };
    auto store = [&](int d, uint32_t buf) {
        if (!DUTY || !dutyb) {
#pragma unroll
            for (int u = 0; u < PA; ++u) a.store(d, u, SAp + buf * SA, lost);
        }
        if (!DUTY || dutyb) {
#pragma unroll
            for (int u = 0; u < PB; ++u) b.store(d, u, SBp + buf * SB, lost);
        }
    };
    // stage st from its buffer; stage st + 1 is converted to the other one
    // from slot d, which then takes stage st + 1 + D (clamped to the last)
    auto stage = [&](uint32_t st, int d) __attribute__((always_inline)) {
        const uint32_t buf = st & 1u, k2 = min(st + 1u + (uint32_t)D, nkf - 1u) * BK;
#pragma unroll
        for (int q = 0; q < NA * ST; ++q) {
            __builtin_amdgcn_sched_barrier(0);
            mult(buf, q % NA, HS == 1 ? (uint32_t)q : 2u * (uint32_t)q + wh);
            if constexpr (!DUTY) {
#pragma unroll
                for (int u = 0; u < PA + PB; ++u) {
                    if (u * (NA * ST) / (PA + PB) != q) continue;
                    if (u < PA) {
                        a.store(d, u, SAp + (buf ^ 1u) * SA, lost);
                        a.load(d, u, p.as[3], k2);
                    } else {
                        b.store(d, u - PA, SBp + (buf ^ 1u) * SB, lost);
                        b.load(d, u - PA, p.bs[2], k2);
                    }
                }
#pragma unroll
                for (int m = 0; m < 6 * MI * NJ; ++m) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, MI * NJ == 1 ? 10 : 4, 0);
                }
            }
        }
        if constexpr (DUTY) {
            store(d, buf ^ 1u);
            load(d, st + 1u + (uint32_t)D);
        }
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();
    };
    if (nkf) {
        load(0, 0u);
        if (D == 2) load(1, 1u);
        store(0, 0u);
        load(0, (uint32_t)D);
        __syncthreads();
        uint32_t st = 0;
        if constexpr (D == 1) {
            for (; st < nkf; ++st) stage(st, 0);
        } else {
            for (; st + 2u <= nkf; st += 2u) {
                stage(st, 1);
                stage(st + 1u, 0);
            }
            if (st < nkf) stage(st, 1);
        }
    }
    if (p.K % BK) {
        // (the buffers' last readers finished before a barrier)
        if (!DUTY || !dutyb) {
#pragma unroll
            for (int u = 0; u < PA; ++u) a.load_tail(0, u, p.as[3], nkf * BK, p.K);
        }
        if (!DUTY || dutyb) {
#pragma unroll
            for (int u = 0; u < PB; ++u) b.load_tail(0, u, p.bs[2], nkf * BK, p.K);
        }
        store(0, 0u);
        __syncthreads();
#pragma unroll
        for (int q = 0; q < NA * ST; ++q) mult(0u, q % NA, HS == 1 ? (uint32_t)q : 2u * (uint32_t)q + wh);
        __syncthreads();
    }
    // Even + odd, to acc[0] (HS 2: of the even waves). Beside it a word: whether
    // the tile needs a closer look.
    uint32_t* word = (uint32_t*)(SBp + 2u * SB);
    if (threadIdx.x == 0u) *word = 0u;
    float* red = (float*)vx_bf_lds + wave % (WM * WN) * (MI * NJ * 1024u) + lane;
    if (HS == 2 && wh) {
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j)
#pragma unroll
                for (int v = 0; v < 16; ++v) red[((i * NJ + j) * 16 + v) * 64] = acc[0][i][j][v];
    }
    __syncthreads();
    if ((lost & 0xFFFFu) != 0u) *word = 1u;
    if (!wh) {
        // f: a NaN when an output is not finite; lo: twice the bits of the
        // smallest |output| above 0, less one
        float f = 0.f;
        uint32_t lo = ~0u;
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                if constexpr (HS == 1) acc[0][i][j] += acc[1][i][j];
                else {
#pragma unroll
                    for (int v = 0; v < 16; ++v) acc[0][i][j][v] += red[((i * NJ + j) * 16 + v) * 64];
                }
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    f = __builtin_fmaf(acc[0][i][j][v], 0.f, f);
                    lo = min(lo, (__float_as_uint(acc[0][i][j][v]) << 1) - 1u);
                }
            }
        if (f != 0.f || lo < (0x03800000u << 1) - 1u /* 2^-120 */) *word = 1u;
    }
    __syncthreads();
    const bool look = *word != 0u;
    const uint32_t rt0 = wm * (32u * MI) + 4u * g, ct0 = wn * (32u * NJ) + n;
    float* c0 = C + (int64_t)(m0 + rt0) * p.cs[2] + (int64_t)(n0 + ct0) * p.cs[3];
    if (!look && !wh && m0 + TM <= p.M && n0 + TN <= p.N) {
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int v = 0; v < 16; ++v)
                    vx_epilogue(c0 + (int64_t)(32 * i + 8 * (v >> 2) + (v & 3)) * p.cs[2] + (int64_t)(32 * j) * p.cs[3],
                                acc[0][i][j][v], p.alpha, p.beta);
        return;
    }
    uint32_t *mx = (uint32_t*)vx_bf_lds, *ls = mx + TM + TN;  // of each row of A and column of B, see vx_scan
    if (look) {
        for (uint32_t i = threadIdx.x; i < 2u * (TM + TN); i += NTH) mx[i] = 0u;
        __syncthreads();
        auto all = [](uint32_t) { return true; };
        vx_scan<AM == MODE_K, TM>(A, p.as[2], p.as[3], m0, p.M, p.K, wave, NTH / 64, lane, mx, ls, all);
        vx_scan<BM == MODE_K, TN>(B, p.bs[3], p.bs[2], n0, p.N, p.K, wave, NTH / 64, lane, mx + TM, ls + TM, all);
        __syncthreads();
    }
    if (wh) return;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        const uint32_t ct = ct0 + 32u * j;
#pragma unroll
        for (int i = 0; i < MI; ++i) {
            float* c1 = c0 + (int64_t)(32 * i) * p.cs[2] + (int64_t)(32 * j) * p.cs[3];
            uint32_t again = 0u;  // outputs to form from f32 products
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const uint32_t rt = rt0 + 32u * i + 8u * (v >> 2) + (v & 3);
                if (m0 + rt < p.M && n0 + ct < p.N) {
                    if (!look || !vx_gemm_bf_again(acc[0][i][j][v], p.K, mx[rt], ls[rt] != 0u, mx[TM + ct], ls[TM + ct] != 0u))
                        vx_epilogue(c1 + (int64_t)(8 * (v >> 2) + (v & 3)) * p.cs[2], acc[0][i][j][v], p.alpha, p.beta);
                    else
                        again |= 1u << v;
                }
            }
            if (!__any(again != 0u)) continue;
            f32x16 f;
            vx_f32_tile<AM, BM>(p, A + (int64_t)min(m0 + wm * (32u * MI) + 32u * i + n, p.M - 1u) * p.as[2],
                                B + (int64_t)min(n0 + ct, p.N - 1u) * p.bs[3], g, f);
#pragma unroll
            for (int v = 0; v < 16; ++v)
                if (again >> v & 1u) vx_epilogue(c1 + (int64_t)(8 * (v >> 2) + (v & 3)) * p.cs[2], f[v], p.alpha, p.beta);
        }
    }
}

// 32 x 32 tiles with K split over the 8 waves of a workgroup: for shapes with
// too few outputs to fill the GPU otherwise (a few rows through a wide layer, a
// small output from a long K). Wave w takes the 32-element chunks w, w + 8, ...
// of K straight from memory to registers (no LDS, no barrier in the loop, one
// chunk ahead), and the waves' sums meet in LDS in wave order.
template <int AM, int BM>
__device__ __forceinline__ void vx_gemm_bf_ks(const vx_gemm_args& p) {
    constexpr uint32_t NWV = 8;
    const uint32_t t = threadIdx.x, lane = t & 63u, n = lane & 31u, g = lane >> 5;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const uint32_t nt = p.tiles_m * p.tiles_n;
    const uint32_t bid = vx_xcd_order(blockIdx.x, nt);  // tiles that share columns of B follow each other on one XCD
    const uint32_t m0 = bid % p.tiles_m * 32u, n0 = bid / p.tiles_m * 32u;
    const uint32_t z = blockIdx.z;
    const uint32_t bn = z / p.batch_c, bc = z % p.batch_c;
    const float* A = p.a + bn * p.as[0] + bc * p.as[1];
    const float* B = p.b + bn * p.bs[0] + bc * p.bs[1];
    float* C = p.c + bn * p.cs[0] + bc * p.cs[1];
    const float* pa = A + (int64_t)min(m0 + n, p.M - 1u) * p.as[2];
    const float* pb = B + (int64_t)min(n0 + n, p.N - 1u) * p.bs[3];

    f32x16 acc[2];
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[0][v] = acc[1][v] = 0.f;
    uint32_t lost = 0u;  // see vx_split8_rne
    auto mult = [&](const auto& a, const auto& b, int) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            u32x4 ta[3], tb[3];
            vx_split8_rne(a.r[h], ta, lost);
            vx_split8_rne(b.r[h], tb, lost);
            constexpr int TA[6] = {2, 0, 1, 1, 0, 0}, TB[6] = {0, 2, 1, 0, 1, 0};  // smallest products first
#pragma unroll
            for (int e = 0; e < 6; ++e)
                acc[h] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, ta[TA[e]]),
                                                                 __builtin_bit_cast(bf16x8, tb[TB[e]]), acc[h], 0, 0, 0);
        }
    };
    constexpr bool SO = AM == MODE_X && BM == MODE_X;
    vx_chunks<vx_chunk<AM, 2, 2, SO>, vx_chunk<BM, 2, 2, SO>>(p, pa, pb, g, wave, NWV, mult);
    // red[wave][v][lane], and whether the tile needs a closer look
    float* red = (float*)vx_bf_lds;
    uint32_t* word = (uint32_t*)(red + NWV * 1024u);
    if (t == 0u) *word = 0u;
#pragma unroll
    for (int v = 0; v < 16; ++v) red[wave * 1024u + (uint32_t)v * 64u + lane] = acc[0][v] + acc[1][v];
    __syncthreads();
    float s[2];
#pragma unroll
    for (uint32_t u = 0; u < 2u; ++u) {
        s[u] = red[t + 512u * u];
#pragma unroll
        for (uint32_t w = 1; w < NWV; ++w) s[u] += red[w * 1024u + t + 512u * u];
    }
    if ((lost & 0xFFFFu) != 0u || vx_gemm_bf_odd(s[0]) || vx_gemm_bf_odd(s[1])) *word = 1u;
    __syncthreads();
    const uint32_t rt0 = 8u * (t >> 8) + 4u * (lane >> 5) + (wave & 3u), ct = lane & 31u;  // output u: row rt0 + 16 u, column ct
    auto write = [&] {
#pragma unroll
        for (uint32_t u = 0; u < 2u; ++u) {
            const uint32_t row = m0 + rt0 + 16u * u, col = n0 + ct;
            if (row < p.M && col < p.N) vx_epilogue(C + (int64_t)row * p.cs[2] + (int64_t)col * p.cs[3], s[u], p.alpha, p.beta);
        }
    };
    // (the usual end first and by itself: with the look between, 512^3 took 7.4
    // us instead of 7.2, 600 x 600 x 1000 17.6 instead of 17.2)
    if (__builtin_expect(*word == 0u, 1)) {
        write();
        return;
    }
    uint32_t *mx = (uint32_t*)vx_bf_lds, *ls = mx + 64;  // of each row of A and column of B, see vx_scan
    if (t < 128u) mx[t] = 0u;
    __syncthreads();
    auto all = [](uint32_t) { return true; };
    vx_scan<AM == MODE_K, 32>(A, p.as[2], p.as[3], m0, p.M, p.K, wave, NWV, lane, mx, ls, all);
    vx_scan<BM == MODE_K, 32>(B, p.bs[3], p.bs[2], n0, p.N, p.K, wave, NWV, lane, mx + 32, ls + 32, all);
    __syncthreads();
    bool again[2];  // outputs to form from f32 products
#pragma unroll
    for (uint32_t u = 0; u < 2u; ++u)
        again[u] = vx_gemm_bf_again(s[u], p.K, mx[rt0 + 16u * u], ls[rt0 + 16u * u] != 0u, mx[32u + ct], ls[32u + ct] != 0u);
    if (again[0] || again[1]) *word = 2u;
    __syncthreads();
    if (*word == 2u) {
        if (wave < 4u) {  // 16 x 16 outputs each
            const uint32_t r0 = 16u * (wave >> 1), c0 = 16u * (wave & 1u), n16 = lane & 15u, g4 = lane >> 4;
            f32x4 f;
            vx_f32_tile<AM, BM>(p, A + (int64_t)min(m0 + r0 + n16, p.M - 1u) * p.as[2],
                                B + (int64_t)min(n0 + c0 + n16, p.N - 1u) * p.bs[3], g4, f);
#pragma unroll
            for (uint32_t v = 0; v < 4u; ++v) red[(r0 + 4u * g4 + v) * 32u + c0 + n16] = f[v];
        }
        __syncthreads();
#pragma unroll
        for (uint32_t u = 0; u < 2u; ++u)
            if (again[u]) s[u] = red[(rt0 + 16u * u) * 32u + ct];
    }
    write();
}

// 16 x 16 tiles on 16 x 16 x 32 products, K split over the 8 waves as above.
// Against 32 x 32 tiles, four times the workgroups, and few enough registers
// for two on a CU: the shapes with about as many 32 x 32 tiles as CUs,
// or fewer, ran at the pace of one workgroup on some of the CUs (or of a second
// round on a few). Each operand is read and split once per 16 outputs of the
// other, so it loses where 32 x 32 tiles fill the card. Graph-replayed, us, 32 x
// 32 / 16 x 16: 8 x 11008 x 4096 B [N, K] 49.4 / 41.0, 16 x 4096 x 4096 24.2 /
// 17.3, 23 x 1989 x 5973 34.6 / 22.4, 96 x 64 x 3776 23.4 / 11.4, 256^3 4.8 / 3.5;
// but 30 x 16384 x 2048 38.7 / 72.4, 512^3 7.3 / 10.9. Tried, when the first of
// these took 44.1 us: 4 or 16 waves (44.4, 47.2), three or four chunks ahead (no
// gain), 32 x 16 tiles (46.3; 31 x 4096 x 4096 25.6 against 33.7 and 34.5, the
// only size where they won).
template <int AM, int BM>
__device__ __forceinline__ void vx_gemm_bf_k16(const vx_gemm_args& p) {
    constexpr uint32_t NWV = 8;
    const uint32_t t = threadIdx.x, lane = t & 63u, n = lane & 15u, g = lane >> 4;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const uint32_t bid = vx_xcd_order(blockIdx.x, p.tiles_m * p.tiles_n);  // tiles that share columns of B on one XCD
    const uint32_t m0 = bid % p.tiles_m * 16u, n0 = bid / p.tiles_m * 16u;
    const uint32_t z = blockIdx.z;
    const uint32_t bn = z / p.batch_c, bc = z % p.batch_c;
    const float* A = p.a + bn * p.as[0] + bc * p.as[1];
    const float* B = p.b + bn * p.bs[0] + bc * p.bs[1];
    float* C = p.c + bn * p.cs[0] + bc * p.cs[1];
    const float* pa = A + (int64_t)min(m0 + n, p.M - 1u) * p.as[2];
    const float* pb = B + (int64_t)min(n0 + n, p.N - 1u) * p.bs[3];

    f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};  // even and odd chunks
    uint32_t lost = 0u;  // see vx_split8_rne
    auto mult = [&](const auto& a, const auto& b, int par) {
        u32x4 ta[3], tb[3];
        vx_split8_rne(a.r[0], ta, lost);
        vx_split8_rne(b.r[0], tb, lost);
        constexpr int TA[6] = {2, 0, 1, 1, 0, 0}, TB[6] = {0, 2, 1, 0, 1, 0};  // smallest products first
#pragma unroll
        for (int e = 0; e < 6; ++e)
            acc[par] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, ta[TA[e]]),
                                                               __builtin_bit_cast(bf16x8, tb[TB[e]]), acc[par], 0, 0, 0);
    };
    constexpr bool SO = AM == MODE_X && BM == MODE_X;
    vx_chunks<vx_chunk<AM, 1, 4, SO>, vx_chunk<BM, 1, 4, SO>>(p, pa, pb, g, wave, NWV, mult);
    // red[wave][v][lane], and whether the tile needs a closer look
    float* red = (float*)vx_bf_lds;
    uint32_t* word = (uint32_t*)(red + NWV * 256u);
    if (t == 0u) *word = 0u;
#pragma unroll
    for (int v = 0; v < 4; ++v) red[wave * 256u + (uint32_t)v * 64u + lane] = acc[0][v] + acc[1][v];
    __syncthreads();
    float s = red[t & 255u];
#pragma unroll
    for (uint32_t w = 1; w < NWV; ++w) s += red[w * 256u + (t & 255u)];
    if ((lost & 0xFFFFu) != 0u || vx_gemm_bf_odd(s)) *word = 1u;
    __syncthreads();
    const uint32_t rt = 4u * (lane >> 4) + (wave & 3u), ct = lane & 15u;  // of the first four waves' outputs
    auto write = [&] {
        const uint32_t row = m0 + rt, col = n0 + ct;
        if (t < 256u && row < p.M && col < p.N) vx_epilogue(C + (int64_t)row * p.cs[2] + (int64_t)col * p.cs[3], s, p.alpha, p.beta);
    };
    if (__builtin_expect(*word == 0u, 1)) {  // (as in vx_gemm_bf_ks)
        write();
        return;
    }
    uint32_t *mx = (uint32_t*)vx_bf_lds, *ls = mx + 32;  // of each row of A and column of B, see vx_scan
    if (t < 64u) mx[t] = 0u;
    __syncthreads();
    auto all = [](uint32_t) { return true; };
    vx_scan<AM == MODE_K, 16>(A, p.as[2], p.as[3], m0, p.M, p.K, wave, NWV, lane, mx, ls, all);
    vx_scan<BM == MODE_K, 16>(B, p.bs[3], p.bs[2], n0, p.N, p.K, wave, NWV, lane, mx + 16, ls + 16, all);
    __syncthreads();
    const bool again = vx_gemm_bf_again(s, p.K, mx[rt], ls[rt] != 0u, mx[16u + ct], ls[16u + ct] != 0u);
    if (again) *word = 2u;
    __syncthreads();
    if (*word == 2u) {
        if (wave == 0u) {
            f32x4 f;
            vx_f32_tile<AM, BM>(p, pa, pb, g, f);
#pragma unroll
            for (uint32_t v = 0; v < 4u; ++v) red[v * 64u + lane] = f[v];
        }
        __syncthreads();
        if (again) s = red[t & 255u];
    }
    write();
}

// 256 x 128 tiles (8 waves of 64 x 64), 128 x 128 (2 x 4 waves of 64 x 64) and
// 64 x 64 (2 x 4 waves of 32 x 32): _s two workgroups per CU, _s2 one, with half
// the barriers.
#define VX_GEMM_BF1(AM, BM, NAME, WPE, ...)                                                              \
    extern "C" __global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, WPE)))            \
    void vx_gemm_bf_##NAME(vx_gemm_args p) {                                                             \
        vx_gemm_bf<AM, BM, __VA_ARGS__>(p);                                                              \
    }
#define VX_GEMM_BF(AM, BM, NAME)                            \
    VX_GEMM_BF1(AM, BM, NAME##_w, 2, 256, 128, 4, 2, 1, 1)  \
    VX_GEMM_BF1(AM, BM, NAME##_n, 2, 128, 128, 2, 2, 2, 1)  \
    VX_GEMM_BF1(AM, BM, NAME##_s2, 4, 64, 64, 2, 2, 2, 2)   \
    VX_GEMM_BF1(AM, BM, NAME##_s, 6, 64, 64, 2, 2, 2, 1)    \
    extern "C" __global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 3)))              \
    void vx_gemm_bf_##NAME##_ks(vx_gemm_args p) {                                                        \
        vx_gemm_bf_ks<AM, BM>(p);                                                                        \
    }                                                                                                    \
    extern "C" __global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(4, 6)))              \
    void vx_gemm_bf_##NAME##_k16(vx_gemm_args p) {                                                       \
        vx_gemm_bf_k16<AM, BM>(p);                                                                       \
    }
VX_GEMM_BF(MODE_K, MODE_X, kx)
VX_GEMM_BF(MODE_K, MODE_K, kk)
VX_GEMM_BF(MODE_X, MODE_X, xx)
VX_GEMM_BF(MODE_X, MODE_K, xk)
