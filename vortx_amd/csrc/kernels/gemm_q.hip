// gemm_q.hip — products of a block-quantized W with many columns of x on the
// bf16 matrix cores (no reference counterpart): y[m, b] = sum_k W[m, k] x[k, b].
//
// Every weight of a block is d times a whole number of at most 8 bits, which
// bf16 holds exactly, and x is split into NT bf16 terms (vx_bf16.hpp): three
// hold a float exactly (x kept in f32), two to 2^-16 of its magnitude (the
// routes that may round x; the int8 split of the narrow batches is off by up
// to 2^-16 of the block's largest |x|). So each 32-block's sum is formed from
// exact products in f32 by chained v_mfma_f32_16x16x32_bf16 (one per term,
// smallest first), and the block's scale multiplies it once.
//
// MFMA layout (one 32-block): A (16 x 32) is x, row n a column of x; B (32 x
// 16) is W, column n a row of W; lane (n, g) of either holds positions
// 8g..8g+7, elements 4g..4g+3 and 16+4g..16+4g+3 of the block (the order of a
// Q4_0 block's nibbles, as in the vx_xq levels); D: lane (n, g) holds W row n
// and columns 4g..4g+3 of x, so a block's scale is one value per lane.
//
// The offset terms (-8 d S for Q4_0's nibbles, -dmin m S for Q4_K, S the
// block's sum of x; smaller ones with three terms, see vx_nib_bf16) are a contraction over blocks: v_mfma_f32_16x16x4_f32
// adds them to the accumulators, four blocks at a time (even, then odd
// blocks of an item: lane row g supplies blocks 2g and 2g + 1, the ones
// whose scales its own 64-weight unit holds).
//
// Measured per call (graph-replayed, same box, against the routes before: the
// int8 split with a launch per 16 columns; f32 vector kernels): two terms,
// 512 columns: Q4_K 14336 x 4096 408 -> 143 us, Q4_0 11008 x 4096 309 -> 141,
// Q8_0 417 -> 167; three terms: Q8_0 4096 x 4096, 67 columns 193 -> 29 us,
// Q4_K 11008 x 4096, 512 columns 2771 -> 195. What bounds the 256 x 128 tiles:
// MFMA 40 % of the cycles and the vector work that does not fit under it
// (scaling 64, decoding ~30, conversion ~30 operations per wave and block),
// and the barrier of each step; the K-split kernels: vector work (each wave
// converts its own x).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../vx_kargs.h"
#include "vx_bf16.hpp"
#include "vx_dpp.hpp"
#include "vx_quant.hpp"

// One item (256 weights of a row, 8 blocks) as this lane keeps it: packed
// bytes in the MFMA layout, decoded to bf16 block by block.
template <int QT>
struct vx_wpack {
    static constexpr bool OFFSET = QT != VX_Q8_0;
    static constexpr int NQ = QT == VX_Q8_0 ? 16 : 8;
    uint32_t q[NQ];      // Q4_0: qs dword g of block b; Q8_0: qs dwords g and 4 + g of block b at 2b, 2b + 1; Q4_K: of chunk k at 2k, 2k + 1
    uint32_t sc[4];      // Q4_0, Q8_0: d of blocks 2k and 2k + 1 (f16 pairs); Q4_K: bytes sc, m of sub-blocks 2k and 2k + 1
    float d;             // Q4_K: d
    float off0, off1;    // OFFSET: coefficient of S of blocks 2g and 2g + 1
};

template <int QT, bool CEN>
__device__ __forceinline__ void vx_wpack_make(const uint32_t (&r)[vx_unit<QT>::NW], uint32_t g, vx_wpack<QT>& w) {
    if constexpr (QT == VX_Q4_0) {
        uint32_t e0 = __builtin_amdgcn_alignbit(r[1], r[0], 16), e1 = __builtin_amdgcn_alignbit(r[2], r[1], 16);
        uint32_t e2 = __builtin_amdgcn_alignbit(r[3], r[2], 16), e3 = __builtin_amdgcn_alignbit(r[4], r[3], 16);
        uint32_t o0 = r[5], o1 = r[6], o2 = r[7], o3 = r[8];
        vx_t4(e0, e1, e2, e3);
        vx_t4(o0, o1, o2, o3);
        w.q[0] = e0; w.q[1] = o0; w.q[2] = e1; w.q[3] = o1;
        w.q[4] = e2; w.q[5] = o2; w.q[6] = e3; w.q[7] = o3;
        vx_gather4((r[0] & 0xFFFFu) | (r[4] & 0xFFFF0000u), w.sc);
        w.off0 = (CEN ? -0.5f : -8.f) * vx_f16_to_f32(r[0]);
        w.off1 = (CEN ? -0.5f : -8.f) * vx_f16_to_f32(r[4] >> 16);
    } else if constexpr (QT == VX_Q8_0) {
        uint32_t a[8], b[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            a[k] = __builtin_amdgcn_alignbit(r[k + 1], r[k], 16);
            b[k] = r[9 + k];
        }
        vx_t4(a[0], a[1], a[2], a[3]);
        vx_t4(a[4], a[5], a[6], a[7]);
        vx_t4(b[0], b[1], b[2], b[3]);
        vx_t4(b[4], b[5], b[6], b[7]);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            w.q[4 * k] = a[k];
            w.q[4 * k + 1] = a[4 + k];
            w.q[4 * k + 2] = b[k];
            w.q[4 * k + 3] = b[4 + k];
        }
        vx_gather4((r[0] & 0xFFFFu) | (r[8] & 0xFFFF0000u), w.sc);
    } else {
        uint32_t c0 = r[4], c1 = r[5], c2 = r[6], c3 = r[7];
        uint32_t c4 = r[8], c5 = r[9], c6 = r[10], c7 = r[11];
        vx_t4(c0, c1, c2, c3);
        vx_t4(c4, c5, c6, c7);
        w.q[0] = c0; w.q[1] = c4; w.q[2] = c1; w.q[3] = c5;
        w.q[4] = c2; w.q[5] = c6; w.q[6] = c3; w.q[7] = c7;
        w.d = vx_f16_to_f32(r[0]);
        const float dmin = vx_f16_to_f32(r[0] >> 16);
        uint32_t sc0, m0, sc1, m1;
        vx_q4k_scales(r[1], r[2], r[3], g, sc0, m0, sc1, m1);
        vx_gather4(sc0 | (sc1 << 16), w.sc);
        w.off0 = -(dmin * (float)m0);
        w.off1 = -(dmin * (float)m1);
        if constexpr (CEN) {
            w.off0 = __builtin_fmaf(7.5f * w.d, (float)sc0, w.off0);
            w.off1 = __builtin_fmaf(7.5f * w.d, (float)sc1, w.off1);
        }
    }
}

// Bytes 0..3 of v, each q = 0..15, as bf16: read as e4m3 a byte q is q 2^-9
// exactly, and v_cvt_scalef32_pk_bf16_fp8 multiplies by 2^9. CEN: q - 7.5
// instead, from the bytes |2q - 15| with the sign in bit 7: block sums are
// then as small as the weights' own, and the offset term with them (-d S / 2
// instead of -8 d S for Q4_0), so less is rounded away when the two cancel:
// against 64 bits at K = 4096 4.2e-7 -> 1.2e-7 (Q4_0), where the f32 vector
// kernels are 2.2e-7 off.
template <bool CEN>
__device__ __forceinline__ void vx_nib_bf16(uint32_t v, uint32_t& lo, uint32_t& hi) {
    if constexpr (CEN) {
        const uint32_t s = ~v & 0x08080808u;  // q < 8
        v = ((((v & 0x07070707u) ^ (s - (s >> 3))) << 1) | 0x01010101u) | (s << 4);
    }
    lo = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(v, CEN ? 256.0f : 512.0f, false));
    hi = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(v, CEN ? 256.0f : 512.0f, true));
}
// Bytes 0..3 of v, signed, as bf16.
__device__ __forceinline__ void vx_i8_bf16(uint32_t v, uint32_t& lo, uint32_t& hi) {
    lo = vx_pk_bf16((float)(int8_t)(v & 0xFFu), (float)(int8_t)((v >> 8) & 0xFFu));
    hi = vx_pk_bf16((float)(int8_t)((v >> 16) & 0xFFu), (float)(int8_t)(v >> 24));
}

// B operand of block b (a constant after unrolling) and the block's scale.
template <int QT, bool CEN>
__device__ __forceinline__ bf16x8 vx_wpack_block(const vx_wpack<QT>& w, int b, float& scale) {
    u32x4 o;
    uint32_t lo, hi;
    if constexpr (QT == VX_Q4_0) {
        vx_nib_bf16<CEN>((w.q[b]) & 0x0F0F0F0Fu, lo, hi);
        o.x = lo; o.y = hi;
        vx_nib_bf16<CEN>((w.q[b] >> 4) & 0x0F0F0F0Fu, lo, hi);
        o.z = lo; o.w = hi;
        scale = vx_f16_to_f32((b & 1) ? w.sc[b >> 1] >> 16 : w.sc[b >> 1]);
    } else if constexpr (QT == VX_Q8_0) {
        vx_i8_bf16(w.q[2 * b], lo, hi);
        o.x = lo; o.y = hi;
        vx_i8_bf16(w.q[2 * b + 1], lo, hi);
        o.z = lo; o.w = hi;
        scale = vx_f16_to_f32((b & 1) ? w.sc[b >> 1] >> 16 : w.sc[b >> 1]);
    } else {
        const uint32_t c0 = w.q[2 * (b >> 1)], c1 = w.q[2 * (b >> 1) + 1];
        vx_nib_bf16<CEN>(((b & 1) ? c0 >> 4 : c0) & 0x0F0F0F0Fu, lo, hi);
        o.x = lo; o.y = hi;
        vx_nib_bf16<CEN>(((b & 1) ? c1 >> 4 : c1) & 0x0F0F0F0Fu, lo, hi);
        o.z = lo; o.w = hi;
        scale = w.d * (float)((b & 1) ? w.sc[b >> 1] >> 16 : w.sc[b >> 1] & 0xFFFFu);
    }
    return __builtin_bit_cast(bf16x8, o);
}

// This lane's 8 elements of a block, p at its element 4g: elements 4g..4g+3
// and 16+4g..16+4g+3. XV: stride 1 and 16-byte aligned columns.
template <bool XV>
__device__ __forceinline__ void vx_x8(const float* p, int64_t xs_k, float (&v)[8]) {
    if constexpr (XV) {
        const f32x4 u = *(const f32x4*)p, w = *(const f32x4*)(p + 16);
        v[0] = u.x; v[1] = u.y; v[2] = u.z; v[3] = u.w;
        v[4] = w.x; v[5] = w.y; v[6] = w.z; v[7] = w.w;
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            v[i] = p[(int64_t)i * xs_k];
            v[4 + i] = p[(int64_t)(16 + i) * xs_k];
        }
    }
}

extern __shared__ __align__(16) uint8_t vx_gq_lds[];

// Weights 8g..8g+7 of 32-block kb of a row as they are (load), and as floats.
typedef uint32_t u32_a1 __attribute__((aligned(1)));
typedef uint16_t u16_a1 __attribute__((aligned(1)));
template <int QT>
struct vx_w8 {
    uint32_t q0, q1, h, s1, s2, s3;
    __device__ __forceinline__ void load(const uint8_t* row, uint32_t kb, uint32_t g) {
        const uint8_t* p = row + (QT == VX_Q4_0 ? 18u * kb : QT == VX_Q8_0 ? 34u * kb : 144u * (kb >> 3));
        const uint8_t* q = p + (QT == VX_Q4_0 ? 2u + 8u * (g & 1u) : QT == VX_Q8_0 ? 2u + 8u * g : 16u + 32u * ((kb & 7u) >> 1) + 8u * g);
        q0 = *(const u32_a1*)q;
        q1 = *(const u32_a1*)(q + 4);
        if constexpr (QT == VX_Q4_K) {
            h = *(const u32_a1*)p;
            s1 = *(const u32_a1*)(p + 4);
            s2 = *(const u32_a1*)(p + 8);
            s3 = *(const u32_a1*)(p + 12);
        } else {
            h = *(const u16_a1*)p;
        }
    }
    __device__ __forceinline__ void decode(uint32_t kb, uint32_t g, float (&o)[8]) const {
        const float d = vx_f16_to_f32(h);
        if constexpr (QT == VX_Q8_0) {
#pragma unroll
            for (int e = 0; e < 8; ++e) o[e] = d * (float)(int8_t)(((e < 4 ? q0 : q1) >> (8 * (e & 3))) & 0xFFu);
        } else {
            const uint32_t sh = 4u * (QT == VX_Q4_0 ? g >> 1 : kb & 1u);
            uint32_t sc0, m0, sc1, m1;
            if constexpr (QT == VX_Q4_K) vx_q4k_scales(s1, s2, s3, (kb & 7u) >> 1, sc0, m0, sc1, m1);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const uint32_t n = ((e < 4 ? q0 : q1) >> (8u * (e & 3) + sh)) & 15u;
                if constexpr (QT == VX_Q4_0) o[e] = (float)((int)n - 8) * d;
                else o[e] = __fsub_rn(__fmul_rn(d * (float)((kb & 1u) ? sc1 : sc0), (float)n), vx_f16_to_f32(h >> 16) * (float)((kb & 1u) ? m1 : m0));
            }
        }
    }
};

// Outputs that are not finite (the terms of an infinite x hold a NaN, where the
// f32 products give an infinity; a block's sum of whole numbers times x may pass
// the largest float before the scale brings it back) or, with x exact, below 2^-56
// (three terms of an x below 2^-110 may miss bits, see vx_split8) are looked at again, in y, with the columns
// of x that they came from. Where the column holds a NaN, so does the output. Any
// other that is not finite, or whose column holds an x with missing bits, is
// formed again from f32 products, 16 x 16 CG outputs of a wave on v_mfma_f32_16x16x4f32 (lane (n, g) of either operand holds elements
// 8g..8g+7 of a block; U blocks requested ahead of their products). Above 2^-56
// the missing bits, below 2^-133 of each x, are less than the roundings: with |w|
// < 2^26 and K <= 2^28 they add up to 2^-79 at most, 2^-23 of the output.
// Bound by its requests (16 rows of x and of W an instruction). Q4_0 2300 x 2048,
// 1500 columns, three terms, us: 106; with a NaN in every column 153 and with zeros
// alone 141 (the look), with an infinity in every column 600 (each of these
// outputs in one lane: 2275).
template <int NT>
__device__ __forceinline__ bool vx_gemm_q_odd(float y) {
    const float v = __builtin_fabsf(y);
    return !((NT == 2 || v >= 0x1p-56f) && v < __builtin_inff());
}

// odd[c]: whether column c of the workgroup holds such an output (in LDS, behind
// what the look overwrites).
template <int QT, int NT, bool XV, uint32_t ROWS, uint32_t COLS, uint32_t NWV>
__device__ __forceinline__ void vx_gemm_q_look(const vx_gemv_args& a, uint32_t row0, uint32_t col0, const uint32_t* odd) {
    constexpr uint32_t CG = COLS >= 64u ? 4u : 1u, U = CG == 1u ? 4u : 2u;
    const uint32_t t = threadIdx.x, lane = t & 63u, n = lane & 15u, g = lane >> 4;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(t >> 6);
    uint32_t *mx = (uint32_t*)vx_gq_lds, *ls = mx + COLS;  // of each column
    __syncthreads();
    if (!__any(odd[lane % COLS] != 0u || (COLS > 64u && odd[lane + 64u] != 0u))) return;  // (uniform over the workgroup)
    for (uint32_t i = t; i < 2u * COLS; i += 64u * NWV) mx[i] = 0u;
    __syncthreads();
    vx_scan<XV, COLS>(a.x, a.xs_b, a.xs_k, col0, a.B, a.K, wave, NWV, lane, mx, ls,
                      [&](uint32_t c) { return odd[c] != 0u; });
    __syncthreads();
    const uint32_t nblk = a.K / 32u;
    for (uint32_t u = wave; u < ROWS / 16u * (COLS / (16u * CG)); u += NWV) {
        const uint32_t r0 = row0 + u % (ROWS / 16u) * 16u, c0 = u / (ROWS / 16u) * (16u * CG);
        if (r0 >= a.M || col0 + c0 >= a.B) continue;
        float* y = a.y + (int64_t)min(r0 + n, a.M - 1u) * a.ys_m;
        float v[4u * CG];  // columns 4g..4g+3 of each subtile (past the last: that one again)
#pragma unroll
        for (uint32_t e = 0; e < 4u * CG; ++e)
            v[e] = y[(int64_t)min(col0 + c0 + 4u * g + 16u * (e >> 2) + (e & 3u), a.B - 1u) * a.ys_b];
        uint32_t again = 0u;
#pragma unroll
        for (uint32_t e = 0; e < 4u * CG; ++e) {
            const uint32_t cc = c0 + 4u * g + 16u * (e >> 2) + (e & 3u);
            const bool in = (r0 + n < a.M) & (col0 + cc < a.B) & (mx[cc] <= 0x7F800000u);
            again |= (uint32_t)(in & vx_gemm_q_odd<NT>(v[e]) & ((ls[cc] != 0u) | !(__builtin_fabsf(v[e]) < __builtin_inff()))) << e;
        }
        if (!__any(again != 0u)) continue;
        const uint8_t* row = a.w + (uint64_t)min(r0 + n, a.M - 1u) * a.row_stride;
        const float* xp[CG];
#pragma unroll
        for (uint32_t c = 0; c < CG; ++c)
            xp[c] = a.x + (int64_t)min(col0 + c0 + 16u * c + n, a.B - 1u) * a.xs_b + (int64_t)(8u * g) * (XV ? 1 : a.xs_k);
        f32x4 acc[CG];
#pragma unroll
        for (uint32_t c = 0; c < CG; ++c) acc[c] = f32x4{0.f, 0.f, 0.f, 0.f};
        for (uint32_t kb = 0; kb < nblk; kb += U) {
            vx_w8<QT> w[U];
            float xv[U][CG][8];
#pragma unroll
            for (uint32_t v = 0; v < U; ++v) {
                const uint32_t k = min(kb + v, nblk - 1u);
                w[v].load(row, k, g);
#pragma unroll
                for (uint32_t c = 0; c < CG; ++c) {
                    const float* p = xp[c] + (int64_t)(32u * k) * (XV ? 1 : a.xs_k);
                    if constexpr (XV) {
                        *(f32x4*)&xv[v][c][0] = *(const f32x4*)p;
                        *(f32x4*)&xv[v][c][4] = *(const f32x4*)(p + 4);
                    } else {
#pragma unroll
                        for (int i = 0; i < 8; ++i) xv[v][c][i] = p[(int64_t)i * a.xs_k];
                    }
                }
            }
            __builtin_amdgcn_sched_barrier(0);  // (or the compiler moves each load to where it is used)
#pragma unroll
            for (uint32_t v = 0; v < U; ++v) {
                if (kb + v >= nblk) break;
                float wv[8];
                w[v].decode(kb + v, g, wv);
#pragma unroll
                for (int i = 0; i < 8; ++i)
#pragma unroll
                    for (uint32_t c = 0; c < CG; ++c) acc[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(xv[v][c][i], wv[i], acc[c], 0, 0, 0);
            }
        }
#pragma unroll
        for (uint32_t e = 0; e < 4u * CG; ++e)
            if (again >> e & 1u) y[(int64_t)(col0 + c0 + 4u * g + 16u * (e >> 2) + (e & 3u)) * a.ys_b] = acc[e >> 2][e & 3u];
    }
}

// K split over the waves of a workgroup: 16 WR rows x 16 CT columns per
// workgroup, wave w takes the items w, w + NW, ... and reads its x itself.
template <int QT, int NT, int WR, int CT, int NWV, bool XV>
__device__ __forceinline__ void vx_gemm_q_ks(const vx_gemv_args& a) {
    constexpr int NW = vx_unit<QT>::NW;
    const uint32_t t = threadIdx.x, lane = t & 63u, n = lane & 15u, g = lane >> 4;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(t >> 6);
    // workgroups that share rows of W follow each other on one XCD; where there
    // are more columns than rows, those that share columns of x (Q4_0 4100 x
    // 4096 x 100, 1 XCD's tiles in a run also where their number is no multiple
    // of 8: 34.0 -> 31.2 us; Q8_0 335 x 11456 x 330 36.1 -> 34.1; 339 x 5568 x
    // 318 rows of W first 20.1, columns of x first 17.3)
    const uint32_t tn = (a.B + 16u * CT - 1u) / (16u * CT), nt = gridDim.x, tm = nt / tn;
    const uint32_t bid = vx_xcd_order(blockIdx.x, nt);
    const uint32_t row0 = (tn > tm ? bid % tm : bid / tn) * (16u * WR), col0 = (tn > tm ? bid / tm : bid % tn) * (16u * CT);
    const uint32_t nblk = a.K / 32u, ipr = (nblk + 7u) >> 3;
    const uint8_t* wrow[WR];
#pragma unroll
    for (int i = 0; i < WR; ++i) wrow[i] = a.w + (uint64_t)min(row0 + 16u * i + n, a.M - 1u) * a.row_stride;
    const float* xp[CT];  // element 4g of block 0
#pragma unroll
    for (int c = 0; c < CT; ++c)
        xp[c] = a.x + (int64_t)min(col0 + 16u * c + n, a.B - 1u) * a.xs_b + (int64_t)(4u * g) * (XV ? 1 : a.xs_k);
    const int64_t xblk = XV ? 32 : 32 * a.xs_k;
    f32x4 acc[WR][CT];
#pragma unroll
    for (int i = 0; i < WR; ++i)
#pragma unroll
        for (int c = 0; c < CT; ++c) acc[i][c] = f32x4{0.f, 0.f, 0.f, 0.f};

    uint32_t raw[WR][NW];
    auto wload = [&](uint32_t item) {
#pragma unroll
        for (int i = 0; i < WR; ++i) vx_load_unit<QT>(wrow[i], min(4u * item + g, a.nunits - 1u), raw[i]);
    };
    if (wave < ipr) wload(wave);
    for (uint32_t item = wave; item < ipr; item += NWV) {
        const uint32_t nb = min(nblk - 8u * item, 8u);  // even: K is a multiple of 64
        vx_wpack<QT> w[WR];
#pragma unroll
        for (int i = 0; i < WR; ++i) {
            vx_wpack_make<QT, NT == 3>(raw[i], g, w[i]);
            // a unit past K repeats the last one: its offset terms count nothing
            if (vx_wpack<QT>::OFFSET && 2u * g >= nb) w[i].off0 = w[i].off1 = 0.f;
        }
        if (item + NWV < ipr) wload(item + NWV);
        float s0[CT], s1[CT];  // S of blocks 2g and 2g + 1 of column n
        float xv[2][CT][8];
#pragma unroll
        for (int c = 0; c < CT; ++c) {
            s0[c] = s1[c] = 0.f;
            vx_x8<XV>(xp[c] + xblk * (int64_t)(8u * item), a.xs_k, xv[0][c]);
        }
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            if ((uint32_t)b >= nb) break;
            if (b < 7) {
#pragma unroll
                for (int c = 0; c < CT; ++c) vx_x8<XV>(xp[c] + xblk * (int64_t)min(8u * item + b + 1u, nblk - 1u), a.xs_k, xv[(b + 1) & 1][c]);
            }
            bf16x8 wb[WR];
            float sc[WR];
#pragma unroll
            for (int i = 0; i < WR; ++i) wb[i] = vx_wpack_block<QT, NT == 3>(w[i], b, sc[i]);
#pragma unroll
            for (int c = 0; c < CT; ++c) {
                const float (&v)[8] = xv[b & 1][c];
                u32x4 xt[NT];
                vx_split8<NT>(v, xt);
                if constexpr (vx_wpack<QT>::OFFSET) {
                    const float s = vx_sum_rows4(((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7])));
                    if ((b & 1) == 0) s0[c] = g == (uint32_t)(b >> 1) ? s : s0[c];
                    else s1[c] = g == (uint32_t)(b >> 1) ? s : s1[c];
                }
#pragma unroll
                for (int i = 0; i < WR; ++i) {
                    f32x4 d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int k = NT - 1; k >= 0; --k)
                        d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, xt[k]), wb[i], d, 0, 0, 0);
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[i][c][e] = __builtin_fmaf(sc[i], d[e], acc[i][c][e]);
                }
            }
        }
        if constexpr (vx_wpack<QT>::OFFSET) {
#pragma unroll
            for (int c = 0; c < CT; ++c)
#pragma unroll
                for (int i = 0; i < WR; ++i) {
                    acc[i][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(s0[c], w[i].off0, acc[i][c], 0, 0, 0);
                    acc[i][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(s1[c], w[i].off1, acc[i][c], 0, 0, 0);
                }
        }
    }
    // red[wave][tile][e][lane]: the waves' sums in wave order
    float* red = (float*)vx_gq_lds;
    constexpr uint32_t PW = WR * CT * 256u;
    uint32_t* odd = (uint32_t*)(red + PW * NWV);  // [16 CT], see vx_gemm_q_look
    if (t < 16u * CT) odd[t] = 0u;
#pragma unroll
    for (int i = 0; i < WR; ++i)
#pragma unroll
        for (int c = 0; c < CT; ++c)
#pragma unroll
            for (int e = 0; e < 4; ++e) red[wave * PW + (uint32_t)((i * CT + c) * 4 + e) * 64u + lane] = acc[i][c][e];
    __syncthreads();
    for (uint32_t o = t; o < PW; o += 64u * NWV) {
        float s = red[o];
#pragma unroll
        for (int k = 1; k < NWV; ++k) s += red[(uint32_t)k * PW + o];
        const uint32_t l = o & 63u, e = (o >> 6) & 3u, tile = o >> 8;
        const uint32_t row = row0 + 16u * (tile / CT) + (l & 15u), cc = col0 + 16u * (tile % CT) + 4u * (l >> 4) + e;
        if (row < a.M && cc < a.B) a.y[(int64_t)row * a.ys_m + (int64_t)cc * a.ys_b] = s;
        if (vx_gemm_q_odd<NT>(s)) odd[cc - col0] = 1u;
    }
    vx_gemm_q_look<QT, NT, XV, 16u * WR, 16u * CT, NWV>(a, row0, col0, odd);
}

// Tiles of 64 WM rows x 64 WN columns on v_mfma_f32_32x32x16_bf16; wave (wm,
// wn) owns 64 x 64 of it. Per 32-block step the workgroup converts its columns
// of x once and shares the terms through LDS (double-buffered, one barrier per
// step); W's rows of an item (256 weights) are copied to LDS as they are, from
// where each lane reads its own dwords of a block (the rows are 144 or 272
// bytes apart, so 16 rows of such a read fall into different banks).
//
// Layout (half h = 0, 1 of a block): lane (n, g) of A (x, column n) and of B
// (W, row n) holds position group p = 2h + g: elements 4p..4p+3 and
// 16+4p..16+4p+3. D: lane (n, g) holds W row n and columns 8 (v / 4) + 4 g +
// v % 4 of x in register v.
//
// Why 32 x 32: measured with 2 waves per SIMD, vector operations add their
// full issue time (2.7 cycles) to a stream of 16x16x32 MFMAs, but up to 5 per
// 32x32x16 MFMA are free (34 cycles each way).
template <bool V> struct vx_bool { static constexpr bool value = V; };
template <int QT> struct vx_gq_item { static constexpr uint32_t BYTES = QT == VX_Q8_0 ? 272u : 144u; };
typedef float f32x16 __attribute__((ext_vector_type(16)));

template <int QT, int NT, int WM, int WN, bool XV>
__device__ __forceinline__ void vx_gemm_q_tile(const vx_gemv_args& a) {
    constexpr int NWV = WM * WN, CT = 2 * WN;  // CT: column tiles of 32
    constexpr uint32_t NTH = 64u * NWV, ROWS = 64u * WM, COLS = 32u * CT, IB = vx_gq_item<QT>::BYTES;
    constexpr bool OFF = QT != VX_Q8_0, CEN = NT == 3;
    static_assert(2 * CT % NWV == 0, "whole pieces");
    constexpr int UPT = 2 * CT / NWV;            // (column tile, half) pieces a wave converts per step
    constexpr uint32_t NCH = ROWS * (IB / 16u);  // 16-byte pieces of W per item
    constexpr int CPT = (int)((NCH + NTH - 1u) / NTH);
    const uint32_t t = threadIdx.x, lane = t & 63u, n = lane & 31u, g = lane >> 5;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(t >> 6);
    // tiles that share rows of W follow each other on one XCD
    const uint32_t tn = (a.B + COLS - 1u) / COLS, nt = gridDim.x;
    const uint32_t bid = vx_xcd_order(blockIdx.x, nt);
    const uint32_t wm = wave / WN, wn = wave % WN;
    const uint32_t row0 = (bid / tn) * ROWS, col0 = (bid % tn) * COLS;
    const uint32_t nblk = a.K / 32u, ipr = (nblk + 7u) >> 3;

    u32x4* X = (u32x4*)vx_gq_lds;  // [2][CT][2 halves][NT][64 lanes]
    constexpr uint32_t XB = 2u * CT * NT * 64u;
    uint8_t* W = (uint8_t*)(X + 2u * XB);           // [ROWS][IB]
    float* S = (float*)(W + ROWS * IB);             // OFF: [2 items][8 blocks][2 halves][COLS] sums of x
    uint32_t wlo = (64u * wm + n) * IB;             // this lane's row of row tile 0
    uint32_t* odd = (uint32_t*)(S + (OFF ? 32u * COLS : 0u));  // [COLS], see vx_gemm_q_look
    if (t < COLS) odd[t] = 0u;

    f32x16 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][c][v] = 0.f;

    const float* xp[UPT];  // this lane's first element of block 0 of the pieces it converts
#pragma unroll
    for (int u = 0; u < UPT; ++u) {
        const uint32_t pc = wave + (uint32_t)(NWV * u);
        xp[u] = a.x + (int64_t)min(col0 + 32u * (pc >> 1) + n, a.B - 1u) * a.xs_b +
                (int64_t)(8u * (pc & 1u) + 4u * g) * (XV ? 1 : a.xs_k);
    }
    const int64_t xblk = XV ? 32 : 32 * a.xs_k;
    // W: 16-byte pieces of the item's bytes. Every load is unconditional (the
    // compiler then counts outstanding loads exactly): pieces of a partial
    // last item are read from no further than the row's last 16 bytes and
    // shifted into place when they are stored.
    const uint8_t* wp[CPT];  // this thread's rows
    uint32_t wo[CPT];        // offsets of its pieces in an item
#pragma unroll
    for (int u = 0; u < CPT; ++u) {
        const uint32_t c = min(t + NTH * (uint32_t)u, NCH - 1u), r = c / (IB / 16u);
        wp[u] = a.w + (uint64_t)min(row0 + r, a.M - 1u) * a.row_stride;
        wo[u] = 16u * (c - r * (IB / 16u));
    }
    u32x4_a4 wr[CPT];
    const uint32_t rb = (nblk / (QT == VX_Q4_K ? 8u : 1u)) * vx_unit<QT>::BB;  // bytes of a row (>= 36)
    auto wload = [&](uint32_t item) {
        const uint32_t io = min(item, ipr - 1u) * IB;
#pragma unroll
        for (int u = 0; u < CPT; ++u) wr[u] = *(const u32x4_a4*)(wp[u] + min(io + wo[u], rb - 16u));
    };
    auto wstore = [&](uint32_t item) {
        const uint32_t io = item * IB;
        if (io + IB > rb) {
#pragma unroll
            for (int u = 0; u < CPT; ++u) {
                const uint32_t o = io + wo[u], sh = (o - min(o, rb - 16u)) >> 2;
                u32x4_a4 v = wr[u];
                if (sh & 1u) v = u32x4_a4{v.y, v.z, v.w, 0u};
                if (sh & 2u) v = u32x4_a4{v.z, v.w, 0u, 0u};
                wr[u] = v;  // pieces past the row's end (sh >= 4) hold nothing that is used
            }
        }
#pragma unroll
        for (int u = 0; u < CPT; ++u) {
            const uint32_t c = t + NTH * (uint32_t)u;
            if (NCH % NTH == 0u || c < NCH) *(u32x4*)(W + 16u * c) = u32x4{wr[u].x, wr[u].y, wr[u].z, wr[u].w};
        }
    };
    // x: two blocks in flight in registers (slot blk & 1) ahead of LDS
    float xr[2][UPT][8];
    auto xload = [&](uint32_t blk, int slot) {
#pragma unroll
        for (int u = 0; u < UPT; ++u) vx_x8<XV>(xp[u] + xblk * (int64_t)min(blk, nblk - 1u), a.xs_k, xr[slot][u]);
    };
    // the terms of the columns of block blk to its LDS buffer; the sums beside them
    auto xstore = [&](uint32_t blk, int slot) {
        u32x4* xb = X + (blk & 1u) * XB;
#pragma unroll
        for (int u = 0; u < UPT; ++u) {
            u32x4 xt[NT];
            vx_split8<NT>(xr[slot][u], xt);
#pragma unroll
            for (int k = 0; k < NT; ++k) xb[((wave + (uint32_t)(NWV * u)) * NT + (uint32_t)k) * 64u + lane] = xt[k];
        }
    };
    auto xsums = [&](uint32_t blk, int slot) {
        if constexpr (OFF) {
#pragma unroll
            for (int u = 0; u < UPT; ++u) {
                const uint32_t pc = wave + (uint32_t)(NWV * u);
                const float (&v)[8] = xr[slot][u];
                uint32_t s0 = __float_as_uint(((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]))), s1 = s0;
                vx_swap32(s0, s1);
                S[((blk & 15u) * 2u + (pc & 1u)) * COLS + 32u * (pc >> 1) + n] =
                    __uint_as_float(s0) + __uint_as_float(s1);  // the same from both g
            }
        }
    };
    // W operands (halves of a block) and scales of the current block and the next
    uint32_t hd[2][4];  // Q4_K: d | dmin << 16 and the 12 packed scale bytes
    bf16x8 wb[2][2][2];
    float sc[2][2];
    auto decode = [&](int b, int i) {
        if (QT == VX_Q4_K && b == 0) {
            const u32x4 h = *(const u32x4*)(W + wlo + (uint32_t)(32 * i) * IB);
            hd[i][0] = h.x; hd[i][1] = h.y; hd[i][2] = h.z; hd[i][3] = h.w;
        }
        const uint8_t* p = W + wlo + (uint32_t)(32 * i) * IB;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const uint32_t po = 8u * (uint32_t)h + 4u * g;  // byte of dword p of the block's qs
            u32x4 o;
            uint32_t lo, hi;
            if constexpr (QT == VX_Q4_0) {
                // block b at byte 18 b: d, then qs from byte 18 b + 2
                uint32_t q;
                if (b & 1) {
                    q = *(const uint32_t*)(p + 18 * b + 2 + po);
                } else {
                    const uint32_t q0 = *(const uint32_t*)(p + 18 * b + po), q1 = *(const uint32_t*)(p + 18 * b + po + 4);
                    q = __builtin_amdgcn_alignbit(q1, q0, 16);
                }
                vx_nib_bf16<CEN>(q & 0x0F0F0F0Fu, lo, hi);
                o.x = lo; o.y = hi;
                vx_nib_bf16<CEN>((q >> 4) & 0x0F0F0F0Fu, lo, hi);
                o.z = lo; o.w = hi;
            } else if constexpr (QT == VX_Q8_0) {
                uint32_t q0, q1;
                if (b & 1) {
                    q0 = *(const uint32_t*)(p + 34 * b + 2 + po);
                    q1 = *(const uint32_t*)(p + 34 * b + 18 + po);
                } else {
                    const uint32_t* r = (const uint32_t*)(p + 34 * b + po);
                    q0 = __builtin_amdgcn_alignbit(r[1], r[0], 16);
                    q1 = __builtin_amdgcn_alignbit(r[5], r[4], 16);
                }
                vx_i8_bf16(q0, lo, hi);
                o.x = lo; o.y = hi;
                vx_i8_bf16(q1, lo, hi);
                o.z = lo; o.w = hi;
            } else {
                const uint32_t* r = (const uint32_t*)(p + 16 + 32 * (b >> 1) + po);
                const uint32_t q0 = (b & 1) ? r[0] >> 4 : r[0], q1 = (b & 1) ? r[4] >> 4 : r[4];
                vx_nib_bf16<CEN>(q0 & 0x0F0F0F0Fu, lo, hi);
                o.x = lo; o.y = hi;
                vx_nib_bf16<CEN>(q1 & 0x0F0F0F0Fu, lo, hi);
                o.z = lo; o.w = hi;
            }
            wb[b & 1][i][h] = __builtin_bit_cast(bf16x8, o);
        }
        if constexpr (QT == VX_Q4_K) {
            uint32_t s0, m0, s1, m1;
            vx_q4k_scales(hd[i][1], hd[i][2], hd[i][3], (uint32_t)(b >> 1), s0, m0, s1, m1);
            sc[b & 1][i] = vx_f16_to_f32(hd[i][0]) * (float)((b & 1) ? s1 : s0);
        } else {
            sc[b & 1][i] = vx_f16_to_f32(*(const uint16_t*)(p + (QT == VX_Q4_0 ? 18 : 34) * b));
        }
        // the scale stays converted (folded into the multiply-adds as f16 it
        // would make each a v_fma_mix_f32, which issues at a lower rate)
        asm("" : "+v"(sc[b & 1][i]));
    };
    // acc += (coefficient of S) x S over the nb blocks of an item, two blocks
    // per v_mfma_f32_32x32x2f32: lane (n, g) supplies block 2j + g
    auto offsets = [&](uint32_t item, uint32_t nb) {
        if constexpr (OFF) {
            const float* sp = S + (item & 1u) * (16u * COLS) + 64u * wn + n;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint32_t blk = 2u * (uint32_t)j + g;
                const bool in = blk < nb;
                float co[2], s[2];
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const uint8_t* p = W + wlo + (uint32_t)(32 * i) * IB;
                    if constexpr (QT == VX_Q4_0) {
                        co[i] = (CEN ? -0.5f : -8.f) * vx_f16_to_f32(*(const uint16_t*)(p + 18u * blk));
                    } else {
                        // the 6-bit scale and minimum of sub-block blk
                        const uint32_t ls = p[4u + (blk & 3u)], lm = p[8u + (blk & 3u)], hi = p[12u + (blk & 3u)];
                        const uint32_t sk = j < 2 ? ls & 63u : (hi & 15u) | ((ls >> 6) << 4);
                        const uint32_t m = j < 2 ? lm & 63u : (hi >> 4) | ((lm >> 6) << 4);
                        co[i] = -(vx_f16_to_f32(*(const uint16_t*)(p + 2)) * (float)m);
                        if constexpr (CEN)
                            co[i] = __builtin_fmaf(7.5f * vx_f16_to_f32(*(const uint16_t*)p), (float)sk, co[i]);
                    }
                    co[i] = in ? co[i] : 0.f;
                    s[i] = in ? sp[blk * 2u * COLS + 32u * i] + sp[(blk * 2u + 1u) * COLS + 32u * i] : 0.f;
                }
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int c = 0; c < 2; ++c) acc[i][c] = __builtin_amdgcn_mfma_f32_32x32x2f32(s[c], co[i], acc[i][c], 0, 0, 0);
            }
        }
    };
    // The sums d of a (column tile, row tile)'s 32-block are scaled and added
    // one slot later, under the next one's MFMAs: a slot pairs each MFMA with
    // a few vector operations (scaling, decoding a row tile of the next
    // block, converting x), as the waves of a workgroup meet at every step
    // and would otherwise all multiply and all convert at the same time.
    f32x16 d[2];
#pragma unroll
    for (int v = 0; v < 16; ++v) d[1][v] = 0.f;
    sc[1][1] = 0.f;
    auto scale = [&](int i, int c, int slot, int b) {
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[i][c][v] = __builtin_fmaf(sc[b & 1][i], d[slot][v], acc[i][c][v]);
        // keeps the multiply-adds in this slot: left free, the compiler put
        // Q8_0's all at the item's end and spilled every d until then
        if constexpr (QT == VX_Q8_0) asm volatile("" : "+v"(acc[i][c]));
    };
    xload(0u, 0);
    wload(0u);
    xload(1u, 1);
    xstore(0u, 0);
    xsums(0u, 0);
    xload(2u, 0);
    wstore(0u);
    __syncthreads();
    // one item; PART: the last one, of nb < 8 blocks (a copy of its own, so that
    // the steps of whole items are one run of code without branches)
    auto step_item = [&](uint32_t item, auto part, uint32_t nb) __attribute__((always_inline)) {
        constexpr bool PART = decltype(part)::value;
        decode(0, 0);
        decode(0, 1);
        wload(item + 1u);
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            if (PART && (uint32_t)b >= nb) break;
            const uint32_t blk = 8u * item + (uint32_t)b;
            const u32x4* xb = X + (blk & 1u) * XB + wn * (4u * NT * 64u) + lane;
            // the LDS addresses of W are formed where they are used: hoisted out
            // of the loop they would take (and spill) more registers than exist
            asm volatile("" : "+v"(wlo));
            bf16x8 xt[2][2][NT];
            auto xread = [&](int c) {
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int k = 0; k < NT; ++k)
                        xt[c][h][k] = __builtin_bit_cast(bf16x8, xb[(uint32_t)((2 * c + h) * NT + k) * 64u]);
            };
            xread(0);
#pragma unroll
            for (int q = 0; q < 4; ++q) {  // slot (column tile c, row tile i)
                const int c = q >> 1, i = q & 1;
                __builtin_amdgcn_sched_barrier(0);
                if (q == 0) xread(1);
#pragma unroll
                for (int k = NT - 1; k >= 0; --k)
#pragma unroll
                    for (int h = 0; h < 2; ++h)
                        d[q & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                            xt[c][h][k], wb[b & 1][i][h], (k == NT - 1 && h == 0) ? f32x16{} : d[q & 1], 0, 0, 0);
                if (q == 0) scale(1, 1, 1, b + 1);
                else scale((q - 1) & 1, (q - 1) >> 1, (q - 1) & 1, b);
                if (q < 2 && b < 7) decode(b + 1, q);
                if (q == 2) xsums(blk + 1u, (b + 1) & 1);
                if (q == 2) xstore(blk + 1u, (b + 1) & 1);
#pragma unroll
                for (int m = 0; m < 2 * NT; ++m) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, 9, 0);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            xload(blk + 3u, (b + 1) & 1);
            if (b < 7) __syncthreads();  // (the item's last step ends below)
        }
    };
    const uint32_t nfull = nblk >> 3;
    for (uint32_t item = 0; item < nfull; ++item) {
        step_item(item, vx_bool<false>{}, 8u);
        __syncthreads();
        if constexpr (OFF) {
            offsets(item, 8u);
            __syncthreads();
        }
        wstore(min(item + 1u, ipr - 1u));
        __syncthreads();
    }
    if (nfull < ipr) {
        step_item(nfull, vx_bool<true>{}, nblk & 7u);
        __syncthreads();
        offsets(nfull, nblk & 7u);
    }
    scale(1, 1, 1, 1);  // the last block's number is odd
    float f = 0.f, lo = 1.f;  // f: a NaN when an output is not finite
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                f = __builtin_fmaf(acc[i][c][v], 0.f, f);
                lo = fminf(lo, __builtin_fabsf(acc[i][c][v]));
            }
    const bool look = f != 0.f || vx_gemm_q_odd<NT>(lo);
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const uint32_t row = row0 + 64u * wm + 32u * i + n;
                const uint32_t cc = col0 + 64u * wn + 32u * c + 8u * (v >> 2) + 4u * g + (v & 3);
                if (row < a.M && cc < a.B) a.y[(int64_t)row * a.ys_m + (int64_t)cc * a.ys_b] = acc[i][c][v];
            }
    if (look) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int c = 0; c < 2; ++c)
#pragma unroll
                for (int v = 0; v < 16; ++v)
                    if (vx_gemm_q_odd<NT>(acc[i][c][v])) odd[64u * wn + 32u * c + 8u * (v >> 2) + 4u * g + (v & 3)] = 1u;
    }
    vx_gemm_q_look<QT, NT, XV, ROWS, COLS, NWV>(a, row0, col0, odd);
}

#define VX_GEMM_Q_KS(QT, QN, NT, WR, CT)                                                                  \
    extern "C" __global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))               \
    void vx_gemm_q_##QN##_t##NT##_ks##WR##x##CT(vx_gemv_args a) {                                         \
        vx_gemm_q_ks<QT, NT, WR, CT, 8, true>(a);                                                         \
    }                                                                                                     \
    extern "C" __global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))               \
    void vx_gemm_q_##QN##_t##NT##_ks##WR##x##CT##_xs(vx_gemv_args a) {                                    \
        vx_gemm_q_ks<QT, NT, WR, CT, 8, false>(a);                                                        \
    }
#define VX_GEMM_Q_TILE(QT, QN, NT, WM, NAME)                                                              \
    extern "C" __global__ __launch_bounds__(128 * WM) __attribute__((amdgpu_waves_per_eu(2, 2)))          \
    void vx_gemm_q_##QN##_t##NT##_##NAME(vx_gemv_args a) {                                                \
        vx_gemm_q_tile<QT, NT, WM, 2, true>(a);                                                     \
    }                                                                                                     \
    extern "C" __global__ __launch_bounds__(128 * WM) __attribute__((amdgpu_waves_per_eu(2, 2)))          \
    void vx_gemm_q_##QN##_t##NT##_##NAME##_xs(vx_gemv_args a) {                                           \
        vx_gemm_q_tile<QT, NT, WM, 2, false>(a);                                                    \
    }
#define VX_GEMM_Q(QT, QN, NT)                 \
    VX_GEMM_Q_KS(QT, QN, NT, 2, 1)            \
    VX_GEMM_Q_KS(QT, QN, NT, 4, 1)            \
    VX_GEMM_Q_KS(QT, QN, NT, 4, 2)            \
    VX_GEMM_Q_TILE(QT, QN, NT, 4, 256x128)
VX_GEMM_Q(VX_Q4_0, q4_0, 2)
VX_GEMM_Q(VX_Q4_0, q4_0, 3)
VX_GEMM_Q(VX_Q8_0, q8_0, 2)
VX_GEMM_Q(VX_Q8_0, q8_0, 3)
VX_GEMM_Q(VX_Q4_K, q4_k, 2)
VX_GEMM_Q(VX_Q4_K, q4_k, 3)
