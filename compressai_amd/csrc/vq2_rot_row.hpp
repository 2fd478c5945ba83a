// vq2_rot_row.hpp -- one workgroup rotates one row: the prologue of the kernels
// that pack activations for the matrix cores (vq2_rows.hip, vq2_moe_rows.hip),
// and the matrix instruction they pack for.
//
// Thread t holds the 8 values of group t: value bits 0-2 are in its
// registers, bits 3-8 across the lanes of its wave, 9-10 and 11-12 across
// waves (one radix-4 exchange through LDS each).  The stages run from bit 0
// up, as in rht_kernel (vq2_rht.hip).  One group a thread keeps a 6144-value
// row about as fast as a 2048-value one (6.9 against 5.8 us for 16 rows): with
// 256 threads and three groups each it took 11.4 us, serial latency on one wave
// per SIMD.
#pragma once

#include "vq2_common.hpp"

namespace vq2 {

typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef __bf16 bhalf8_t __attribute__((ext_vector_type(8)));

// v_mfma_f32_16x16x32 of 16-byte operands, fp16 (F16) or bf16
template <int F16>
__device__ __forceinline__ f32x4_t mfma_16(u32x4 x, u32x4 b, f32x4_t acc)
{
    if constexpr (F16)
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, x), __builtin_bit_cast(half8_t, b), acc,
                                                      0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bhalf8_t, x),
                                                       __builtin_bit_cast(bhalf8_t, b), acc, 0, 0, 0);
}

constexpr int ROT_ROW_MAX_T = 1024;  // threads, and groups of the widest row

// The 8 permutation and sign words of group g (16- and 8-byte aligned tables;
// either may be null).
__device__ __forceinline__ void rot_tables(const int32_t* perm, const int8_t* sign, int g, int32_t (&pw)[8],
                                           uint32_t (&sg)[2])
{
    if (perm) {
        const u32x4 p0 = *((const u32x4*)perm + 2 * g), p1 = *((const u32x4*)perm + 2 * g + 1);
#pragma unroll
        for (int k = 0; k < 4; k++) { pw[k] = (int32_t)p0[k]; pw[4 + k] = (int32_t)p1[k]; }
    } else {
#pragma unroll
        for (int k = 0; k < 8; k++) pw[k] = g * 8 + k;
    }
    if (sign) {
        const u32x2 w = *((const u32x2*)sign + g);
        sg[0] = w.x;
        sg[1] = w.y;
    } else {
        sg[0] = sg[1] = 0x01010101u;
    }
}

// n values of x from element x0 on into s_x as fp32 (vec: 16-byte aligned).
__device__ __forceinline__ void rot_stage_row(const void* x, int x_dt, int vec, int64_t x0, int n, float* s_x, int tid,
                                              int T)
{
    if (!vec) {
        for (int i = tid; i < n; i += T) s_x[i] = load_as_f32(x, x_dt, x0 + i);
    } else if (x_dt == VQ2_DT_F32) {
        const u32x4* xr = (const u32x4*)((const float*)x + x0);
        for (int c = tid; c < n / 4; c += T) *((u32x4*)s_x + c) = xr[c];
    } else if (tid < n / 8) {
        const u32x4 w = *((const u32x4*)((const uint16_t*)x + x0) + tid);
#pragma unroll
        for (int k = 0; k < 4; k++) {
            s_x[tid * 8 + 2 * k] = x_dt == VQ2_DT_BF16 ? __uint_as_float(w[k] << 16)
                                                       : f16_bits_to_f32((uint16_t)(w[k] & 0xFFFFu));
            s_x[tid * 8 + 2 * k + 1] = x_dt == VQ2_DT_BF16 ? __uint_as_float(w[k] & 0xFFFF0000u)
                                                           : f16_bits_to_f32((uint16_t)(w[k] >> 16));
        }
    }
}

// This thread's 8 permuted, signed values of the staged row (after a
// barrier); a table entry outside the row poisons its value, in bounds.
__device__ __forceinline__ void rot_gather(const float* s_x, const int32_t (&pw)[8], const uint32_t (&sg)[2], int n,
                                           bool g_ok, float (&v)[8])
{
#pragma unroll
    for (int k = 0; k < 8; k++) {
        const bool bad = (uint32_t)pw[k] >= (uint32_t)n;
        const float s = (float)(int8_t)(sg[k >> 2] >> (8 * (k & 3)));
        const float w = s_x[bad ? 0 : pw[k]] * s;
        v[k] = !g_ok ? 0.0f : (bad ? __builtin_nanf("") : w);
    }
}

// Blockwise FWHT over 2^hb_log2 values (64 at least), unscaled; s_x: 8 T
// floats, read by rot_gather before.  Every thread of the workgroup calls it.
__device__ __forceinline__ void rot_transform(float (&v)[8], float* s_x, int tid, int T, int hb_log2)
{
    const int lane = tid & 63;
#pragma unroll
    for (int h = 1; h < 8; h <<= 1)
#pragma unroll
        for (int k = 0; k < 8; k++)
            if ((k & h) == 0) {
                const float p = v[k], q = v[k | h];
                v[k] = p + q;
                v[k | h] = p - q;
            }
    auto stage = [&](int bit, auto partner) {
        if (hb_log2 > bit) {
            const bool up = (lane >> (bit - 3)) & 1;
#pragma unroll
            for (int k = 0; k < 8; k++) {
                const float o = partner(v[k]);
                v[k] = up ? o - v[k] : v[k] + o;
            }
        }
    };
    stage(3, [](float f) { return dpp_xor1(f); });
    stage(4, [](float f) { return dpp_xor2(f); });
    stage(5, [](float f) { return __int_as_float(__builtin_amdgcn_ds_swizzle(__float_as_int(f), 0x101F)); });
    stage(6, [](float f) { return __int_as_float(__builtin_amdgcn_ds_swizzle(__float_as_int(f), 0x201F)); });
    stage(7, [](float f) { return swz_xor16(f); });
    stage(8, [](float f) { return xor32(f); });
    // bits b and b + 1 across waves: component k of group t at k * T + t
    for (int b = 9; b < hb_log2; b += 2) {
        const int d = 1 << (b - 3);
        __syncthreads();
#pragma unroll
        for (int k = 0; k < 8; k++) s_x[k * T + tid] = v[k];
        __syncthreads();
        const bool u0 = tid & d, u1 = tid & (2 * d), two = hb_log2 > b + 1;
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const float o = s_x[k * T + (tid ^ d)];
            const float r = u0 ? o - v[k] : v[k] + o;
            if (two) {
                const float p2 = s_x[k * T + (tid ^ (2 * d))], o2 = s_x[k * T + (tid ^ (3 * d))];
                const float r2 = u0 ? o2 - p2 : p2 + o2;
                v[k] = u1 ? r2 - r : r + r2;
            } else {
                v[k] = r;
            }
        }
    }
}

// The exponent of the row's power-of-two fp16 scale from each thread's
// largest magnitude: the row's largest value lands in [2^14, 2^15), exact
// and far below 65504; a row of zeros or with an infinity keeps scale 1.
// s_max: one float per wave.
__device__ __forceinline__ int rot_row_exponent(float am, float* s_max, int tid, int T)
{
    am = wave_max_all(am);
    if ((tid & 63) == 0) s_max[tid >> 6] = am;
    __syncthreads();
    for (int w = 0; w < T / 64; w++) am = fmaxf(am, s_max[w]);
    const uint32_t ab = __float_as_uint(am);
    return ab != 0u && ab < 0x7F800000u ? 14 - ilogbf(am) : 0;
}

}  // namespace vq2
