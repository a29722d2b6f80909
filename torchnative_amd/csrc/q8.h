// The Q8_0 activation quantiser's shared pieces (qlinear.hip, qgemm.hip).
#pragma once

#include "tn_common.h"

namespace tn {

enum WeightFormat { FMT_Q4_0 = 0, FMT_Q8_0 = 1 };

namespace {

constexpr int QK = 32;

// ---- Rust cast semantics ---------------------------------------------------

// Truncation toward zero after clamping to the type's range, NaN to 0. The
// clamp and the NaN test are selects: written as early returns they became
// three nested exec-mask branches per element.
__device__ inline int sat_i8(float v) {  // `f as i8`
    const int q = (int)fminf(fmaxf(v, -128.0f), 127.0f);
    return v != v ? 0 : q;
}

__device__ inline int sat_u8(float v) {  // `f as u8`
    const int q = (int)fminf(fmaxf(v, 0.0f), 255.0f);
    return v != v ? 0 : q;
}

// Eight consecutive activations as floats: 16 bytes of bf16 or 32 of f32, at any
// element (the vector types carry the elements' alignment only).
template <typename XT>
__device__ inline void load_x8(const XT* p, float (&v)[8]);
template <>
__device__ inline void load_x8<float>(const float* p, float (&v)[8]) {
    typedef float f4 __attribute__((ext_vector_type(4), aligned(4)));
    const f4 a = reinterpret_cast<const f4*>(p)[0], b = reinterpret_cast<const f4*>(p)[1];
#pragma unroll
    for (int i = 0; i < 4; i++) v[i] = a[i], v[4 + i] = b[i];
}
template <>
__device__ inline void load_x8<uint16_t>(const uint16_t* p, float (&v)[8]) {
    typedef uint32_t u4 __attribute__((ext_vector_type(4), aligned(2)));
    const u4 w = *reinterpret_cast<const u4*>(p);
#pragma unroll
    for (int i = 0; i < 4; i++) {
        v[2 * i] = __builtin_bit_cast(float, w[i] << 16);
        v[2 * i + 1] = __builtin_bit_cast(float, w[i] & 0xffff0000u);
    }
}

// The Q8_0 codes of one block held by four lanes, eight elements each: the
// block's amax (order-free), d = amax/127, id = 1/d (the f32 d, not the stored
// f16 one), codes rounded half away from zero (BlockQ8_0::from_float,
// k_quants.rs:676-705); the code sum comes back through `s`.
__device__ inline void q8_0_quad(const float (&v)[8], int (&q)[8], float* dx, int* s) {
    float a = 0.0f;  // f32::max from 0: NaNs are skipped (k_quants.rs:676-705)
#pragma unroll
    for (int e = 0; e < 8; e++) a = fmaxf(a, fabsf(v[e]));
    a = fmaxf(a, __shfl_xor(a, 1, 4));
    a = fmaxf(a, __shfl_xor(a, 2, 4));
    const float d = a / 127.0f;
    const float id = (d != 0.0f) ? 1.0f / d : 0.0f;
    *dx = f16_to_f32(f16_from_f32(d));
    int sum = 0;
#pragma unroll
    for (int e = 0; e < 8; e++) {
        q[e] = sat_i8(roundf(v[e] * id));
        sum += q[e];
    }
    sum += __shfl_xor(sum, 1, 4);
    sum += __shfl_xor(sum, 2, 4);
    *s = sum;
}

// How the prepass finds a row's activations (XM_* in tn_common.h). XM_ROWS:
// row r is x[r][0..K). XM_GLU: x holds [M][2K] rows (gate | up) and the
// activation is silu(gate) * up, k_silu_mul's arithmetic (decode.hip).
// XM_HEADS: x is an attention output [K / hd][M][hd] (head-major) and row r
// is its heads' rows of token r side by side. The last two let a prompt's
// down and o projections read their producers' outputs without a copy in
// between.

template <typename XT, int XM>
__device__ inline void load_part(const XT* __restrict__ x, int row, int M, int K, int b, int part, int hd,
                                 float (&v)[8]) {
    if constexpr (XM == XM_GLU) {
        float g[8], u[8];
        load_x8<XT>(x + (int64_t)row * 2 * K + b * QK + 8 * part, g);
        load_x8<XT>(x + (int64_t)row * 2 * K + K + b * QK + 8 * part, u);
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = (g[e] / (1.0f + expf(-g[e]))) * u[e];
    } else if constexpr (XM == XM_HEADS) {
        const int e0 = b * QK, h = e0 / hd;
        load_x8<XT>(x + ((int64_t)h * M + row) * hd + (e0 - h * hd) + 8 * part, v);
    } else {
        load_x8<XT>(x + (int64_t)row * K + b * QK + 8 * part, v);
    }
}

}  // namespace
}  // namespace tn
