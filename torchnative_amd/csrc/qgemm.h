// qgemm.hip's interface: the q4_0 / q8_0 linear of more rows than the GEMV takes.
#pragma once

#include "q8.h"

namespace tn {

struct QGemmArgs {
    int fmt;        // WeightFormat
    const void* x;  // activations, f32 or bf16 (XM_ROWS), found as xm says (XM_*)
    int x_bf16;
    int64_t m, k;
    int xm, hd;
    const uint8_t* qs;  // any alignment (16-byte aligned ones are read straight into LDS)
    const uint16_t* d;
    int64_t n;
    const float* bias;
    void* y;
    int y_bf16;
    const float* resid;  // added after the sum (and bias), may be y
};

// Bytes of the stream's workspace that qgemm_launch uses.
inline size_t qgemm_workspace(const QGemmArgs& a) { return (size_t)(cdiv(a.m, 16) * 16 * (a.k / QK)) * (32 + 4); }
// Quantises the rows into the stream's workspace, then the product.
tn_status qgemm_launch(hipStream_t st, const QGemmArgs& a);

}  // namespace tn
