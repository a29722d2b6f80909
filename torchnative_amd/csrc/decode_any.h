// f32 decode attention at any head dim that is a multiple of four (decode_any.hip).
#pragma once

#include "tn_common.h"

namespace tn {

bool decode_any_f32_takes(int64_t Hq, int64_t D);
// The splits it takes (the result's bits depend on them); the caller provides the
// partials (part_o B*Hq*nsplit rows of D floats, part_ml as many pairs) if it can:
// without them one workgroup takes all the splits of its rows.
int decode_any_f32_splits(int64_t B, int64_t Hq, int64_t Hkv, int64_t D, int64_t max_len);
// Pointers 16-byte aligned; lens, B, Hq, cap and max_len as tn_sdpa_decode checks them.
tn_status decode_any_f32(hipStream_t st, const float* q, const float* k, const float* v, int64_t B, int64_t Hq,
                         int64_t Hkv, int64_t cap, int64_t D, const int32_t* lens, int64_t max_len, double sc,
                         float* out, float* lse, float* part_o, float2* part_ml, int nsplit);

}  // namespace tn
