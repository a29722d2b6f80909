// flash_any.hip's interface: attention on the 16-bit matrix cores for any head
// dim that is a multiple of 8 (up to 256) and a scale of either sign.
#pragma once

#include "tn_common.h"

namespace tn {

struct AnyArgs {
    const uint16_t *q, *k, *v;  // q [BH][L][D], k/v [B][Hkv][S][D]
    uint16_t* out;              // [BH][L][D]
    float* lse;                 // nullable [BH][L]
    int BH, Hq, Hkv, L, S, D;   // BH = B * Hq; head h reads kv head h / (Hq / Hkv)
    float sl2;                  // scale * log2(e)
    int causal;
    const int32_t* lens;  // nullable [B]: keys of sequence b (at most max_len and S)
    int max_len;
    int nsplit;        // splits of the keys (the result's bits depend on it); above 1 the partials below hold
    float* part_o;     // BH * L * nsplit * D floats and
    float2* part_ml;   // BH * L * nsplit pairs; null: a workgroup takes its row's splits one after another
    int nwg;           // workgroups (set by the launch)
    int mk;            // mask kind: 0 none, 1 f32, 2 the input format, 3 bool
    int mahead;        // its quads are loaded with their keys (mask_ahead)
    const void* mask;  // and its element strides over (B, Hq, L, S)
    int64_t msb, msh, msl, msk;
};

constexpr int FLASH_ANY_MAX_SPLIT = 64;

// Whether the kernel takes this call (head dim, alignment, sizes).
bool flash_any_takes(const AnyArgs& a);
// The splits it takes; the caller provides partials for them if it can.
int flash_any_splits(const AnyArgs& a);
tn_status flash_any_launch(hipStream_t st, bool f16, const AnyArgs& a);

}  // namespace tn
