// f32 decode attention at any head dim that is a multiple of four, up to 256.
//
// Memory-bound: every key and value of the cache is read once per group of NR
// query heads. TP lanes (the power of two that covers D/4) share a key row, a
// float4 each, so a wave's loads read whole rows; a group of TP lanes keeps its
// own running (max, sum, output) over its rows and the groups of a workgroup's
// four waves merge in LDS at the end. Rows come UR at a time per group, K and V
// requested together. The sequence's rows are split evenly over nsplit x 4 waves
// by its length on the device; with one split the workgroup writes the result,
// else k_decode_any_combine merges the splits, or (SEQ, no partials) a workgroup
// takes all of its row's splits in turn and merges them the same way.
//
// Head dim 96, us on the plain kernel -> here: 8 sequences of up to 900 keys, 9/3
// heads: 527 -> 11.0; one of 3900 keys, 8 heads: 1022 -> 9.5 (1.3 TB/s); 32 of up
// to 300 keys, 32/8 heads: 506 -> 18.0 (1.7 TB/s).
#include "decode_any.h"

#include <algorithm>
#include <cmath>

#include "attn_common.h"

namespace tn {

namespace {

struct DecArgs {
    const float *q, *k, *v;
    float* out;
    float* lse;  // nullable
    const int32_t* lens;
    float* part_o;    // [B * Hq][nsplit][D] and
    float2* part_ml;  // [B * Hq][nsplit], above one split; null: SEQ
    int Hq, Hkv, nrep, cap, D, max_len, nsplit;
    float sl2;  // scale * log2(e)
};

// sum over the 2^n lanes that share a row, the same value in all of them
template <int TP>
__device__ __attribute__((always_inline)) inline float row_sum(float v) {
#if __HIP_DEVICE_COMPILE__
    auto dpp = [](float x, auto ctrl) __attribute__((always_inline)) {
        return __builtin_bit_cast(
            float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), decltype(ctrl)::value, 0xf, 0xf, false));
    };
    v = v + dpp(v, std::integral_constant<int, 0xB1>{});   // quads: lane ^ 1
    v = v + dpp(v, std::integral_constant<int, 0x4E>{});   // lane ^ 2
    v = v + dpp(v, std::integral_constant<int, 0x141>{});  // 7 - lane
    if constexpr (TP >= 16) v = v + dpp(v, std::integral_constant<int, 0x140>{});  // 15 - lane
    if constexpr (TP >= 32) v = xor16_sum(v);
    if constexpr (TP >= 64) v = xor32_sum(v);
#endif
    return v;
}

constexpr int UR = 8;  // rows in flight per group of lanes

// The merge of a row's splits in split order, as flash_any.hip's SplitMerge: the
// same bits from the partials and from one workgroup's splits in turn.
__device__ __attribute__((always_inline)) inline void merge_split(float2 s, f32x4 os, float& m, float& l, f32x4& o) {
    const float mn = fmaxf(m, s.x);
    const float mu = mn == -INFINITY ? 0.0f : mn;
    const float a = exp2f(m - mu), b = exp2f(s.x - mu);
    l = l * a + s.y * b;
#pragma unroll
    for (int e = 0; e < 4; e++) o[e] = o[e] * a + os[e] * b;
    m = mn;
}

template <int TP, int NR, bool SEQ>
__global__ __launch_bounds__(256) void k_decode_any_f32(const DecArgs a) {
    constexpr int G = 64 / TP, SLOTS = 4 * G;  // row groups per wave, per workgroup
    __shared__ __align__(16) float so[SLOTS][NR][TP * 4];
    __shared__ float2 sml[SLOTS][NR];
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane / TP, c4 = (lane % TP) * 4;
    int split = blockIdx.x;
    const int b = blockIdx.z;
    const int ng = a.nrep / NR;  // workgroups per kv head
    const int kvh = (int)blockIdx.y / ng, h0 = kvh * a.nrep + ((int)blockIdx.y % ng) * NR;
    const int D = a.D;
    const bool in = c4 < D;
    const int len = max(0, min(min(a.lens[b], a.max_len), a.cap));
    const float* kp = a.k + ((int64_t)b * a.Hkv + kvh) * a.cap * D;
    const float* vp = a.v + ((int64_t)b * a.Hkv + kvh) * a.cap * D;

    f32x4 q[NR], o[NR];
    float m[NR], l[NR];
#pragma unroll
    for (int r = 0; r < NR; r++) {
        q[r] = (f32x4){0.f, 0.f, 0.f, 0.f};
        if (in) q[r] = *reinterpret_cast<const f32x4*>(a.q + ((int64_t)b * a.Hq + h0 + r) * D + c4);
    }
    const int nb = (len + G * UR - 1) / (G * UR);
    [[maybe_unused]] float sm = -INFINITY, sl = 0.0f;  // SEQ: this thread's output over the splits so far
    [[maybe_unused]] f32x4 sacc = {0.f, 0.f, 0.f, 0.f};
    do {
        if (SEQ && split > 0) __syncthreads();  // the last split's merge has read so and sml
#pragma unroll
        for (int r = 0; r < NR; r++) {
            o[r] = (f32x4){0.f, 0.f, 0.f, 0.f};
            m[r] = -INFINITY;
            l[r] = 0.0f;
        }
        // this wave's batches of G * UR rows
        const int nw = a.nsplit * 4, gw = split * 4 + w;
        const int lo = (int)((int64_t)gw * nb / nw), hi = (int)((int64_t)(gw + 1) * nb / nw);
        for (int i = lo; i < hi; i++) {
            const int r0 = i * (G * UR);
            const uint32_t bytes = (uint32_t)min(len - r0, G * UR) * (uint32_t)(D * 4);  // rows past the length read as zeros
            const buf_rsrc rk = make_rsrc(kp + (int64_t)r0 * D, bytes), rv = make_rsrc(vp + (int64_t)r0 * D, bytes);
            f32x4 kr[UR], vr[UR];
#pragma unroll
            for (int u = 0; u < UR; u++) {
                const uint32_t off = in ? (uint32_t)((u * G + g) * D + c4) * 4u : BUF_OOB;
#if __HIP_DEVICE_COMPILE__
                kr[u] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rk, off, 0, 0));
#else
                kr[u] = f32x4{}, (void)rk, (void)off;
#endif
            }
#pragma unroll
            for (int u = 0; u < UR; u++) {
                const uint32_t off = in ? (uint32_t)((u * G + g) * D + c4) * 4u : BUF_OOB;
#if __HIP_DEVICE_COMPILE__
                vr[u] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rv, off, 0, 0));
#else
                vr[u] = f32x4{}, (void)rv, (void)off;
#endif
            }
#pragma unroll
            for (int r = 0; r < NR; r++) {
                float s[UR], mx = m[r];
#pragma unroll
                for (int u = 0; u < UR; u++) {
                    float d = q[r][0] * kr[u][0];
                    d = d + q[r][1] * kr[u][1];
                    d = d + q[r][2] * kr[u][2];
                    d = d + q[r][3] * kr[u][3];
                    s[u] = row_sum<TP>(d) * a.sl2;
                    if (r0 + u * G + g >= len) s[u] = -INFINITY;
                    mx = fmaxf(mx, s[u]);
                }
                const float mu = mx == -INFINITY ? 0.0f : mx;
                const float alpha = exp2f(m[r] - mu);  // no key seen yet: 0 times zeros
                m[r] = mx;
                l[r] = l[r] * alpha;
                o[r] = o[r] * alpha;
#pragma unroll
                for (int u = 0; u < UR; u++) {
                    const float p = exp2f(s[u] - mu);
                    l[r] = l[r] + p;
#pragma unroll
                    for (int e = 0; e < 4; e++) o[r][e] = o[r][e] + p * vr[u][e];
                }
            }
        }
#pragma unroll
        for (int r = 0; r < NR; r++) {
            *reinterpret_cast<f32x4*>(&so[w * G + g][r][c4]) = o[r];
            if (c4 == 0) sml[w * G + g][r] = make_float2(m[r], l[r]);
        }
        __syncthreads();
        const int q4 = D / 4;
        for (int t = tid; t < NR * q4; t += 256) {
            const int r = t / q4, c = (t - r * q4) * 4;
            float mm = -INFINITY;
#pragma unroll
            for (int s = 0; s < SLOTS; s++) mm = fmaxf(mm, sml[s][r].x);
            const float mu = mm == -INFINITY ? 0.0f : mm;
            float tl = 0.0f;
            f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < SLOTS; s++) {
                const float f = exp2f(sml[s][r].x - mu);
                tl = tl + sml[s][r].y * f;
                const f32x4 ov = *reinterpret_cast<const f32x4*>(&so[s][r][c]);
#pragma unroll
                for (int e = 0; e < 4; e++) acc[e] = acc[e] + ov[e] * f;
            }
            const int64_t row = (int64_t)b * a.Hq + h0 + r;
            if constexpr (SEQ) {  // NR * D / 4 <= 256: one output a thread
                merge_split(make_float2(mm, tl), acc, sm, sl, sacc);
                if (split + 1 < a.nsplit) continue;
                acc = sacc, mm = sm, tl = sl;
            }
            if (SEQ || a.nsplit == 1) {
                const float inv = 1.0f / tl;
                *reinterpret_cast<f32x4*>(a.out + row * D + c) = acc * inv;
                if (a.lse && c == 0) a.lse[row] = mm == -INFINITY ? -INFINITY : mm * LN2 + logf(tl);
            } else {
                *reinterpret_cast<f32x4*>(a.part_o + (row * a.nsplit + split) * D + c) = acc;
                if (c == 0) a.part_ml[row * a.nsplit + split] = make_float2(mm, tl);
            }
        }
    } while (SEQ && ++split < a.nsplit);
}

// one thread per four output columns
__global__ __launch_bounds__(256) void k_decode_any_combine(const DecArgs a, int64_t rows) {
    const int q4 = a.D / 4;
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t row = t / q4;
    const int c = (int)(t - row * q4) * 4;
    if (row >= rows) return;
    const float2* ml = a.part_ml + row * a.nsplit;
    const float* po = a.part_o + row * a.nsplit * a.D + c;
    float mm = -INFINITY, tl = 0.0f;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
    for (int s = 0; s < a.nsplit; s++)
        merge_split(ml[s], *reinterpret_cast<const f32x4*>(po + (int64_t)s * a.D), mm, tl, acc);
    *reinterpret_cast<f32x4*>(a.out + row * a.D + c) = acc * (1.0f / tl);
    if (a.lse && c == 0) a.lse[row] = mm == -INFINITY ? -INFINITY : mm * LN2 + logf(tl);
}

int heads_per_wg(int64_t nrep) { return nrep % 4 == 0 ? 4 : nrep % 3 == 0 ? 3 : nrep % 2 == 0 ? 2 : 1; }

}  // namespace

bool decode_any_f32_takes(int64_t Hq, int64_t D) { return D % 4 == 0 && D <= 256 && Hq <= 65535; }

// Enough workgroups for two a compute unit, each wave with at least two batches
// (64 lanes' worth of rows, UR deep), at most 32 partials a row.
int decode_any_f32_splits(int64_t B, int64_t Hq, int64_t Hkv, int64_t D, int64_t max_len) {
    const int64_t wgs = B * Hkv * ((Hq / Hkv) / heads_per_wg(Hq / Hkv));
    const int64_t rows = UR * (D <= 32 ? 8 : D <= 64 ? 4 : D <= 128 ? 2 : 1);  // of a wave's batch
    return (int)std::max<int64_t>(1, std::min<int64_t>({cdiv(512, wgs), cdiv(max_len, 8 * rows), 32}));
}

tn_status decode_any_f32(hipStream_t st, const float* q, const float* k, const float* v, int64_t B, int64_t Hq,
                         int64_t Hkv, int64_t cap, int64_t D, const int32_t* lens, int64_t max_len, double sc,
                         float* out, float* lse, float* part_o, float2* part_ml, int nsplit) {
    DecArgs a{};
    a.q = q, a.k = k, a.v = v, a.out = out, a.lse = lse, a.lens = lens;
    a.part_o = part_o, a.part_ml = part_ml;
    a.Hq = (int)Hq, a.Hkv = (int)Hkv, a.nrep = (int)(Hq / Hkv), a.cap = (int)cap, a.D = (int)D;
    a.max_len = (int)max_len, a.nsplit = nsplit;
    a.sl2 = (float)sc * LOG2E;
    const int nr = heads_per_wg(a.nrep);
    const bool seq = nsplit > 1 && !part_o;
    const dim3 grid(seq ? 1u : (unsigned)nsplit, (unsigned)(Hq / nr), (unsigned)B);
#define TN_DK(TP, NR)                                                                                          \
    do {                                                                                                       \
        if (seq) hipLaunchKernelGGL((k_decode_any_f32<TP, NR, true>), grid, dim3(256), 0, st, a);              \
        else hipLaunchKernelGGL((k_decode_any_f32<TP, NR, false>), grid, dim3(256), 0, st, a);                 \
    } while (0)
#define TN_DA(TP)                   \
    do {                            \
        if (nr == 4) TN_DK(TP, 4);  \
        else if (nr == 3) TN_DK(TP, 3); \
        else if (nr == 2) TN_DK(TP, 2); \
        else TN_DK(TP, 1);          \
    } while (0)
    if (D <= 32) TN_DA(8);
    else if (D <= 64) TN_DA(16);
    else if (D <= 128) TN_DA(32);
    else TN_DA(64);
#undef TN_DA
#undef TN_DK
    TN_LAUNCHED();
    if (nsplit > 1 && !seq) {
        const int64_t rows = B * Hq;
        hipLaunchKernelGGL(k_decode_any_combine, dim3((unsigned)cdiv(rows * (D / 4), 256)), dim3(256), 0, st, a, rows);
        TN_LAUNCHED();
    }
    return TN_OK;
}

}  // namespace tn
