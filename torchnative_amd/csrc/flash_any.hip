// Prefill and decode attention on the 16-bit matrix cores for the head dims
// that flash64.hip, k_flash16 and the stream-K decode do not take (any multiple
// of 8 up to 256), and for a scale of at most zero.
//
// The probabilities go into the product as P = hi + lo, both in the input format:
// 16 bits of the f32 value in bf16, 22 in f16; O += V^T hi + V^T lo in f32. The
// plain kernel, which ran these head dims before, keeps all 24. The error against
// 64 bits, which the output's own rounding sets, is the same to six digits (bf16
// 1.592e-3, f16 1.98e-4 at 300 causal tokens, D 32 to 256; up to 4096 keys, masked,
// and decode likewise).
//
// What bounds it: at these sizes one workgroup's chain of stages (load, S^T,
// softmax, P.V; about 1.3 us each), so 64 rows a workgroup (32 when there are
// no more) share a stage of 128 keys among four key groups, and the keys
// split over workgroups when the rows alone leave the device idle. Measured
// against the f32 VALU kernel: 12 heads, 777 causal tokens, D 96, bf16: 516 ->
// 20 us (70 TFLOP/s), f16 866 -> 20.5; D 256, 8 heads, 512 tokens: 629 -> 23.5;
// decode of 24 heads over 12000 keys, D 96: 6587 -> 37 us. Where the splits' partials
// have no place (a capture that may not allocate, a decode that must not), a
// workgroup takes its rows' splits in turn, the same bits: 146 us there.
//
// Decode is the same call on other rows: the query heads that share a
// key/value head are consecutive rows of q, out and lse, so (sequence, kv
// head) is a "head" of nrep query rows over a cache of `cap` keys of which
// the first lens[b] count.
#include <algorithm>

#include "attn_common.h"
#include "flash_any.h"

namespace tn {
namespace {

// 32 x DT head columns; NQ query halves of 32 rows times KG key groups of 32
// keys. LDS rows are padded to a power of two of 16-byte chunks so that the
// XOR swizzle of k_flash16 applies (the padding chunks load nothing).
template <int DT, int NQ>
struct AnyCfg {
    static constexpr int P = DT <= 2 ? 64 : DT <= 4 ? 128 : 256;  // LDS row pitch in elements
    static constexpr int KG = DT <= 4 ? 4 : 2;
    static constexpr int BQ = 32 * NQ, NW = NQ * KG, NT = 64 * NW;
    static constexpr int ROWS = 32 * KG;  // keys per ring stage
    static constexpr int STAGE = ROWS * P * 2;  // bytes of one K (or V) stage
};

// Additive mask value in natural units, its format at run time (MaskRef).
template <bool F16>
__device__ inline f32x4 any_mask_quad(int kind, const MaskRef& m, int64_t row, int key, int S) {
    if (kind == 1) return mask_quad<1, F16>(m, row, key, S);
    if (kind == 3) return mask_quad<3, F16>(m, row, key, S);
    return mask_quad<2, F16>(m, row, key, S);
}

// The same from a quad loaded ahead (MaskAhead), its format at run time.
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
template <bool F16>
__device__ inline f32x4 any_mask_values(int kind, u32x4 v, uint32_t shift) {
    if (kind == 1) return mask_values<1, F16>(v, shift);
    if (kind == 3) return mask_values<3, F16>(v, shift);
    return mask_values<2, F16>(v, shift);
}

// f16: probabilities times 2^6 (at most 2^14 with the lazy rescale's slack),
// so that they leave f16's normal range six powers of two later
template <bool F16>
constexpr float P_BIAS = F16 ? 6.0f : 0.0f;
template <bool F16>
constexpr float P_UNIT = F16 ? 1.0f / 64 : 1.0f;  // takes the factor out of the sum again, exactly

// P = hi + lo must give P * V's infinity where V holds one. hi carries the sign
// of P and is positive wherever P is: an f16 hi would round to zero under 2^-25
// (x times 2^126 is x, or past the smallest f16, or zero). lo has either sign and
// is zero where hi is exact, so it multiplies V clamped to the largest finite
// value (a NaN too: hi's product keeps it).
template <bool F16>
__device__ __attribute__((always_inline)) inline float hi_of(float x) {
    if constexpr (F16) return __builtin_amdgcn_fmed3f(x, x * 0x1p126f, 0x1p-24f);
    else return x;
}

typedef short s16x2 __attribute__((ext_vector_type(2)));
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
// As signed numbers only positive patterns lie past +max, as unsigned ones only
// negative patterns past -max.
template <bool F16>
__device__ __attribute__((always_inline)) inline uint32_t finite2(uint32_t w) {
    constexpr short TOP = F16 ? 0x7bff : 0x7f7f;
    constexpr unsigned short LOW = F16 ? 0xfbff : 0xff7f;
    const s16x2 a = __builtin_elementwise_min(__builtin_bit_cast(s16x2, w), (s16x2){TOP, TOP});
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_min(__builtin_bit_cast(u16x2, a), (u16x2){LOW, LOW}));
}

// The merge of a row's splits, one after another in split order from
// m = -inf, l = 0, o = 0: o = o * a + o_s * b, l likewise. k_any_combine and the
// kernel that takes its splits in turn (SEQ) give the same bits.
struct SplitMerge {
    float a, b;
    __device__ __attribute__((always_inline)) inline SplitMerge(float2 s, float& m, float& l) {
        const float mn = fmaxf(m, s.x);
        const float mu = mn == -INFINITY ? 0.0f : mn;
        a = exp2f(m - mu);
        b = exp2f(s.x - mu);
        l = l * a + s.y * b;
        m = mn;
    }
    __device__ __attribute__((always_inline)) inline float operator()(float o, float os) const { return o * a + os * b; }
};

// SEQ: no partials, one workgroup takes all the splits of its rows.
template <int DT, int NQ, bool MASKED, bool F16, bool SEQ>
__global__ __launch_bounds__((AnyCfg<DT, NQ>::NT)) void k_flash_any(const AnyArgs a) {
    using C = AnyCfg<DT, NQ>;
    using E = El<F16>;
    using V8 = typename E::v8;
    constexpr int P = C::P, KG = C::KG, CPR = P / 8, LPT = C::ROWS * CPR / C::NT;
    static_assert(LPT * C::NT == C::ROWS * CPR, "stage must split evenly over the threads");
    __shared__ __align__(16) uint8_t ring[4 * C::STAGE];  // K, V of two stages
    __shared__ float2 s_ml[KG / 2][NQ][64];

    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int qw = w % NQ, kg = w / NQ;
    const int lq = lane & 31, hh = lane >> 5;
    // long causal blocks first; the splits of a block side by side
    const int nqb = (a.L + C::BQ - 1) / C::BQ;
    const int wg = wg_number();
    if (wg >= a.nwg) return;
    int split = SEQ ? 0 : wg % a.nsplit;
    const int unit = SEQ ? wg : wg / a.nsplit;
    const int bh = unit % a.BH, qt = nqb - 1 - unit / a.BH;
    const int h = bh % a.Hq, b = bh / a.Hq;
    const int kvh = h / (a.Hq / a.Hkv);
    const int D = a.D;
    const int q0 = qt * C::BQ, qw0 = q0 + qw * 32, qi = qw0 + lq;
    const int kvalid = a.lens ? max(0, min(min(a.lens[b], a.max_len), a.S)) : a.S;
    const int kend = a.causal ? min(kvalid, q0 + C::BQ) : kvalid;
    const int nst_row = (kend + C::ROWS - 1) / C::ROWS;

    const uint16_t* qp = a.q + (int64_t)bh * a.L * D;
    const uint16_t* kp = a.k + ((int64_t)b * a.Hkv + kvh) * a.S * D;
    const uint16_t* vp = a.v + ((int64_t)b * a.Hkv + kvh) * a.S * D;

    auto swz = [](int r, int c) { return P == 64 ? (c ^ ((r >> 1) & 7)) : (c ^ (r & 15)); };

    V8 qf[2 * DT];
#pragma unroll
    for (int c = 0; c < 2 * DT; c++) {
        uint4 v = make_uint4(0, 0, 0, 0);
        const int d = 16 * c + 8 * hh;
        if (qi < a.L && d < D) v = *reinterpret_cast<const uint4*>(qp + (int64_t)qi * D + d);
        qf[c] = __builtin_bit_cast(V8, v);
    }
    // this thread's 16-byte pieces of a stage: LDS place p holds chunk
    // swz(row, p % CPR) of row p / CPR; columns past D load zeros
    uint32_t voff[LPT];
#pragma unroll
    for (int i = 0; i < LPT; i++) {
        const int p = (w * LPT + i) * 64 + lane, row = p / CPR, c = swz(row, p % CPR);
        voff[i] = c * 8 < D ? (uint32_t)(row * D + c * 8) * 2u : BUF_OOB;
    }
    auto issue = [&](int st) __attribute__((always_inline)) {
        const int k0 = st * C::ROWS;
        const uint32_t bytes = (uint32_t)(kvalid - k0) * (uint32_t)(D * 2);  // keys past the last read as zero
        const LdsDma rk(kp + (int64_t)k0 * D, bytes), rv(vp + (int64_t)k0 * D, bytes);
        uint8_t* const s = ring + (st & 1) * 2 * C::STAGE;
#pragma unroll
        for (int i = 0; i < LPT; i++) rk.load16(voff[i], s + (w * LPT + i) * 1024);
#pragma unroll
        for (int i = 0; i < LPT; i++) rv.load16(voff[i], s + C::STAGE + (w * LPT + i) * 1024);
    };

    // a stage's mask quads come with its K and V (four dwords whatever the
    // format; past the plane they read as zeros)
    const MaskRef mask{a.mask, a.msb, a.msh, a.msl, a.msk};
    const int mes = a.mk == 1 ? 4 : a.mk == 3 ? 1 : 2;
    [[maybe_unused]] const MaskRow mr(mask, mes, b, h, qi, a.L, a.S);
    [[maybe_unused]] u32x4 mq[4] = {}, mcur[4];
    auto mload = [&](int st) __attribute__((always_inline)) {
#if __HIP_DEVICE_COMPILE__
        if constexpr (MASKED) {
            if (a.mahead) {
#pragma unroll
                for (int rq = 0; rq < 4; rq++)
                    mq[rq] = __builtin_bit_cast(
                        u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                   mr.r, mr.off + (uint32_t)((st * C::ROWS + kg * 32 + 8 * rq + 4 * hh) * mes), 0, 0));
            }
        }
#endif
    };

    f32x16 o[DT];
    float m, l;
    [[maybe_unused]] f32x16 so[SEQ ? DT : 1];  // SEQ: the splits so far
    [[maybe_unused]] float sm = -INFINITY, sl = 0.0f;
    if constexpr (SEQ) {
#pragma unroll
        for (int i = 0; i < DT; i++)
#pragma unroll
            for (int r = 0; r < 16; r++) so[i][r] = 0.0f;
    }
    do {
        if (SEQ && split > 0) __syncthreads();  // the last split's merge has read the ring
#pragma unroll
        for (int i = 0; i < DT; i++)
#pragma unroll
            for (int r = 0; r < 16; r++) o[i][r] = 0.0f;
        m = -INFINITY, l = 0.0f;
        const int st_lo = (int)((int64_t)split * nst_row / a.nsplit);
        const int st_hi = (int)((int64_t)(split + 1) * nst_row / a.nsplit);
        if (st_lo < st_hi) {
            issue(st_lo);
            mload(st_lo);
        }
        for (int st = st_lo; st < st_hi; st++) {
            wait_vmcnt<0>();  // the only loads in flight are this stage's
            if constexpr (MASKED) {
#pragma unroll
                for (int rq = 0; rq < 4; rq++) {
                    // the compiler's own wait falls here, where nothing is in flight
                    asm volatile("" : "+v"(mq[rq]));
                    mcur[rq] = mq[rq];
                }
            }
            // this wave's reads of the other stage, which the barrier opens to issue()
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            if (st + 1 < st_hi) {
                issue(st + 1);  // into the stage read before the barrier
                mload(st + 1);
            }
            const int k0 = st * C::ROWS + kg * 32;
            if (k0 >= kend || (a.causal && qw0 + 31 < k0)) continue;
            const uint16_t* tK = reinterpret_cast<const uint16_t*>(ring + (st & 1) * 2 * C::STAGE);
            const uint16_t* tV = tK + C::STAGE / 2;
            const int kr = 32 * kg;

            f32x16 acc;
#pragma unroll
            for (int r = 0; r < 16; r++) acc[r] = 0.0f;
#pragma unroll
            for (int c = 0; c < 2 * DT; c++) {
                const int row = kr + lq;
                const V8 ka = *reinterpret_cast<const V8*>(tK + row * P + swz(row, 2 * c + hh) * 8);
                acc = E::mfma(ka, qf[c], acc);
            }
            // the XDL wait states before VALU reads the products (as k_flash16)
            asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 3" : "+v"(acc));
            float v[16];
#pragma unroll
            for (int r = 0; r < 16; r++) v[r] = acc[r] * a.sl2;
            if constexpr (MASKED) {
                if (a.mahead) {
#pragma unroll
                    for (int rq = 0; rq < 4; rq++) {
                        const f32x4 mv = any_mask_values<F16>(a.mk, mcur[rq], mr.shift);
#pragma unroll
                        for (int e = 0; e < 4; e++) v[4 * rq + e] = v[4 * rq + e] + mv[e] * LOG2E;
                    }
                } else if (qi < a.L) {
                    const int64_t mrow = (int64_t)b * mask.sb + (int64_t)h * mask.sh + (int64_t)qi * mask.sl;
#pragma unroll
                    for (int rq = 0; rq < 4; rq++) {
                        const f32x4 mv = any_mask_quad<F16>(a.mk, mask, mrow, k0 + 8 * rq + 4 * hh, a.S);
#pragma unroll
                        for (int e = 0; e < 4; e++) v[4 * rq + e] = v[4 * rq + e] + mv[e] * LOG2E;
                    }
                }
            }
            if (k0 + 32 > kvalid || (a.causal && k0 + 31 > qw0)) {
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const int key = k0 + 8 * (r >> 2) + 4 * hh + (r & 3);
                    if (key >= kvalid || (a.causal && key > qi)) v[r] = -INFINITY;
                }
            }
            float mx = max3f(max3f(max3f(v[0], v[1], v[2]), v[3], v[4]), max3f(v[5], v[6], v[7]),
                             max3f(max3f(v[8], v[9], v[10]), v[11], v[12]));
            mx = xor32_max(max3f(mx, max3f(v[13], v[14], v[15]), mx));
            const bool need = mx > m + RESCALE_SLACK;
            if (__any(need)) {
                const float mn = need ? mx : m;
                // a row with no key seen yet keeps m = mn = -inf: alpha 1, not 2^NaN
                const float alpha = mn == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f(m - mn);
                l = l * alpha;
#pragma unroll
                for (int i = 0; i < DT; i++) o[i] = o[i] * alpha;
                m = mn;
            }
            const float mu = ((m == -INFINITY) ? 0.0f : m) - P_BIAS<F16>;
            float p[16];
#pragma unroll
            for (int r = 0; r < 16; r++) p[r] = __builtin_amdgcn_exp2f(v[r] - mu);
            float ps = 0.0f;
#pragma unroll
            for (int r = 0; r < 16; r += 4) ps = ps + ((p[r] + p[r + 1]) + (p[r + 2] + p[r + 3]));
            l = l + ps;
            V8 ph[2], pl[2];  // p = hi + lo
#pragma unroll
            for (int j = 0; j < 2; j++) {
                uint32_t hi[4], lo[4];
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const float x0 = p[8 * j + 2 * e], x1 = p[8 * j + 2 * e + 1];
                    hi[e] = E::pack_p(hi_of<F16>(x0), hi_of<F16>(x1));
                    lo[e] = E::pack_p(x0 - E::lo(hi[e]), x1 - E::hi(hi[e]));
                }
                ph[j] = __builtin_bit_cast(V8, make_uint4(hi[0], hi[1], hi[2], hi[3]));
                pl[j] = __builtin_bit_cast(V8, make_uint4(lo[0], lo[1], lo[2], lo[3]));
            }
            const int gi = lane & 15;
            const int dcol = 16 * ((lane >> 4) & 1) + 4 * (gi & 3);  // the V^T operand's source columns (k_flash16)
#pragma unroll
            for (int dt = 0; dt < DT; dt++) {
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    const int r0 = kr + 16 * j + 4 * hh + (gi >> 2), r1 = r0 + 8;
                    const int col = 32 * dt + dcol;
                    const uint2 lo = lds_read_tr16(tV + r0 * P + swz(r0, col >> 3) * 8 + (col & 7));
                    const uint2 hi = lds_read_tr16(tV + r1 * P + swz(r1, col >> 3) * 8 + (col & 7));
                    const V8 va = __builtin_bit_cast(V8, make_uint4(lo.x, lo.y, hi.x, hi.y));
                    const V8 vf = __builtin_bit_cast(V8, make_uint4(finite2<F16>(lo.x), finite2<F16>(lo.y),
                                                                    finite2<F16>(hi.x), finite2<F16>(hi.y)));
                    o[dt] = E::mfma(va, ph[j], o[dt]);
                    o[dt] = E::mfma(vf, pl[j], o[dt]);
                }
            }
        }
#pragma unroll
        for (int i = 0; i < DT; i++) asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 3" : "+v"(o[i]));

        l = xor32_sum(l);
        // tree merge of the key groups through LDS, over the ring (every load has
        // landed and been read once the first barrier has passed)
        constexpr int WSLOT = DT * 16 * 64;  // floats per wave
        static_assert((KG / 2) * NQ * WSLOT * 4 <= 4 * C::STAGE, "merge slots must fit in the ring");
#pragma unroll
        for (int half = KG / 2; half >= 1; half /= 2) {
            __syncthreads();
            if (kg >= half && kg < 2 * half) {
                float* xo = reinterpret_cast<float*>(ring) + ((kg - half) * NQ + qw) * WSLOT;
#pragma unroll
                for (int dt = 0; dt < DT; dt++)
#pragma unroll
                    for (int r = 0; r < 16; r++) xo[(dt * 16 + r) * 64 + lane] = o[dt][r];
                s_ml[kg - half][qw][lane] = make_float2(m, l);
            }
            __syncthreads();
            if (kg < half) {
                const float* xo = reinterpret_cast<const float*>(ring) + (kg * NQ + qw) * WSLOT;
                const float2 ml1 = s_ml[kg][qw][lane];
                const float mm = fmaxf(m, ml1.x);
                const float mu = (mm == -INFINITY) ? 0.0f : mm;
                const float a0 = __builtin_amdgcn_exp2f(m - mu), a1 = __builtin_amdgcn_exp2f(ml1.x - mu);
                l = l * a0 + ml1.y * a1;
#pragma unroll
                for (int dt = 0; dt < DT; dt++)
#pragma unroll
                    for (int r = 0; r < 16; r++) o[dt][r] = o[dt][r] * a0 + xo[(dt * 16 + r) * 64 + lane] * a1;
                m = mm;
            }
        }
        if constexpr (SEQ) {
            if (kg == 0) {
                const SplitMerge mg(make_float2(m, l), sm, sl);
#pragma unroll
                for (int i = 0; i < DT; i++)
#pragma unroll
                    for (int r = 0; r < 16; r++) so[i][r] = mg(so[i][r], o[i][r]);
            }
        }
    } while (SEQ && ++split < a.nsplit);
    if constexpr (SEQ) {
#pragma unroll
        for (int i = 0; i < DT; i++) o[i] = so[i];
        m = sm, l = sl;
    }
    if (kg != 0 || qi >= a.L) return;
    const int64_t row = (int64_t)bh * a.L + qi;
    if (!SEQ && a.nsplit > 1) {
        float* po = a.part_o + (row * a.nsplit + split) * D;
#pragma unroll
        for (int dt = 0; dt < DT; dt++)
#pragma unroll
            for (int g4 = 0; g4 < 4; g4++) {
                const int d = 32 * dt + 8 * g4 + 4 * hh;
                if (d < D)
                    *reinterpret_cast<float4*>(po + d) =
                        make_float4(o[dt][4 * g4], o[dt][4 * g4 + 1], o[dt][4 * g4 + 2], o[dt][4 * g4 + 3]);
            }
        if (hh == 0) a.part_ml[row * a.nsplit + split] = make_float2(m, l);
        return;
    }
    const float inv = 1.0f / l;  // a row with no key: 0 * inf = NaN, as the reference's (aten.rs:10392-10420)
    uint16_t* op = a.out + row * D;
#pragma unroll
    for (int dt = 0; dt < DT; dt++)
#pragma unroll
        for (int g4 = 0; g4 < 4; g4++) {
            // O^T[d = 32dt + 8g4 + 4hh + e][q = lq]
            const int d = 32 * dt + 8 * g4 + 4 * hh;
            if (d < D)
                *reinterpret_cast<uint2*>(op + d) =
                    make_uint2(E::pack_out(o[dt][4 * g4] * inv, o[dt][4 * g4 + 1] * inv),
                               E::pack_out(o[dt][4 * g4 + 2] * inv, o[dt][4 * g4 + 3] * inv));
        }
    // a row with no key: NaN; a decode sequence of length 0: -inf
    if (a.lse && hh == 0)
        a.lse[row] = m == -INFINITY ? (a.lens ? -INFINITY : NAN) : m * LN2 + logf(l * P_UNIT<F16>);
}

// The splits of a row, merged in split order: a thread per four columns.
template <bool F16>
__global__ __launch_bounds__(256) void k_any_combine(const AnyArgs a, int64_t rows) {
    const int q4 = a.D / 4;
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t row = t / q4;
    const int c = (int)(t - row * q4) * 4;
    if (row >= rows) return;
    float mm = -INFINITY, tl = 0.0f;
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll 4
    for (int s = 0; s < a.nsplit; s++) {
        const float4 v = *reinterpret_cast<const float4*>(a.part_o + (row * a.nsplit + s) * a.D + c);
        const SplitMerge mg(a.part_ml[row * a.nsplit + s], mm, tl);
        acc = make_float4(mg(acc.x, v.x), mg(acc.y, v.y), mg(acc.z, v.z), mg(acc.w, v.w));
    }
    const float inv = 1.0f / tl;
    *reinterpret_cast<uint2*>(a.out + row * a.D + c) =
        make_uint2(El<F16>::pack_out(acc.x * inv, acc.y * inv), El<F16>::pack_out(acc.z * inv, acc.w * inv));
    if (a.lse && c == 0)
        a.lse[row] = mm == -INFINITY ? (a.lens ? -INFINITY : NAN) : mm * LN2 + logf(tl * P_UNIT<F16>);
}

template <int DT, int NQ, bool SEQ>
void launch_nq(hipStream_t st, AnyArgs a, bool f16, int64_t wgs) {
    using C = AnyCfg<DT, NQ>;
    const dim3 grid = wg_grid(wgs);
    a.nwg = (int)wgs;
#define TN_FA(M, H) hipLaunchKernelGGL((k_flash_any<DT, NQ, M, H, SEQ>), grid, dim3(C::NT), 0, st, a)
    if (a.mk) {
        if (f16) TN_FA(true, true);
        else TN_FA(true, false);
    } else {
        if (f16) TN_FA(false, true);
        else TN_FA(false, false);
    }
#undef TN_FA
}

template <int DT>
void launch_dt(hipStream_t st, const AnyArgs& a, bool f16, int nq) {
    const int64_t units = (int64_t)a.BH * cdiv(a.L, 32 * nq);
    if (a.nsplit > 1 && !a.part_o) {
        if (nq == 1) launch_nq<DT, 1, true>(st, a, f16, units);
        else launch_nq<DT, 2, true>(st, a, f16, units);
    } else {
        if (nq == 1) launch_nq<DT, 1, false>(st, a, f16, units * a.nsplit);
        else launch_nq<DT, 2, false>(st, a, f16, units * a.nsplit);
    }
}

}  // namespace

bool flash_any_takes(const AnyArgs& a) {
    const uintptr_t all = reinterpret_cast<uintptr_t>(a.q) | reinterpret_cast<uintptr_t>(a.k) |
                          reinterpret_cast<uintptr_t>(a.v) | reinterpret_cast<uintptr_t>(a.out);
    return a.D % 8 == 0 && a.D <= 256 && all % 16 == 0 && (int64_t)a.S * a.D * 2 <= INT32_MAX &&
           (int64_t)a.BH * cdiv(a.L, 32) <= INT32_MAX / FLASH_ANY_MAX_SPLIT;
}

// Splits of the keys: enough workgroups for the device when the rows alone
// give few, each at least two ring stages of 128 keys.
int flash_any_splits(const AnyArgs& a) {
    const int64_t units = (int64_t)a.BH * cdiv(a.L, a.L <= 32 ? 32 : 64);
    const int64_t keys = a.lens ? a.max_len : a.S;
    const int64_t want = std::min<int64_t>(cdiv(256, units), keys / 256);
    return (int)std::max<int64_t>(1, std::min<int64_t>(want, FLASH_ANY_MAX_SPLIT));
}

tn_status flash_any_launch(hipStream_t st, bool f16, const AnyArgs& a) {
    const int nq = a.L <= 32 ? 1 : 2;
    const int dt = (a.D + 31) / 32;
    if (dt == 1) launch_dt<1>(st, a, f16, nq);
    else if (dt == 2) launch_dt<2>(st, a, f16, nq);
    else if (dt == 3) launch_dt<3>(st, a, f16, nq);
    else if (dt == 4) launch_dt<4>(st, a, f16, nq);
    else launch_dt<8>(st, a, f16, nq);
    TN_LAUNCHED();
    if (a.nsplit > 1 && a.part_o) {
        const int64_t rows = (int64_t)a.BH * a.L;
        const dim3 grid((unsigned)cdiv(rows * (a.D / 4), 256));
        if (f16) hipLaunchKernelGGL(k_any_combine<true>, grid, dim3(256), 0, st, a, rows);
        else hipLaunchKernelGGL(k_any_combine<false>, grid, dim3(256), 0, st, a, rows);
        TN_LAUNCHED();
    }
    return TN_OK;
}

}  // namespace tn
