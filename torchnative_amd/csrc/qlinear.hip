// GGML block-quantised weights on gfx950 (q4_0 and q8_0): upload/repack,
// quantise, dequantise, and the quantised linear (the decode GEMV here; more
// rows on qgemm.hip).
//
// Arithmetic contract (candle-core/src/quantized/k_quants.rs, the reference's
// vendored candle): every output is
//     sumf = 0; for b in blocks: sumf += ((float)S_b * d_w[b]) * d_x[b]
// where S_b is the exact integer dot of the weight's codes (q4_0: nib - 8,
// vec_dot_unopt k_quants.rs:312-329; q8_0: the int8 codes, k_quants.rs:738-757)
// and the activation's Q8_0 codes, and the activation row is quantised by
// BlockQ8_0::from_float (k_quants.rs:676-705) -- Q8_0 is the VecDotType of
// both weight formats. The integer dot is exact in any order, and every kernel
// below performs the float steps in exactly that order with separate
// roundings (the library is built with -ffp-contract=off), so results are
// bit-identical to the reference's x86_64 scalar path for every row count.
#include "q8.h"
#include "qgemm.h"

namespace tn {
namespace {

// Weight formats. On the device a weight is two planes: the codes of every
// block back to back in row-major block order (q4_0: the 16 nibble bytes of
// the GGML block; q8_0: its 32 int8 codes) and the f16 block scales.
template <int FMT>
struct Fmt;
template <>
struct Fmt<FMT_Q4_0> {
    static constexpr int CODE_BYTES = 16, BLOB_BYTES = 18;
    static constexpr int GEMV_ITEMS = 3;  // (row, block) items per GEMV thread: 3 streamed best on C1 (76% of HBM, 71% for 4)
    static constexpr const char* name = "q4_0";
};
template <>
struct Fmt<FMT_Q8_0> {
    static constexpr int CODE_BYTES = 32, BLOB_BYTES = 34;
    static constexpr int GEMV_ITEMS = 3;  // 32-byte items: 96 bytes in flight per thread (5.40 TB/s at the C1 shape; 5.12 for 2, 5.34 for 4)
    static constexpr const char* name = "q8_0";
};

// ---- layout conversion --------------------------------------------------------

// GGML blocks (f16 d, then the codes) <-> the two planes, one thread per block.
template <int FMT>
__global__ void k_from_blob(const uint8_t* __restrict__ blob, int64_t nblocks, uint8_t* __restrict__ qs,
                            uint16_t* __restrict__ d) {
    constexpr int CB = Fmt<FMT>::CODE_BYTES;
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nblocks) return;
    const uint8_t* s = blob + i * Fmt<FMT>::BLOB_BYTES;
    d[i] = (uint16_t)(s[0] | (s[1] << 8));
#pragma unroll
    for (int c = 0; c < CB / 16; c++) {
        uint32_t w[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const uint8_t* b = s + 2 + 16 * c + 4 * j;
            w[j] = (uint32_t)b[0] | ((uint32_t)b[1] << 8) | ((uint32_t)b[2] << 16) | ((uint32_t)b[3] << 24);
        }
        reinterpret_cast<uint4*>(qs + i * CB)[c] = make_uint4(w[0], w[1], w[2], w[3]);
    }
}

template <int FMT>
__global__ void k_to_blob(const uint8_t* __restrict__ qs, const uint16_t* __restrict__ d, int64_t nblocks,
                          uint8_t* __restrict__ blob) {
    constexpr int CB = Fmt<FMT>::CODE_BYTES;
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nblocks) return;
    uint8_t* o = blob + i * Fmt<FMT>::BLOB_BYTES;
    uint16_t h = d[i];
    o[0] = (uint8_t)(h & 0xff);
    o[1] = (uint8_t)(h >> 8);
#pragma unroll
    for (int c = 0; c < CB / 16; c++) {
        const uint4 w = reinterpret_cast<const uint4*>(qs + i * CB)[c];
        const uint32_t ws[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
        for (int j = 0; j < 16; j++) o[2 + 16 * c + j] = (uint8_t)(ws[j >> 2] >> (8 * (j & 3)));
    }
}

// BlockQ4_0::from_float (k_quants.rs:241-277) and BlockQ8_0::from_float
// (k_quants.rs:676-705), one thread per block.
template <int FMT>
__global__ void k_quantize_w(const float* __restrict__ w, int64_t nblocks, uint8_t* __restrict__ qs,
                             uint16_t* __restrict__ d) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nblocks) return;
    const float* xs = w + i * QK;
    float v[QK];
#pragma unroll
    for (int j = 0; j < QK; j += 4) {
        float4 t = *reinterpret_cast<const float4*>(xs + j);
        v[j] = t.x; v[j + 1] = t.y; v[j + 2] = t.z; v[j + 3] = t.w;
    }
    if constexpr (FMT == FMT_Q8_0) {
        float amax = 0.0f;
#pragma unroll
        for (int j = 0; j < QK; j++) amax = fmaxf(amax, fabsf(v[j]));
        const float dd = amax / 127.0f;
        const float id = (dd != 0.0f) ? 1.0f / dd : 0.0f;  // the f32 d, not the f16 one
        d[i] = f16_from_f32(dd);
        uint32_t out[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
        for (int j = 0; j < QK; j++) out[j >> 2] |= ((uint32_t)sat_i8(roundf(v[j] * id)) & 0xffu) << (8 * (j & 3));
        uint4* o = reinterpret_cast<uint4*>(qs + i * QK);
        o[0] = make_uint4(out[0], out[1], out[2], out[3]);
        o[1] = make_uint4(out[4], out[5], out[6], out[7]);
    } else {
        float amax = 0.0f, mx = 0.0f;
#pragma unroll
        for (int j = 0; j < QK; j++) {
            float a = fabsf(v[j]);
            if (amax < a) { amax = a; mx = v[j]; }  // first of the largest |x|, sign kept
        }
        float dd = mx / -8.0f;
        float id = (dd != 0.0f) ? 1.0f / dd : 0.0f;
        d[i] = f16_from_f32(dd);
        uint32_t out[4] = {0, 0, 0, 0};
#pragma unroll
        for (int j = 0; j < QK / 2; j++) {
            int q0 = sat_u8(v[j] * id + 8.5f);
            int q1 = sat_u8(v[j + QK / 2] * id + 8.5f);
            q0 = q0 < 15 ? q0 : 15;
            q1 = q1 < 15 ? q1 : 15;
            out[j >> 2] |= (uint32_t)(q0 | (q1 << 4)) << (8 * (j & 3));
        }
        *reinterpret_cast<uint4*>(qs + i * 16) = make_uint4(out[0], out[1], out[2], out[3]);
    }
}

// BlockQ4_0::to_float (k_quants.rs:219-239): (nib - 8) as f32 * f32(d);
// BlockQ8_0::to_float (k_quants.rs:659-674): q as f32 * f32(d). Both exact.
template <int FMT>
__global__ void k_dequantize(const uint8_t* __restrict__ qs, const uint16_t* __restrict__ d, int64_t nblocks,
                             float* __restrict__ out) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nblocks) return;
    float s = f16_to_f32(d[i]);
    float e[QK];
    if constexpr (FMT == FMT_Q8_0) {
        const uint4* src = reinterpret_cast<const uint4*>(qs + i * QK);
#pragma unroll
        for (int c = 0; c < 2; c++) {
            const uint4 w = src[c];
            const uint32_t ws[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
            for (int j = 0; j < 16; j++) e[16 * c + j] = (float)(int8_t)(ws[j >> 2] >> (8 * (j & 3))) * s;
        }
    } else {
        uint4 w = *reinterpret_cast<const uint4*>(qs + i * 16);
        uint32_t ws[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
        for (int j = 0; j < 16; j++) {
            uint32_t byte = (ws[j >> 2] >> (8 * (j & 3))) & 0xffu;
            e[j] = (float)((int)(byte & 0xf) - 8) * s;
            e[j + 16] = (float)((int)(byte >> 4) - 8) * s;
        }
    }
    float4* o = reinterpret_cast<float4*>(out + i * QK);
#pragma unroll
    for (int j = 0; j < QK / 4; j++) o[j] = make_float4(e[4 * j], e[4 * j + 1], e[4 * j + 2], e[4 * j + 3]);
}

// ---- decode GEMV (m <= GEMV_MAX_M) ---------------------------------------------
//
// One workgroup owns `rows` consecutive weight rows. Phase 1 quantises the MR
// activation rows into LDS (every workgroup repeats this: x is a few KB and
// L2-resident). Phase 2 streams the weight: the (row, block) items of the
// workgroup are a contiguous range of the codes plane, so consecutive lanes
// issue consecutive 16-byte loads (two per q8_0 item); each item's exact
// integer dot is 8 v_dot4_i32_i8 (q4_0: on the unsigned nibbles, minus
// 8 * sum(x codes)), and its scaled term goes to LDS. Phase 3 adds each
// output's terms in block order.

constexpr int GEMV_THREADS = 256;
constexpr int GEMV_MAX_M = 4;

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

__device__ inline int dot_block(uint4 w, const int* __restrict__ xw) {
    // xw: the 32 int8 codes of the block as 8 dwords, natural element order.
    // w dword j holds bytes 4j..4j+3: low nibbles = elements 4j..4j+3, high
    // nibbles = elements 16+4j..16+4j+3.
    int s = 0;
    s = __builtin_amdgcn_sdot4((int)(w.x & 0x0f0f0f0fu), xw[0], s, false);
    s = __builtin_amdgcn_sdot4((int)((w.x >> 4) & 0x0f0f0f0fu), xw[4], s, false);
    s = __builtin_amdgcn_sdot4((int)(w.y & 0x0f0f0f0fu), xw[1], s, false);
    s = __builtin_amdgcn_sdot4((int)((w.y >> 4) & 0x0f0f0f0fu), xw[5], s, false);
    s = __builtin_amdgcn_sdot4((int)(w.z & 0x0f0f0f0fu), xw[2], s, false);
    s = __builtin_amdgcn_sdot4((int)((w.z >> 4) & 0x0f0f0f0fu), xw[6], s, false);
    s = __builtin_amdgcn_sdot4((int)(w.w & 0x0f0f0f0fu), xw[3], s, false);
    s = __builtin_amdgcn_sdot4((int)((w.w >> 4) & 0x0f0f0f0fu), xw[7], s, false);
    return s;
}

__device__ inline int dot_block_q8(const uint4& w0, const uint4& w1, const int* __restrict__ xw) {
    // both operands hold the 32 int8 codes in natural order, 4 per dword
    int s = 0;
    s = __builtin_amdgcn_sdot4((int)w0.x, xw[0], s, false);
    s = __builtin_amdgcn_sdot4((int)w0.y, xw[1], s, false);
    s = __builtin_amdgcn_sdot4((int)w0.z, xw[2], s, false);
    s = __builtin_amdgcn_sdot4((int)w0.w, xw[3], s, false);
    s = __builtin_amdgcn_sdot4((int)w1.x, xw[4], s, false);
    s = __builtin_amdgcn_sdot4((int)w1.y, xw[5], s, false);
    s = __builtin_amdgcn_sdot4((int)w1.z, xw[6], s, false);
    s = __builtin_amdgcn_sdot4((int)w1.w, xw[7], s, false);
    return s;
}

// Phase 1 gives each 32-element block to 8 lanes, a float4 each: lane l of
// the workgroup holds elements 4 (l % 8) .. 4 (l % 8) + 3 of block l / 8 + 32 p
// in pass p, so for one row thread t holds elements 1024p + 4t .. 1024p + 4t + 3.
// The block's amax and code sum are 8-lane DPP reductions (no LDS round
// trip). The RMSNorm prologue's sum of squares uses that partition -- thread
// t adds the squares of its elements in order, then block_sum256 -- which is
// k_rmsnorm's order, so the fused norm reproduces it bit for bit.
//
// Prologues (MR == 1, f32 x only):
//   PRO_RMSNORM  x -> w * (x * r), r = 1/sqrt(sum(x^2)/K + eps)
//   PRO_SILU     x holds [gate | up] (2K floats) -> gate/(1 + exp(-gate)) * up
//   PRO_COMBINE  the row is the attention output h * D + d, merged from the
//                split partials: sum_s O_s 2^(m_s - M) * (1 / sum_s l_s 2^(m_s - M))
// Epilogue: y = acc (+ bias, or + resid: never both); y may alias resid (each
// output's thread reads its residual before writing it), never x. x must be 16-byte aligned.
constexpr int GEMV_HOLD = 4;  // passes of 32 blocks held in registers (K <= 4096 per row at once)
constexpr int GEMV_ONE = 0, GEMV_STREAM = 1, GEMV_PASSES = 2;  // k_gemv's SHAPE

// The best (value, index) over a workgroup of GEMV_THREADS threads, in
// thread 0 (arg_before's order: any pairing gives the same winner).
__device__ inline void block_arg_best(float& v, int& i) {
    __shared__ float sv[GEMV_THREADS / 64];
    __shared__ int si[GEMV_THREADS / 64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        const float ov = __shfl_xor(v, off);
        const int oi = __shfl_xor(i, off);
        if (arg_before(ov, oi, v, i)) {
            v = ov;
            i = oi;
        }
    }
    if (lane == 0) {
        sv[w] = v;
        si[w] = i;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int k = 1; k < GEMV_THREADS / 64; k++)
            if (arg_before(sv[k], si[k], v, i)) {
                v = sv[k];
                i = si[k];
            }
    }
}

// The argmax epilogue after a workgroup's last tile: its best (value, index)
// goes to arg_v/arg_i[workgroup] with plain stores. k_argmax_parts, the next
// launch, reduces them: a kernel boundary is all the ordering the partials
// need. (Reducing them inside this launch, the workgroup drawing the last
// ticket reading the others' partials back, kept the lm_head on the step's
// critical path for the stores' acknowledgement and the ticket's round trip:
// 17.8 us for the C5 lm_head, against 9.0 us without the argmax.)
__device__ inline void gemv_argmax_epilogue(float v, int i, const GemvPro& po) {
    block_arg_best(v, i);
    if (threadIdx.x == 0) {
        po.arg_v[blockIdx.x] = v;
        po.arg_i[blockIdx.x] = i;
    }
}

// One workgroup: the best of `parts` (<= GEMV_ARG_MAX_PARTS) (value, index)
// partials of an n-wide row (argmax's order, arg_before), into state[3], then
// the decode step's advance as k_argmax<true, ...> does. Every load is issued
// at the start: the partials all at once, and the position with the prompt
// token it may pick, so that nothing waits on memory after the reduction.
__global__ __launch_bounds__(GEMV_THREADS) void k_argmax_parts(const float* __restrict__ arg_v,
                                                             const int32_t* __restrict__ arg_i, int parts, int n,
                                                             int32_t* state, int32_t* tokens,
                                                             const int32_t* __restrict__ prompt, int prompt_len,
                                                             int cap) {
    constexpr int PER = GEMV_ARG_MAX_PARTS / GEMV_THREADS;
    static_assert(PER * GEMV_THREADS == GEMV_ARG_MAX_PARTS, "partials per thread");
    int pos = 0, ptok = 0;
    if (threadIdx.x == 0) {
        pos = state[0] + 1;
        if (pos < prompt_len) ptok = prompt[pos];
    }
    float pv[PER];
    int pi[PER];
#pragma unroll
    for (int j = 0; j < PER; j++) {
        const int g = threadIdx.x + j * GEMV_THREADS;
        pv[j] = -INFINITY;
        pi[j] = INT32_MAX;
        if (g < parts) {
            pv[j] = arg_v[g];
            pi[j] = arg_i[g];
        }
    }
    float v = pv[0];
    int i = pi[0];
#pragma unroll
    for (int j = 1; j < PER; j++)
        if (arg_before(pv[j], pi[j], v, i)) {
            v = pv[j];
            i = pi[j];
        }
    block_arg_best(v, i);
    if (threadIdx.x == 0) {
        const int am = i < n ? i : 0;
        state[3] = am;
        llama_commit(state, tokens, pos, pos < prompt_len ? ptok : am, cap);
    }
}

// Epilogue ARG (MR == 1, f32 y; linear_decode_argmax): each workgroup's best
// output of y to po.arg_v/arg_i[workgroup], for k_argmax_parts.
// Epilogue GLU (MR == 1, f32 y, no bias or residual): the weight is
// [gate; up], 2N rows, and y[n] = silu(gate_n) * up_n over the N outputs
// (tn_silu_mul of the two halves, its arithmetic): a tile holds gate rows
// row0 .. row0+rows-1 and the matching up rows, and the thread that sums
// output n's gate row sums its up row too.
// SHAPE (launch_gemv picks):
//   GEMV_ONE     the activation rows fit the registers (MR * nb <= 32 * HOLD
//                blocks) and every workgroup has one row tile: the rows are
//                loaded once, ahead of the weights, in straight-line code,
//                and every weight load is unconditional, so the compiler's
//                waits for the rows do not also wait for the weights (the
//                decode step's GEMVs, latency-bound)
//   GEMV_STREAM  rows held, several tiles per workgroup with the next tile's
//                loads in flight (a streamed weight, bandwidth-bound; these
//                loads stay conditional: the unconditional form takes ten
//                more VGPRs, which costs a wave per SIMD here)
//   GEMV_PASSES  rows too long to hold, loaded in passes (twice with the
//                RMSNorm prologue), several tiles per workgroup
// Separate instantiations rather than branches: in one kernel the compiler
// joins the paths, and the waits on one path then count the other's loads.
template <int FMT, int MR, typename XT, int PRO, bool ARG = false, bool GLU = false, int SHAPE = GEMV_ONE>
__global__ __launch_bounds__(GEMV_THREADS) void k_gemv(const XT* __restrict__ x, int K, int nb,
                                                     const uint8_t* __restrict__ qs,
                                                     const uint16_t* __restrict__ dw, int N, int rows,
                                                     const float* __restrict__ bias, const float* resid, void* y,
                                                     int y_bf16, const GemvPro po) {
    static_assert(PRO == PRO_NONE || (MR == 1 && sizeof(XT) == 4), "prologues take one f32 row");
    static_assert(!ARG || MR == 1, "the argmax epilogue takes one row");
    static_assert(!GLU || (MR == 1 && !ARG), "the SiLU epilogue takes one row");
    constexpr int HOLD = PRO == PRO_COMBINE ? 1 : GEMV_HOLD;
    constexpr int ITEMS = Fmt<FMT>::GEMV_ITEMS, NV = Fmt<FMT>::CODE_BYTES / 16;
    constexpr bool HELD = SHAPE != GEMV_PASSES, ONE = SHAPE == GEMV_ONE;
    extern __shared__ __align__(16) char smem[];
    __shared__ float red[4];
    int* xq = reinterpret_cast<int*>(smem);               // [MR][K/4] packed int8 codes
    float* dxs = reinterpret_cast<float*>(xq + MR * (K / 4));  // [MR][nb]
    int* sxs = reinterpret_cast<int*>(dxs + MR * nb);     // [MR][nb]
    // [2][rows (GLU: 2 rows)][MR][nbp]: term rows padded to 16 bytes for the float4 reads of phase 3
    const int nbp = (nb + 3) & ~3;
    float* terms = reinterpret_cast<float*>(smem + ((MR * K + 8 * MR * nb + 15) & ~15));
    const int tid = threadIdx.x;
    // PRO_COMBINE: the weight items start at the first wave that merges no
    // block of the row (wave 3 at K = 576), so that the merging waves issue
    // only their partial loads and wait on nothing else (a wave's loads
    // complete in order)
    int wt = tid;
    if constexpr (PRO == PRO_COMBINE) {
        const int busy = 8 * (nb < 32 ? nb : 32);  // threads with a block in phase 1 (MR == 1)
        wt = (tid + GEMV_THREADS - (((busy + 63) & ~63) & (GEMV_THREADS - 1))) & (GEMV_THREADS - 1);
    }

    const int ntiles = (N + rows - 1) / rows;
    const int tstride = (int)gridDim.x;
    // two register buffers: the tile being computed and the next one in flight
    // (a third, two tiles ahead, measured slower: fewer resident waves)
    uint4 wv[ITEMS][NV], wn[ITEMS][NV];
    uint16_t dv[ITEMS], dn[ITEMS];
    constexpr int RW = GLU ? 2 : 1;  // weight rows per output
    // GEMV_ONE: the weight loads are unconditional buffer loads, one
    // descriptor per plane over the tile's span; an item past the tile reads
    // at an offset past the descriptor, which returns zero without a memory
    // access. Otherwise they are plain loads of the items that exist.
    constexpr uint32_t OOB = 0x80000000u;  // past every descriptor here (spans < 2^31 bytes)
    constexpr int NT = 2;                  // cache policy: non-temporal, the weights are streamed once
    auto gload = [&](int tile, uint4 (*wr)[NV], uint16_t* dr) {
        const int64_t row0 = (int64_t)tile * rows;
        const int nrows = (int)((N - row0) < rows ? (N - row0) : rows);
        const int total = RW * nrows * nb;
        if constexpr (ONE) {
            // GLU: the tile's up rows sit N rows after its gate rows
            const uint32_t span = (uint32_t)((GLU ? N + nrows : nrows) * nb);
            const buf_rsrc rq = make_rsrc(qs + row0 * nb * (16 * NV), span * (16u * NV));
            const buf_rsrc rd = make_rsrc(dw + row0 * nb, span * 2u);
#pragma unroll
            for (int it = 0; it < ITEMS; it++) {
                const int g0 = wt + it * GEMV_THREADS;
                const int g = (GLU && g0 >= nrows * nb) ? g0 + (N - nrows) * nb : g0;
                const bool on = g0 < total;
                const uint32_t qo = on ? (uint32_t)g * (16u * NV) : OOB, dof = on ? (uint32_t)g * 2u : OOB;
#if __HIP_DEVICE_COMPILE__
#pragma unroll
                for (int v = 0; v < NV; v++)
                    wr[it][v] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rq, qo, 16 * v, NT));
                dr[it] = __builtin_amdgcn_raw_buffer_load_b16(rd, dof, 0, 0);
#else
                (void)rq, (void)rd, (void)qo, (void)dof;
#endif
            }
        } else {
            const uint4* qbase = reinterpret_cast<const uint4*>(qs) + row0 * nb * NV;
            const uint16_t* dbase = dw + row0 * nb;
#pragma unroll
            for (int it = 0; it < ITEMS; it++) {
                int g = wt + it * GEMV_THREADS;
                if (g < total) {
                    // GLU: items past the tile's gate rows are its up rows, N rows on
                    if (GLU && g >= nrows * nb) g += (N - nrows) * nb;
                    // streamed once: a non-temporal load keeps it from evicting x and the terms
#pragma unroll
                    for (int v = 0; v < NV; v++) {
                        const u32x4 t =
                            __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(qbase + g * NV + v));
                        wr[it][v] = make_uint4(t[0], t[1], t[2], t[3]);
                    }
                    dr[it] = dbase[g];
                }
            }
        }
    };
    int tile = (int)blockIdx.x;
    float pre_add = 0.0f;
    // the first tile's weight loads (and this thread's residual or bias for
    // it), in flight during the activation work; unconditional as gload's
    // (the grid never exceeds the tile count, so the first tile exists)
    // the bias or residual of this thread's first output of tile t (output
    // o = tid), an unconditional buffer load: resid and bias are not
    // combined, and with neither the descriptor is empty
    [[maybe_unused]] auto load_add = [&](int t) -> float {
        const int64_t row0 = (int64_t)t * rows;
        const int nrows = (int)((N - row0) < rows ? (N - row0) : rows);
        const int r = tid / MR, mr = tid - r * MR;
        const float* src = bias ? bias : resid;
        const buf_rsrc rb = make_rsrc(src, src ? (uint32_t)((bias ? 1 : MR) * N) * 4u : 0u);
        const uint32_t off = tid < nrows * MR ? (uint32_t)((bias ? 0 : (int64_t)mr * N) + row0 + r) * 4u : OOB;
#if __HIP_DEVICE_COMPILE__
        return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rb, off, 0, 0));
#else
        (void)rb, (void)off;
        return 0.0f;
#endif
    };
    auto first_loads = [&]() {
        if constexpr (ONE) {
            gload(tile, wv, dv);
            pre_add = load_add(tile);
        } else if (tile < ntiles) {  // always true; the branch keeps this shape at 64 VGPRs (66 without)
            gload(tile, wv, dv);
            const int64_t row0 = (int64_t)tile * rows;
            const int nrows = (int)((N - row0) < rows ? (N - row0) : rows);
            if (tid < nrows * MR) {
                const int r = tid / MR, mr = tid - r * MR;
                if (bias) pre_add = bias[row0 + r];
                if (resid) pre_add = resid[(int64_t)mr * N + row0 + r];  // resid and bias are not combined
            }
        }
    };

    // phase 1: Q8_0 of the MR activation rows (after the prologue)
    {
        const int g8 = tid & 7, slot = tid >> 3;
        const int nblk = MR * nb, npass = (nblk + 31) / 32;
        // a row that fits the registers is loaded before the weights, whose
        // loads would otherwise stand in front of it in the memory pipeline
        // (the merge of the attention partials, PRO_COMBINE, after them: its
        // waves hold no weight items)
        (void)npass;
        float4 xv[HOLD], av[HOLD];  // the row, and the prologue's second operand
        int ns = 0;
        if constexpr (PRO == PRO_COMBINE) {
            int len = *po.len;
            len = len < 0 ? 0 : (len > po.cap ? po.cap : len);
            ns = (len + STEP_SPLIT - 1) / STEP_SPLIT;
            ns = ns < po.nsplit ? ns : po.nsplit;
        }
        // PRO_COMBINE: row block blk merged over the splits. Every split's
        // (m, l) and O piece is in flight at once, read before the length is
        // known (splits past it are not used). The loads are unconditional --
        // a split index past the launch's count reads the last split's row
        // again, a block past the row's reads its last block, and neither is
        // used -- so the compiler counts the loads in flight exactly.
        auto merge_block = [&](int blk) -> float4 {
            const int bc = blk < nblk ? blk : nblk - 1;
            const int o32 = bc * QK + 4 * g8;  // MR == 1: the element offset in the row
            const int h = o32 >> po.head_shift, d = o32 & ((1 << po.head_shift) - 1);
            // one descriptor per plane: a lane's (head, column) is its vector
            // offset and a split's row the scalar one
            const uint32_t rows = (uint32_t)(K >> po.head_shift) * (uint32_t)po.nsplit;
            const buf_rsrc rml = make_rsrc(po.part_ml, rows * 8u);
            const buf_rsrc ro = make_rsrc(po.part_o, rows * (uint32_t)po.head_dim * 4u);
            const uint32_t vml = (uint32_t)(h * po.nsplit) * 8u;
            const uint32_t vo = ((uint32_t)(h * po.nsplit) * (uint32_t)po.head_dim + (uint32_t)d) * 4u;
            u32x2 mlr[STEP_MAX_SPLITS] = {};
            u32x4 orr[STEP_MAX_SPLITS] = {};
#if __HIP_DEVICE_COMPILE__
#pragma unroll
            for (int sp = 0; sp < STEP_MAX_SPLITS; sp++) {
                const uint32_t spc = (uint32_t)(sp < po.nsplit ? sp : po.nsplit - 1);
                mlr[sp] = __builtin_amdgcn_raw_buffer_load_b64(rml, vml, spc * 8u, 0);
            }
#pragma unroll
            for (int sp = 0; sp < STEP_MAX_SPLITS; sp++) {
                const uint32_t spc = (uint32_t)(sp < po.nsplit ? sp : po.nsplit - 1);
                orr[sp] = __builtin_amdgcn_raw_buffer_load_b128(ro, vo, spc * (uint32_t)po.head_dim * 4u, 0);
            }
#else
            (void)rml, (void)ro, (void)vml, (void)vo;
#endif
            // every load issued before any result is used
            __builtin_amdgcn_sched_barrier(0);
            float2 ml[STEP_MAX_SPLITS];
            float4 o4[STEP_MAX_SPLITS];
#pragma unroll
            for (int sp = 0; sp < STEP_MAX_SPLITS; sp++) {
                ml[sp] = make_float2(__uint_as_float(mlr[sp][0]), __uint_as_float(mlr[sp][1]));
                o4[sp] = make_float4(__uint_as_float(orr[sp][0]), __uint_as_float(orr[sp][1]),
                                     __uint_as_float(orr[sp][2]), __uint_as_float(orr[sp][3]));
            }
            float mm = -INFINITY;
#pragma unroll
            for (int sp = 0; sp < STEP_MAX_SPLITS; sp++)
                if (sp < ns) mm = fmaxf(mm, ml[sp].x);
            const float mu = (mm == -INFINITY) ? 0.0f : mm;
            float tl = 0.0f;
            float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
            // One wave issues this whole merge, so its instruction count is
            // its time: the hardware exp2 (a factor below 2^-126 becomes 0,
            // where the library's would keep a subnormal), and one
            // reciprocal of the sum for the four columns.
#pragma unroll
            for (int sp = 0; sp < STEP_MAX_SPLITS; sp++) {
                if (sp < ns) {
                    const float f = __builtin_amdgcn_exp2f(ml[sp].x - mu);
                    tl = tl + ml[sp].y * f;
                    acc.x = acc.x + o4[sp].x * f;
                    acc.y = acc.y + o4[sp].y * f;
                    acc.z = acc.z + o4[sp].z * f;
                    acc.w = acc.w + o4[sp].w * f;
                }
            }
            const float inv = 1.0f / tl;
            return make_float4(acc.x * inv, acc.y * inv, acc.z * inv, acc.w * inv);
        };
        auto load_passes = [&](int p0) {
#pragma unroll
            for (int u = 0; u < HOLD; u++) {
                const int blk = (p0 + u) * 32 + slot;
                if constexpr (PRO == PRO_COMBINE) {
                    // waves with no block of the row skip it
                    if (__builtin_amdgcn_readfirstlane(blk) < nblk) xv[u] = merge_block(blk);
                } else if (blk < nblk) {
                    const int mr = blk / nb, b = blk - mr * nb;
                    const int64_t off = (int64_t)mr * K + b * QK + 4 * g8;
                    if constexpr (sizeof(XT) == 4) {
                        xv[u] = *reinterpret_cast<const float4*>(x + off);
                    } else {
                        const uint2 h = *reinterpret_cast<const uint2*>(x + off);
                        xv[u] = make_float4(bf16_to_f32((uint16_t)(h.x & 0xffffu)), bf16_to_f32((uint16_t)(h.x >> 16)),
                                            bf16_to_f32((uint16_t)(h.y & 0xffffu)), bf16_to_f32((uint16_t)(h.y >> 16)));
                    }
                    if constexpr (PRO == PRO_RMSNORM) av[u] = *reinterpret_cast<const float4*>(po.w + off);
                    if constexpr (PRO == PRO_SILU)
                        av[u] = *reinterpret_cast<const float4*>(reinterpret_cast<const float*>(x) + K + off);
                }
            }
        };
        if constexpr (PRO == PRO_COMBINE) {
            first_loads();
            if constexpr (HELD) load_passes(0);
        } else {
            if constexpr (HELD) load_passes(0);
            first_loads();
        }
        // thread t's squares in order (k_rmsnorm's), over the passes held in xv
        auto ss_pass = [&](int p0, float& ss) {
#pragma unroll
            for (int u = 0; u < HOLD; u++) {
                if ((p0 + u) * 32 + slot < nblk) {
                    ss = ss + xv[u].x * xv[u].x;
                    ss = ss + xv[u].y * xv[u].y;
                    ss = ss + xv[u].z * xv[u].z;
                    ss = ss + xv[u].w * xv[u].w;
                }
            }
        };
        int8_t* xb = reinterpret_cast<int8_t*>(xq);
        auto q8_pass = [&](int p0, float r) {
#pragma unroll
            for (int u = 0; u < HOLD; u++) {
                const int blk = (p0 + u) * 32 + slot;
                if (blk < nblk) {  // uniform over the block's 8 lanes
                    float e[4] = {xv[u].x, xv[u].y, xv[u].z, xv[u].w};
                    const float o[4] = {av[u].x, av[u].y, av[u].z, av[u].w};
                    float amax = 0.0f;
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        if constexpr (PRO == PRO_RMSNORM) e[i] = o[i] * (e[i] * r);
                        if constexpr (PRO == PRO_SILU) e[i] = (e[i] / (1.0f + expf(-e[i]))) * o[i];
                        amax = fmaxf(amax, fabsf(e[i]));
                    }
                    // BlockQ8_0::from_float (k_quants.rs:676-705)
                    amax = group8_max(amax);
                    const float d = amax / 127.0f;
                    const float id = (d != 0.0f) ? 1.0f / d : 0.0f;
                    uint32_t wd = 0;
                    int sq = 0;
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const int q = sat_i8(roundf(e[i] * id));
                        sq += q;
                        wd |= ((uint32_t)q & 0xffu) << (8 * i);
                    }
                    sq = group8_sum(sq);
                    reinterpret_cast<uint32_t*>(xb)[blk * 8 + g8] = wd;  // blocks of all rows are contiguous
                    if (g8 == 0) {
                        dxs[blk] = f16_round_hw(d);  // d is never NaN: amax ignores NaN
                        sxs[blk] = sq;
                    }
                }
            }
        };
        if constexpr (HELD) {
            // the held row in straight-line code: the waits for the row count
            // only the loads issued after it
            float r = 0.0f;
            if constexpr (PRO == PRO_RMSNORM) {
                float ss = 0.0f;
                ss_pass(0, ss);
                r = rms_scale(block_sum256(ss, red), K, po.eps);
            }
            q8_pass(0, r);
        } else {
            float r = 0.0f;
            if constexpr (PRO == PRO_RMSNORM) {
                float ss = 0.0f;
                for (int p0 = 0; p0 < npass; p0 += HOLD) {
                    load_passes(p0);
                    ss_pass(p0, ss);
                }
                r = rms_scale(block_sum256(ss, red), K, po.eps);
            }
            for (int p0 = 0; p0 < npass; p0 += HOLD) {
                load_passes(p0);
                q8_pass(p0, r);
            }
        }
    }
    __syncthreads();

    // phase 2/3, persistent over row tiles: the next tile's weight loads are in
    // flight while this tile's terms are computed and summed; the terms live
    // in two LDS buffers, so one barrier per tile suffices
    float best_v = -INFINITY;  // ARG: this thread's best output so far
    int best_i = INT32_MAX;    // loses every tie against a real output
    for (int buf = 0; tile < ntiles; tile += tstride, buf ^= 1) {
        // GEMV_ONE: this is the workgroup's only tile
        if constexpr (!ONE) {
            if (tile + tstride < ntiles) gload(tile + tstride, wn, dn);
        }
        const int64_t row0 = (int64_t)tile * rows;
        const int nrows = (int)((N - row0) < rows ? (N - row0) : rows);
        const int total = RW * nrows * nb;
        float* tb = terms + buf * RW * rows * MR * nbp;
#pragma unroll
        for (int it = 0; it < ITEMS; it++) {
            const int g = wt + it * GEMV_THREADS;
            if (g < total) {
                const int r = g / nb, b = g - r * nb;
                const float dwf = f16_bits_hw(dv[it]);
#pragma unroll
                for (int mr = 0; mr < MR; mr++) {
                    const int* xw = xq + mr * (K / 4) + b * 8;
                    int s;
                    if constexpr (FMT == FMT_Q8_0)
                        s = dot_block_q8(wv[it][0], wv[it][1], xw);
                    else
                        s = dot_block(wv[it][0], xw) - 8 * sxs[mr * nb + b];
                    float t = (float)s * dwf;
                    t = t * dxs[mr * nb + b];
                    tb[(r * MR + mr) * nbp + b] = t;
                }
            }
        }
        __syncthreads();
        // each output's terms in block order, read 16 at a time
        // one row's terms in block order
        auto ordered_sum = [&](const float* tr) {
            float acc = 0.0f;
            int b = 0;
            for (; b + 16 <= nb; b += 16) {
                float4 t4[4];
#pragma unroll
                for (int j = 0; j < 4; j++) t4[j] = reinterpret_cast<const float4*>(tr + b)[j];
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    acc = acc + t4[j].x;
                    acc = acc + t4[j].y;
                    acc = acc + t4[j].z;
                    acc = acc + t4[j].w;
                }
            }
            for (; b + 4 <= nb; b += 4) {
                const float4 t4 = *reinterpret_cast<const float4*>(tr + b);
                acc = acc + t4.x;
                acc = acc + t4.y;
                acc = acc + t4.z;
                acc = acc + t4.w;
            }
            for (; b < nb; b++) acc = acc + tr[b];
            return acc;
        };
        auto out_row = [&](int o, float add) {
            const int r = o / MR, mr = o - r * MR;
            const int64_t n = row0 + r;
            float acc = ordered_sum(tb + (r * MR + mr) * nbp);
            if constexpr (GLU) {
                // silu(gate) * up, tn_silu_mul's arithmetic
                const float up = ordered_sum(tb + (nrows + r) * nbp);
                acc = (acc / (1.0f + expf(-acc))) * up;
            }
            if (bias || resid) acc = acc + add;
            if constexpr (ARG) {
                if (arg_before(acc, (int)n, best_v, best_i)) {
                    best_v = acc;
                    best_i = (int)n;
                }
            }
            if (y_bf16)
                reinterpret_cast<uint16_t*>(y)[(int64_t)mr * N + n] = bf16_out(acc);
            else
                reinterpret_cast<float*>(y)[(int64_t)mr * N + n] = acc;
        };
        if constexpr (ONE) {
            // the thread's first output outside the loop: its add was loaded
            // unconditionally, before the weights, and its wait counts them out
            if (tid < nrows * MR) out_row(tid, pre_add);
            for (int o = tid + GEMV_THREADS; o < nrows * MR; o += GEMV_THREADS) {
                const int r = o / MR, mr = o - r * MR;
                const int64_t n = row0 + r;
                out_row(o, bias ? bias[n] : resid ? resid[(int64_t)mr * N + n] : 0.0f);
            }
        } else {
            for (int o = tid; o < nrows * MR; o += GEMV_THREADS) {
                const int r = o / MR, mr = o - r * MR;
                const int64_t n = row0 + r;
                float add = pre_add;
                if (tile != (int)blockIdx.x || o != tid)
                    add = bias ? bias[n] : resid ? resid[(int64_t)mr * N + n] : 0.0f;
                out_row(o, add);
            }
        }
        if constexpr (ONE) break;  // the launch gives every workgroup one tile
#pragma unroll
        for (int it = 0; it < ITEMS; it++) {
#pragma unroll
            for (int v = 0; v < NV; v++) wv[it][v] = wn[it][v];
            dv[it] = dn[it];
        }
    }
    if constexpr (ARG) gemv_argmax_epilogue(best_v, best_i, po);
}

tn_status check_weight(const char* op, const char* fmt, int64_t n, int64_t k) {
    if (n < 0 || k <= 0 || k % QK != 0) {
        char buf[384];
        std::snprintf(buf, sizeof buf,
                      "%s: %s stores 32 elements per block, so it must have their last dim divisible by "
                      "block size -- got %lld, which is not a multiple of 32 (shape [%lld, %lld])",
                      op, fmt, (long long)k, (long long)n, (long long)k);
        return fail(TN_ENOTIMPL, buf);
    }
    if (n * (k / QK) > ((int64_t)1 << 40)) return fail(TN_EVALUE, std::string(op) + ": weight too large");
    return TN_OK;
}

template <int FMT, int MR, typename XT, int PRO = PRO_NONE, bool ARG = false, bool GLU = false>
tn_status launch_gemv(hipStream_t st, const XT* x, int K, const uint8_t* qs, const uint16_t* dw, int N,
                      const float* bias, void* y, int y_bf16, const float* resid = nullptr,
                      const GemvPro& po = GemvPro(), unsigned* grid_out = nullptr) {
    const int nb = K / QK;
    constexpr int ITEMS = Fmt<FMT>::GEMV_ITEMS;
    // rows per tile: as many as ITEMS items per thread allow, but no more
    // than it takes to give every CU a tile of a small matrix
    constexpr int RW = GLU ? 2 : 1;  // weight rows per output (GLU: gate and up)
    int rows = (GEMV_THREADS * ITEMS) / (RW * nb);
    const int spread = (int)cdiv(N, 256);
    if (rows > spread) rows = spread;
    if (rows < 1) rows = 1;
    if (rows > N) rows = N;
    // two term buffers (double-buffered across tiles)
    if (bias && resid) return fail(TN_EINVAL, "quantised GEMV: bias and residual together are not supported");
    const int nbp = (nb + 3) & ~3;
    auto lds_of = [&](int r) {
        return (((size_t)MR * K + (size_t)MR * nb * 8 + 15) & ~(size_t)15) + 2 * (size_t)RW * r * MR * nbp * 4;
    };
    size_t lds = lds_of(rows);
    while (rows > 1 && lds > 64 * 1024) {
        rows >>= 1;
        lds = lds_of(rows);
    }
    if (lds > 64 * 1024) return TN_ENOTIMPL;  // caller falls through to the GEMM path
    // (row, block) items must fit ITEMS per thread
    if ((int64_t)RW * rows * nb > GEMV_THREADS * ITEMS) return TN_ENOTIMPL;
    if (GLU && (bias || resid)) return fail(TN_EINVAL, "quantised GEMV: the SiLU epilogue takes no bias or residual");
    const int64_t ntiles = cdiv(N, rows);
    // persistent: exactly as many workgroups as the device holds at once (a
    // workgroup that had to wait for a slot would start its whole share of
    // tiles late). SHAPE: the activation rows held in registers (k_gemv's
    // HOLD passes of 32 blocks), and GEMV_ONE when the resident workgroups
    // cover the tiles and its buffer descriptors (a tile's weight span, GLU:
    // N + rows rows; the bias or residual rows) stay below 2^31 bytes
    const bool held = MR * nb <= 32 * (PRO == PRO_COMBINE ? 1 : GEMV_HOLD);
    const bool spans = (int64_t)(GLU ? N + rows : rows) * nb * Fmt<FMT>::CODE_BYTES < (int64_t(1) << 31) &&
                       (int64_t)MR * N * 4 < (int64_t(1) << 31);
    auto kern_of = [](int shape) -> const void* {
        return shape == GEMV_ONE      ? reinterpret_cast<const void*>(&k_gemv<FMT, MR, XT, PRO, ARG, GLU, GEMV_ONE>)
               : shape == GEMV_STREAM ? reinterpret_cast<const void*>(&k_gemv<FMT, MR, XT, PRO, ARG, GLU, GEMV_STREAM>)
                                      : reinterpret_cast<const void*>(&k_gemv<FMT, MR, XT, PRO, ARG, GLU, GEMV_PASSES>);
    };
    const int64_t cap = ARG ? GEMV_ARG_MAX_PARTS : INT32_MAX;
    int shape = held ? GEMV_ONE : GEMV_PASSES, resident = 0;
    tn_status s = resident_workgroups(kern_of(shape), GEMV_THREADS, lds, &resident);
    if (s != TN_OK) return s;
    if (shape == GEMV_ONE && (ntiles > resident || ntiles > cap || !spans)) {
        shape = GEMV_STREAM;
        s = resident_workgroups(kern_of(shape), GEMV_THREADS, lds, &resident);
        if (s != TN_OK) return s;
    }
    unsigned grid = (unsigned)(ntiles < resident ? ntiles : resident);
    if (grid > (unsigned)cap) grid = (unsigned)cap;
#define TN_GEMV(SH)                                                                                                   \
    hipLaunchKernelGGL((k_gemv<FMT, MR, XT, PRO, ARG, GLU, SH>), dim3(grid), dim3(GEMV_THREADS), lds, st, x, K, nb, qs, \
                       dw, N, rows, bias, resid, y, y_bf16, po)
    if (shape == GEMV_ONE) TN_GEMV(GEMV_ONE);
    else if (shape == GEMV_STREAM) TN_GEMV(GEMV_STREAM);
    else TN_GEMV(GEMV_PASSES);
#undef TN_GEMV
    TN_LAUNCHED();
    if (grid_out) *grid_out = grid;
    return TN_OK;
}

template <int FMT, typename XT>
tn_status linear_impl(hipStream_t st, const XT* x, int64_t m, int64_t k, const uint8_t* qs, const uint16_t* d,
                      int64_t n, const float* bias, void* y, int y_bf16) {
    if (m == 0 || n == 0) return TN_OK;
    const int nb = (int)(k / QK);
    const size_t ysz = y_bf16 ? 2 : 4;
    const QGemmArgs rows{FMT, x, sizeof(XT) == 2, m, k, XM_ROWS, 0, qs, d, n, bias, y, y_bf16, nullptr};
    // Two to four rows: the GEMV's time grows with the work (0.13 us per
    // million of m n k beyond its launch), the GEMM's with k alone (about 7 us +
    // 2.7 us per 1024 of k up to n = 16384), so a large product goes there: [4, 4096]
    // x [14336, 4096] 33.9 -> 17.8 us, three rows 25.2 -> 18.0, two 19.8 -> 17.5,
    // [4, 1024] x [16000, 1024] 9.9 -> 8.6. Short rows stay ([3, 576] x [49152, 576]:
    // 8.7, and 10.4 there). It needs the stream's workspace; a capture that could
    // not grow it keeps the GEMV.
    if (m >= 2 && m <= GEMV_MAX_M && k >= 1024 && m * n > 16384 + 44000000 / k &&
        reinterpret_cast<uintptr_t>(qs) % 16 == 0) {
        void* ws = nullptr;
        TN_TRY(workspace_or_none(st, qgemm_workspace(rows), &ws));
        if (ws) return qgemm_launch(st, rows);
    }
    // the GEMV reads x in 16-byte pieces; an unaligned x takes the GEMM
    if (m <= GEMV_MAX_M && nb <= GEMV_THREADS * Fmt<FMT>::GEMV_ITEMS && reinterpret_cast<uintptr_t>(x) % 16 == 0) {
        // decode: GEMV in chunks of up to 4 rows of x (a row's result does not
        // depend on the chunking: every output is the same recurrence)
        int64_t r = 0;
        tn_status s = TN_OK;
        while (r < m && s == TN_OK) {
            const int64_t c = (m - r) >= 4 ? 4 : (m - r);
            const XT* xr = x + r * k;
            void* yr = static_cast<char*>(y) + r * n * ysz;
            switch (c) {
                case 4: s = launch_gemv<FMT, 4, XT>(st, xr, (int)k, qs, d, (int)n, bias, yr, y_bf16); break;
                case 3: s = launch_gemv<FMT, 3, XT>(st, xr, (int)k, qs, d, (int)n, bias, yr, y_bf16); break;
                case 2: s = launch_gemv<FMT, 2, XT>(st, xr, (int)k, qs, d, (int)n, bias, yr, y_bf16); break;
                default: s = launch_gemv<FMT, 1, XT>(st, xr, (int)k, qs, d, (int)n, bias, yr, y_bf16); break;
            }
            r += c;
        }
        if (s == TN_OK) return TN_OK;
        if (s != TN_ENOTIMPL) return s;
        // too large for the LDS-resident GEMV: the GEMM, which computes the
        // identical recurrence
    }
    return qgemm_launch(st, rows);
}

// The codec entry points of one format.
template <int FMT>
tn_status codec_launch(const char* op, void* stream, int64_t n, int64_t k, int kind, const void* in0,
                       const void* in1, void* out0, void* out1) {
    tn_status s = check_weight(op, Fmt<FMT>::name, n, k);
    if (s != TN_OK) return s;
    const int64_t nblocks = n * (k / QK);
    if (!nblocks) return TN_OK;
    if (!in0 || !out0 || (kind >= 2 ? !in1 : !out1)) return fail(TN_EVALUE, std::string(op) + ": null pointer");
    const dim3 grid((unsigned)cdiv(nblocks, 256));
    hipStream_t st = (hipStream_t)stream;
    switch (kind) {
        case 0:  // blob -> planes
            hipLaunchKernelGGL(k_from_blob<FMT>, grid, dim3(256), 0, st, static_cast<const uint8_t*>(in0), nblocks,
                               static_cast<uint8_t*>(out0), static_cast<uint16_t*>(out1));
            break;
        case 1:  // f32 -> planes
            hipLaunchKernelGGL(k_quantize_w<FMT>, grid, dim3(256), 0, st, static_cast<const float*>(in0), nblocks,
                               static_cast<uint8_t*>(out0), static_cast<uint16_t*>(out1));
            break;
        case 2:  // planes -> blob
            hipLaunchKernelGGL(k_to_blob<FMT>, grid, dim3(256), 0, st, static_cast<const uint8_t*>(in0),
                               static_cast<const uint16_t*>(in1), nblocks, static_cast<uint8_t*>(out0));
            break;
        default:  // planes -> f32
            hipLaunchKernelGGL(k_dequantize<FMT>, grid, dim3(256), 0, st, static_cast<const uint8_t*>(in0),
                               static_cast<const uint16_t*>(in1), nblocks, static_cast<float*>(out0));
            break;
    }
    TN_LAUNCHED();
    return TN_OK;
}

template <int FMT>
tn_status linear_entry(void* stream, const void* x, int x_dtype, int64_t m, int64_t k, const uint8_t* qs,
                       const uint16_t* d, int64_t n, const float* bias, void* y, int y_dtype) {
    const char* OP = "torch._C._quantized_linear";
    if (x_dtype != TN_F32 && x_dtype != TN_BF16)
        return fail(TN_ENOTIMPL, std::string(OP) +
                                     ": the activation must be float32 (or bfloat16, widened exactly in-kernel) "
                                     "on the hip device");
    if (y_dtype != TN_F32 && y_dtype != TN_BF16)
        return fail(TN_ENOTIMPL, std::string(OP) + ": the output must be float32 or bfloat16");
    if (k <= 0 || k % QK != 0 || m < 0 || n < 0) {
        char buf[256];
        std::snprintf(buf, sizeof buf, "%s: mat1 and mat2 shapes cannot be multiplied ([%lld, %lld] and %lldx%lld)",
                      OP, (long long)m, (long long)k, (long long)k, (long long)n);
        return fail(TN_EINVAL, buf);
    }
    if (m > 0 && n > 0 && (!x || !qs || !d || !y)) return fail(TN_EVALUE, std::string(OP) + ": null pointer");
    hipStream_t st = (hipStream_t)stream;
    const int yb = y_dtype == TN_BF16;
    if (x_dtype == TN_F32)
        return linear_impl<FMT, float>(st, static_cast<const float*>(x), m, k, qs, d, n, bias, y, yb);
    return linear_impl<FMT, uint16_t>(st, static_cast<const uint16_t*>(x), m, k, qs, d, n, bias, y, yb);
}

}  // namespace

// One activation row through a q4_0 linear for the decode step, with the
// step's neighbouring elementwise ops fused in (see k_gemv): bit-identical to
// running tn_rmsnorm / tn_silu_mul, then tn_q4_0_linear, then tn_add.
tn_status linear_decode(hipStream_t st, const float* x, int64_t k, int pro, const GemvPro& po, const uint8_t* qs,
                        const uint16_t* d, int64_t n, const float* resid, float* y) {
    tn_status s = check_weight("linear_decode", "q4_0", n, k);
    if (s != TN_OK) return s;
    if (k > LINEAR_DECODE_MAX_K || n > INT32_MAX) return fail(TN_ENOTIMPL, "linear_decode: shape too large");
    if (n == 0) return TN_OK;
    switch (pro) {
        case PRO_RMSNORM:
            if (po.glu)
                s = launch_gemv<FMT_Q4_0, 1, float, PRO_RMSNORM, false, true>(st, x, (int)k, qs, d, (int)n, nullptr, y, 0,
                                                                             resid, po);
            else
                s = launch_gemv<FMT_Q4_0, 1, float, PRO_RMSNORM>(st, x, (int)k, qs, d, (int)n, nullptr, y, 0, resid, po);
            break;
        case PRO_SILU: s = launch_gemv<FMT_Q4_0, 1, float, PRO_SILU>(st, x, (int)k, qs, d, (int)n, nullptr, y, 0, resid, po); break;
        case PRO_COMBINE:
            // head_dim a power of two (the merge addresses by shifts), at least a 4-column piece
            if (po.head_dim < 4 || po.head_dim != (1 << po.head_shift) || k % po.head_dim != 0 || po.nsplit < 1 ||
                po.nsplit > STEP_MAX_SPLITS || !po.part_o || !po.part_ml || !po.len)
                return fail(TN_EINVAL, "linear_decode: bad attention partials");
            s = launch_gemv<FMT_Q4_0, 1, float, PRO_COMBINE>(st, po.part_o, (int)k, qs, d, (int)n, nullptr, y, 0, resid, po);
            break;
        default: s = launch_gemv<FMT_Q4_0, 1, float, PRO_NONE>(st, x, (int)k, qs, d, (int)n, nullptr, y, 0, resid, po); break;
    }
    if (s == TN_ENOTIMPL) return fail(TN_ENOTIMPL, "linear_decode: the activation row does not fit the GEMV");
    return s;
}

tn_status linear_decode_argmax(hipStream_t st, const float* x, int64_t k, const GemvPro& po, const uint8_t* qs,
                               const uint16_t* d, int64_t n, float* y) {
    tn_status s = check_weight("linear_decode_argmax", "q4_0", n, k);
    if (s != TN_OK) return s;
    if (k > LINEAR_DECODE_MAX_K || n > INT32_MAX || n < 1) return TN_ENOTIMPL;
    if (!po.arg_v || !po.arg_i || !po.state || !po.tokens || (po.prompt_len > 0 && !po.prompt))
        return fail(TN_EINVAL, "linear_decode_argmax: missing argmax operands");
    unsigned parts = 0;
    s = launch_gemv<FMT_Q4_0, 1, float, PRO_RMSNORM, true>(st, x, (int)k, qs, d, (int)n, nullptr, y, 0, nullptr, po,
                                                           &parts);
    if (s != TN_OK) return s;
    hipLaunchKernelGGL(k_argmax_parts, dim3(1), dim3(GEMV_THREADS), 0, st, po.arg_v, po.arg_i, (int)parts, (int)n,
                       po.state, po.tokens, po.prompt, po.prompt_len, po.cap);
    TN_LAUNCHED();
    return TN_OK;
}

// A prompt's projection through the q4 GEMM, its input in one of the
// prepass's layouts and the residual added in its epilogue.
tn_status linear_prefill(hipStream_t st, const float* x, int64_t m, int64_t k, int xm, int hd, const uint8_t* qs,
                         const uint16_t* d, int64_t n, const float* resid, float* y) {
    tn_status s = check_weight("linear_prefill", "q4_0", n, k);
    if (s != TN_OK) return s;
    if (m == 0 || n == 0) return TN_OK;
    if (reinterpret_cast<uintptr_t>(x) % 16 != 0) return fail(TN_EINVAL, "linear_prefill: x must be 16-byte aligned");
    if (xm == XM_HEADS && (hd <= 0 || hd % QK != 0 || k % hd != 0))
        return fail(TN_EINVAL, "linear_prefill: the head dim must divide the row and be a multiple of 32");
    return qgemm_launch(st, QGemmArgs{FMT_Q4_0, x, 0, m, k, xm, hd, qs, d, n, nullptr, y, 0, resid});
}

}  // namespace tn

using namespace tn;

extern "C" {

tn_status tn_q4_0_from_blob(void* stream, const uint8_t* blob, int64_t n, int64_t k, uint8_t* qs, uint16_t* d) {
    return codec_launch<FMT_Q4_0>("torch._C._quantized_to", stream, n, k, 0, blob, nullptr, qs, d);
}

tn_status tn_q4_0_to_blob(void* stream, const uint8_t* qs, const uint16_t* d, int64_t n, int64_t k, uint8_t* blob) {
    return codec_launch<FMT_Q4_0>("torch._C._quantized_blob", stream, n, k, 2, qs, d, blob, nullptr);
}

tn_status tn_q4_0_quantize(void* stream, const float* w, int64_t n, int64_t k, uint8_t* qs, uint16_t* d) {
    return codec_launch<FMT_Q4_0>("torch._C._quantize", stream, n, k, 1, w, nullptr, qs, d);
}

tn_status tn_q4_0_dequantize(void* stream, const uint8_t* qs, const uint16_t* d, int64_t n, int64_t k, float* out) {
    return codec_launch<FMT_Q4_0>("torch._C._dequantize", stream, n, k, 3, qs, d, out, nullptr);
}

tn_status tn_q8_0_from_blob(void* stream, const uint8_t* blob, int64_t n, int64_t k, int8_t* qs, uint16_t* d) {
    return codec_launch<FMT_Q8_0>("torch._C._quantized_to", stream, n, k, 0, blob, nullptr, qs, d);
}

tn_status tn_q8_0_to_blob(void* stream, const int8_t* qs, const uint16_t* d, int64_t n, int64_t k, uint8_t* blob) {
    return codec_launch<FMT_Q8_0>("torch._C._quantized_blob", stream, n, k, 2, qs, d, blob, nullptr);
}

tn_status tn_q8_0_quantize(void* stream, const float* w, int64_t n, int64_t k, int8_t* qs, uint16_t* d) {
    return codec_launch<FMT_Q8_0>("torch._C._quantize", stream, n, k, 1, w, nullptr, qs, d);
}

tn_status tn_q8_0_dequantize(void* stream, const int8_t* qs, const uint16_t* d, int64_t n, int64_t k, float* out) {
    return codec_launch<FMT_Q8_0>("torch._C._dequantize", stream, n, k, 3, qs, d, out, nullptr);
}

tn_status tn_q4_0_linear_decode(void* stream, const float* x, int64_t k, int prologue, const float* prologue_w,
                                double eps, const uint8_t* qs, const uint16_t* d, int64_t n, const float* resid,
                                float* y) {
    const char* op = "q4_0_linear_decode";
    if (prologue != TN_PRO_NONE && prologue != TN_PRO_RMSNORM && prologue != TN_PRO_SILU &&
        prologue != TN_PRO_RMSNORM_SILU)
        return fail(TN_EINVAL, std::string(op) + ": unknown prologue");
    if (k <= 0 || n < 0) return fail(TN_EINVAL, std::string(op) + ": bad sizes");
    const bool glu = prologue == TN_PRO_RMSNORM_SILU;
    if (glu && resid) return fail(TN_EINVAL, std::string(op) + ": the SiLU epilogue takes no residual");
    if (n == 0) return TN_OK;
    if (!x || !qs || !d || !y || ((prologue == TN_PRO_RMSNORM || glu) && !prologue_w))
        return fail(TN_EVALUE, std::string(op) + ": null pointer");
    // y is written while other workgroups still read x
    const char* xb = reinterpret_cast<const char*>(x);
    const char* yb = reinterpret_cast<const char*>(y);
    const int64_t xlen = (prologue == TN_PRO_SILU ? 2 * k : k) * 4;
    if (yb < xb + xlen && xb < yb + n * 4) return fail(TN_EINVAL, std::string(op) + ": y overlaps x");
    if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(prologue_w)) % 16 != 0)
        return fail(TN_EINVAL, std::string(op) + ": x and prologue_w must be 16-byte aligned");
    static_assert(TN_PRO_NONE == PRO_NONE && TN_PRO_RMSNORM == PRO_RMSNORM && TN_PRO_SILU == PRO_SILU, "prologues");
    GemvPro po;
    po.w = prologue_w;
    po.eps = (float)eps;
    po.glu = glu ? 1 : 0;
    return linear_decode((hipStream_t)stream, x, k, glu ? PRO_RMSNORM : prologue, po, qs, d, n, resid, y);
}

tn_status tn_q4_0_linear(void* stream, const void* x, int x_dtype, int64_t m, int64_t k, const uint8_t* qs,
                         const uint16_t* d, int64_t n, const float* bias, void* y, int y_dtype) {
    return linear_entry<FMT_Q4_0>(stream, x, x_dtype, m, k, qs, d, n, bias, y, y_dtype);
}

tn_status tn_q8_0_linear(void* stream, const void* x, int x_dtype, int64_t m, int64_t k, const int8_t* qs,
                         const uint16_t* d, int64_t n, const float* bias, void* y, int y_dtype) {
    return linear_entry<FMT_Q8_0>(stream, x, x_dtype, m, k, reinterpret_cast<const uint8_t*>(qs), d, n, bias, y,
                                  y_dtype);
}

}  // extern "C"
