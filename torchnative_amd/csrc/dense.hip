// The dense "quantised" formats f32 / f16 / bf16 and the dense linear.
//
// `_quantize(t, "f32" | "f16" | "bf16")` stores the weight element by element
// (candle k_quants.rs:2778-2910: GgmlType for f32 copies, for f16 and bf16
// narrows with half's round-to-nearest-even), and `_quantized_linear` on such
// a weight is the exactness control: QMatMul::from_arc widens it to f32 up
// front and takes a plain matmul (candle quantized/mod.rs:836-852), so the
// call must give exactly the bits of the dense linear on the widened weight
// (quant.rs:273-279). Here both go through the same kernels (k_dense_lds,
// k_dense_any, k_dense_valu), whose every output is one fixed chain: acc = 0, then acc = fma(x[k], w[k], acc)
// for k = 0, 1, ..., K-1, then acc + bias (the addmm that nn.Linear's bias
// branch emits, aten.rs:9686-9700, adds the bias once after the product).
// The chain does not depend on the tiling, the launch or the row count, so
// a batched call equals its one-row calls and the C oracle's sequential fmaf
// loop gives the same bits.

#include <algorithm>
#include <type_traits>

#include "attn_common.h"  // the MFMA operand type, LdsDma, wait_vmcnt

namespace tn {
namespace {

// half's to_f32 (the reference's widening): exact, and a NaN comes back with
// its payload and the quiet bit set (0x7fc00000 | sign | payload << 13 for
// f16, (h | 0x40) << 16 for bf16).
template <int WT>
__device__ inline float widen_w(const void* w, int64_t i) {
    if constexpr (WT == TN_F32) {
        return reinterpret_cast<const float*>(w)[i];
    } else if constexpr (WT == TN_F16) {
        const uint16_t h = reinterpret_cast<const uint16_t*>(w)[i];
        const float f = f16_bits_hw(h);
        if (f == f) return f;
        return __builtin_bit_cast(float, ((uint32_t)(h & 0x8000u) << 16) | 0x7fc00000u | ((uint32_t)(h & 0x3ffu) << 13));
    } else {
        const uint16_t h = reinterpret_cast<const uint16_t*>(w)[i];
        return bf16_to_f32((h & 0x7fffu) > 0x7f80u ? (uint16_t)(h | 0x40u) : h);
    }
}

// y[m, n] = (sequential fma chain over k of x[m, k] * w[n, k]) (+ bias[n]), on
// the f32 matrix core: one v_mfma_f32_16x16x4_f32 is four steps of the chain
// for a 16 x 16 tile, acc = fma(x[k], w[k], acc) for k, k + 1, k + 2, k + 3 in
// order, each rounded on its own and with subnormals (compared with the VALU
// chain over normal, wide-range, subnormal, overflowing and arbitrary bit
// patterns on gfx950: the same bits, NaN payloads aside).
//
// A product takes k = 4 c + g of row i from lane (i = lane % 16, g = lane / 16).
//
// What bounds it: the matrix core. 32 cycles per product and SIMD whatever the
// tile, so K steps of the chain take 8 K cycles at least (7.8 us at K = 2048)
// and a SIMD that holds several tiles queues them.

// four consecutive stored weights, read with the elements' own alignment
template <int WT>
struct WQuad;
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
template <>
struct WQuad<TN_F32> {
    typedef f32x4 vec __attribute__((aligned(4)));
    f32x4 v;
    __device__ void load(const void* w, int64_t i) { v = *reinterpret_cast<const vec*>(static_cast<const float*>(w) + i); }
    __device__ void widen(float (&f)[4]) const { f[0] = v[0], f[1] = v[1], f[2] = v[2], f[3] = v[3]; }
};
template <int WT>
struct WQuad {
    typedef u32x2 vec __attribute__((aligned(2)));
    u32x2 v;
    __device__ void load(const void* w, int64_t i) {
        v = *reinterpret_cast<const vec*>(static_cast<const uint16_t*>(w) + i);
    }
    // (a NaN stays a NaN; its payload does not reach the result)
    __device__ void widen(float (&f)[4]) const {
        const uint32_t h[4] = {v[0] & 0xffffu, v[0] >> 16, v[1] & 0xffffu, v[1] >> 16};
#pragma unroll
        for (int j = 0; j < 4; j++) f[j] = WT == TN_F16 ? f16_bits_hw((uint16_t)h[j]) : bf16_to_f32((uint16_t)h[j]);
    }
};

// f[j] of lane group g becomes f[g] of lane group j
__device__ inline void transpose4(float (&f)[4]) {
#pragma unroll
    for (int e = 0; e < 2; e++) {
        const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(f[e]), __float_as_uint(f[e + 2]), false, false);
        f[e] = __uint_as_float(p[0]), f[e + 2] = __uint_as_float(p[1]);
    }
#pragma unroll
    for (int e = 0; e < 4; e += 2) {
        const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(f[e]), __float_as_uint(f[e + 1]), false, false);
        f[e] = __uint_as_float(p[0]), f[e + 1] = __uint_as_float(p[1]);
    }
}

// The last K % 16 steps, element by element: past K the operands are -0 and
// +0, whose product -0 leaves every accumulator as it is, its sign included.
// x rows and w rows past the last read the last one (their outputs are not
// stored).
template <int WT, int RT, int CT>
__device__ inline void dense_tail(const float* __restrict__ x, int M, int m0, const void* __restrict__ w, int N, int n0,
                                  int K, int lane, f32x4 (&acc)[RT][CT]) {
    const int i16 = lane & 15, g = lane >> 4;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int k = K / 16 * 16 + 4 * q + g, kc = min(k, K - 1);
        float a[RT], b[CT];
#pragma unroll
        for (int i = 0; i < RT; i++) a[i] = k < K ? x[(int64_t)min(m0 + 16 * i + i16, M - 1) * K + kc] : -0.0f;
#pragma unroll
        for (int j = 0; j < CT; j++) b[j] = k < K ? widen_w<WT>(w, (int64_t)min(n0 + 16 * j + i16, N - 1) * K + kc) : 0.0f;
#pragma unroll
        for (int i = 0; i < RT; i++)
#pragma unroll
            for (int j = 0; j < CT; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], b[j], acc[i][j], 0, 0, 0);
    }
}

template <int RT, int CT>
__device__ inline void dense_store(const f32x4 (&acc)[RT][CT], int M, int m0, int N, int n0, int lane,
                                   const float* __restrict__ bias, float* __restrict__ y) {
    const int i16 = lane & 15, g = lane >> 4;
#pragma unroll
    for (int j = 0; j < CT; j++) {
        const int n = n0 + 16 * j + i16;
        if (n >= N) continue;
        const float bv = bias ? bias[n] : 0.0f;
#pragma unroll
        for (int i = 0; i < RT; i++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int m = m0 + 16 * i + 4 * g + r;
                if (m < M) y[(int64_t)m * N + n] = bias ? acc[i][j][r] + bv : acc[i][j][r];
            }
    }
}

constexpr int DL_THREADS = 256, DL_WAVES = DL_THREADS / 64;
constexpr int DL_XCD = 8;

// tiles numbered down the rows first, consecutive numbers on one XCD (its
// workgroups share the columns of w in its L2)
__device__ inline int dense_wg(int id, int nwg) {
    return nwg % DL_XCD == 0 ? (id % DL_XCD) * (nwg / DL_XCD) + id / DL_XCD : id;
}

// Any row width and alignment: a wave walks all of K for one tile alone, the
// operands straight from memory, DL_RING steps in flight ahead of the one
// computed. Each quad of lanes reads four rows, which the vector memory path
// takes one row at a time (about 77 cycles per 1 KB load against 16), so this
// is the form for rows that k_dense_lds cannot read in 16-byte pieces (33
// rows, K 2050, N 999, f16: 286 -> 21 us). A lane
// reads four consecutive k, k = 16 s + 4 g .. + 3, which a 4 x 4 transpose
// between the lane groups turns into the operands of four products.
// The steps in flight are whole vectors: as scalars, the loop's copies of
// single elements waited for each load right after it was issued.
template <int WT>
__global__ void __launch_bounds__(DL_THREADS) k_dense_any(const float* __restrict__ x, int M, int K,
                                                          const void* __restrict__ w, int N,
                                                          const float* __restrict__ bias, float* __restrict__ y,
                                                          int mtiles, int ntiles, int nwg) {
    constexpr int RING = 8;
    if (wg_number() >= nwg) return;
    const int lane = threadIdx.x & 63, i16 = lane & 15, g = lane >> 4;
    const int64_t tile = (int64_t)dense_wg(wg_number(), nwg) * DL_WAVES + (threadIdx.x >> 6);
    if (tile >= (int64_t)mtiles * ntiles) return;
    const int m0 = (int)(tile % mtiles) * 16, n0 = (int)(tile / mtiles) * 16;
    const float* xr = x + (int64_t)min(m0 + i16, M - 1) * K;
    const int64_t wr = (int64_t)min(n0 + i16, N - 1) * K;
    f32x4 acc[1][1] = {{(f32x4){0.f, 0.f, 0.f, 0.f}}};
    struct Step {
        WQuad<TN_F32> a;
        WQuad<WT> b;
    };
    auto load = [&](Step& t, int s) __attribute__((always_inline)) {
        t.a.load(xr, 16 * s + 4 * g);
        t.b.load(w, wr + 16 * s + 4 * g);
    };
    auto compute = [&](const Step& t) __attribute__((always_inline)) {
        float a[4], b[4];
        t.a.widen(a);
        t.b.widen(b);
        transpose4(a);
        transpose4(b);
#pragma unroll
        for (int q = 0; q < 4; q++) acc[0][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[q], b[q], acc[0][0], 0, 0, 0);
    };
    const int nfull = K / 16;
    if (nfull > 0) {
        Step ring[RING];
        // loads are unconditional (a step past the last reads the last again,
        // unused), so the waits count exactly the loads in flight
#pragma unroll
        for (int u = 0; u < RING; u++) load(ring[u], min(u, nfull - 1));
        int s = 0;
        for (; s + RING <= nfull; s += RING) {
#pragma unroll
            for (int u = 0; u < RING; u++) {
                compute(ring[u]);
                load(ring[u], min(s + u + RING, nfull - 1));
                __builtin_amdgcn_sched_barrier(0);
            }
        }
#pragma unroll
        for (int u = 0; u < RING; u++)
            if (s + u < nfull) compute(ring[u]);
    }
    if (16 * nfull < K) dense_tail<WT, 1, 1>(x, M, m0, w, N, n0, K, lane, acc);
    dense_store<1, 1>(acc, M, m0, N, n0, lane, bias, y);
}

// Rows that start at multiples of 16 bytes: WM x WN waves of RT x CT tiles
// share x and w through LDS, which the vector memory path fills at its full
// width (loads straight into LDS, 64 consecutive bytes of a row per quad of
// lanes). A stage is KS of k, in a ring of NS; the operands of stage st + 1
// are read from LDS while the products of stage st run, behind one barrier a
// stage.
//
// LDS holds a stage in 64-byte granules, [granule][row], the 16-byte chunk c
// of a row's granule at place c ^ (row / 2 mod 4). Lane (i, g) reads single
// elements, k = 16 u + 4 j + g of row i, straight into a product's operand:
// the 16 rows of an operand cover every bank, and no lane exchange is left.
// (With 16-byte reads and transposes, a step's eight swaps at 10 cycles each
// on a lone wave took as long as its four products.)
//
// Measured, against a 64 x 64 VALU tile with one LDS buffer: [200, 2048] x
// [2048, 2048] f16 weights 310 -> 27 us (62 TFLOP/s), f32 298 -> 24.6; one row,
// K = N = 2048, f32: 265 -> 16.3 us; 16 rows, K 8192, N 1024: 1145 -> 58 us,
// 7.1 ns a k where the products alone are 3.8.
template <int WT, int WM, int WN, int RT, int CT, int KS, int NS>
__global__ void __launch_bounds__(DL_THREADS) k_dense_lds(const float* __restrict__ x, int M, int K,
                                                          const void* __restrict__ w, int N,
                                                          const float* __restrict__ bias, float* __restrict__ y,
                                                          int mtiles, int nwg) {
    if (wg_number() >= nwg) return;
    static_assert(WM * WN == DL_WAVES, "waves");
    static_assert(NS >= 3, "ring");
    constexpr int WS = WT == TN_F32 ? 4 : 2;             // bytes of a stored weight
    constexpr int BM = 16 * RT * WM, BN = 16 * CT * WN;  // the workgroup's tile
    constexpr int NU = KS / 16;                          // 16-k steps of a stage
    constexpr int LA = BM * KS * 4 / 16 / DL_THREADS, LB = BN * KS * WS / 16 / DL_THREADS;  // loads per thread
    static_assert(LA * DL_THREADS * 16 == BM * KS * 4 && LB * DL_THREADS * 16 == BN * KS * WS, "whole loads");
    static_assert(KS * WS % 64 == 0, "whole granules");
    constexpr int STAGE = BM * KS * 4 + BN * KS * WS;
    __shared__ __align__(16) uint8_t ring[NS * STAGE];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int i16 = lane & 15, g = lane >> 4;
    const int wg = dense_wg(wg_number(), nwg);
    const int m0 = wg % mtiles * BM, n0 = wg / mtiles * BN;
    const int wm0 = wave / WN * 16 * RT, wn0 = wave % WN * 16 * CT;  // the wave's first row and column in the tile

    // rows past the last lie past the descriptor and read as zero
    const LdsDma ra(x + (int64_t)m0 * K, (uint32_t)(min(BM, M - m0) * (int64_t)K * 4));
    const LdsDma rb(static_cast<const uint8_t*>(w) + (int64_t)n0 * K * WS, (uint32_t)(min(BN, N - n0) * (int64_t)K * WS));
    // byte offset in an operand of the 16 bytes that go to place p of its stage
    auto place = [&](int p, int rows, int rowbytes) {
        const int gran = p / (4 * rows), r = p % (4 * rows) / 4, c = (p & 3) ^ ((r >> 1) & 3);
        return (uint32_t)(r * rowbytes + gran * 64 + c * 16);
    };
    uint32_t va[LA], vb[LB];
#pragma unroll
    for (int i = 0; i < LA; i++) va[i] = place((wave * LA + i) * 64 + lane, BM, K * 4);
#pragma unroll
    for (int i = 0; i < LB; i++) vb[i] = place((wave * LB + i) * 64 + lane, BN, K * WS);
    auto issue = [&](int st, int slot) __attribute__((always_inline)) {
        uint8_t* const sa = ring + slot * STAGE;
#pragma unroll
        for (int i = 0; i < LA; i++) ra.load16(va[i] + (uint32_t)(st * KS * 4), sa + (wave * LA + i) * 1024);
#pragma unroll
        for (int i = 0; i < LB; i++)
            rb.load16(vb[i] + (uint32_t)(st * KS * WS), sa + BM * KS * 4 + (wave * LB + i) * 1024);
    };

    // this lane's place in an operand for chunk c of a granule, and one stage's elements
    const int rsw = (i16 >> 1) & 3;
    uint32_t pa[4], pb[4];
#pragma unroll
    for (int c = 0; c < 4; c++) {
        pa[c] = (uint32_t)((wm0 + i16) * 64 + (c ^ rsw) * 16 + g * 4);
        pb[c] = (uint32_t)(BM * KS * 4 + (wn0 + i16) * 64 + (c ^ rsw) * 16 + g * WS);
    }
    using WE = typename std::conditional<WT == TN_F32, float, uint16_t>::type;
    struct Stage {
        float a[NU][RT][4];
        WE b[NU][CT][4];
    };
    // element j of 16-k step u of the stage at s
    auto lread = [&](const uint8_t* s, int u, int j, Stage& t) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < RT; i++) t.a[u][i][j] = *reinterpret_cast<const float*>(s + pa[j] + u * BM * 64 + i * 1024);
#pragma unroll
        for (int i = 0; i < CT; i++) {
            if constexpr (WT == TN_F32)
                t.b[u][i][j] = *reinterpret_cast<const float*>(s + pb[j] + u * BN * 64 + i * 1024);
            else  // 32 k to a granule
                t.b[u][i][j] = *reinterpret_cast<const uint16_t*>(s + pb[(u & 1) * 2 + (j >> 1)] + (j & 1) * 8 +
                                                                  (u >> 1) * BN * 64 + i * 1024);
        }
    };
    auto wide = [](WE v) {
        if constexpr (WT == TN_F32) return v;
        else if constexpr (WT == TN_F16) return f16_bits_hw(v);
        else return bf16_to_f32(v);
    };
    f32x4 acc[RT][CT];
#pragma unroll
    for (int i = 0; i < RT; i++)
#pragma unroll
        for (int j = 0; j < CT; j++) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
    // The first nu steps' products. A product waits for the one before it on
    // the same accumulator, and what follows it in the wave waits too: what
    // else the stage has to do (`other`) goes a little behind each product.
    auto products = [&](const Stage& t, int nu, auto other) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < NU; u++) {
            if (u >= nu) break;
#pragma unroll
            for (int q = 0; q < 4; q++) {
#pragma unroll
                for (int i = 0; i < RT; i++)
#pragma unroll
                    for (int j = 0; j < CT; j++)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(t.a[u][i][q], wide(t.b[u][j][q]), acc[i][j], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                other(u, q);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };

    const int nfull = K / 16, nst = (nfull + NU - 1) / NU;
    // stage st has landed in LDS for every wave, and every wave has read
    // stage st - 1, whose slot the stage NS - 1 further on takes
    auto landed = [&](int st) __attribute__((always_inline)) {
        if (st + NS - 2 < nst) wait_vmcnt<(NS - 2) * (LA + LB)>();
        else wait_vmcnt<0>();
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    for (int st = 0; st < min(NS - 1, nst); st++) issue(st, st);
    if (nst > 0) {
        Stage t[2];
        landed(0);
        if (NS - 1 < nst) issue(NS - 1, NS - 1);
#pragma unroll
        for (int u = 0; u < NU; u++)
#pragma unroll
            for (int q = 0; q < 4; q++) lread(ring, u, q, t[0]);
        int st = 0, slot = 0;
        // stage st's products while stage st + 1 is read
        auto step = [&](const Stage& cur, Stage& next) __attribute__((always_inline)) {
            const int free = slot;
            slot = slot + 1 < NS ? slot + 1 : 0;
            const uint8_t* const s = ring + slot * STAGE;
            landed(st + 1);
            products(cur, NU, [&](int u, int q) __attribute__((always_inline)) {
                lread(s, u, q, next);
                if (u == 0 && q == 3 && st + NS < nst) issue(st + NS, free);
            });
            st++;
        };
        while (st + 2 < nst) {
            step(t[0], t[1]);
            step(t[1], t[0]);
        }
        auto none = [](int, int) {};
        if (st + 1 < nst) {
            step(t[0], t[1]);
            products(t[1], nfull - st * NU, none);
        } else {
            products(t[0], nfull - st * NU, none);
        }
    }
    if (16 * nfull < K) dense_tail<WT, RT, CT>(x, M, m0 + wm0, w, N, n0 + wn0, K, lane, acc);
    dense_store<RT, CT>(acc, M, m0 + wm0, N, n0 + wn0, lane, bias, y);
}

constexpr int DV_T = 64;   // rows of x and output features per workgroup
constexpr int DV_TK = 16;  // k per LDS stage
constexpr int DV_LD = 68;  // LDS row stride in floats (float4-aligned, staggers the banks)

// The same chain on the VALU, 64 x 64 outputs a workgroup, for many short rows,
// above all ones that k_dense_lds cannot read (dense_valu). 256 threads; thread (tx, ty) = (t %
// 16, t / 16) owns rows ty*4..ty*4+3 and features tx*4..tx*4+3. Stage s holds
// x[:, 16s..16s+15] and w[:, 16s..16s+15] k-major in LDS; only k < K is ever
// accumulated. An operand element is read once a workgroup where k_dense_any
// reads it once a 16 x 16 tile.
template <int WT>
__global__ void __launch_bounds__(DL_THREADS) k_dense_valu(const float* __restrict__ x, int M, int K,
                                                           const void* __restrict__ w, int N,
                                                           const float* __restrict__ bias, float* __restrict__ y) {
    __shared__ __align__(16) float xs[DV_TK][DV_LD];
    __shared__ __align__(16) float ws[DV_TK][DV_LD];
    const int t = threadIdx.x;
    const int tx = t % 16, ty = t / 16;
    const int n0 = blockIdx.x * DV_T, m0 = blockIdx.y * DV_T;
    const int lk = t % DV_TK, lr = t / DV_TK;  // loader: k column, first row (rows lr + 16i)
    float acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) acc[i][j] = 0.0f;
    for (int k0 = 0; k0 < K; k0 += DV_TK) {
        const int kk = k0 + lk;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int r = lr + 16 * i;
            const int m = m0 + r, n = n0 + r;
            xs[lk][r] = (m < M && kk < K) ? x[(int64_t)m * K + kk] : 0.0f;
            ws[lk][r] = (n < N && kk < K) ? widen_w<WT>(w, (int64_t)n * K + kk) : 0.0f;
        }
        __syncthreads();
        const int kend = min(DV_TK, K - k0);  // the same for every thread
        for (int k = 0; k < kend; k++) {
            const float4 a = *reinterpret_cast<const float4*>(&xs[k][ty * 4]);
            const float4 b = *reinterpret_cast<const float4*>(&ws[k][tx * 4]);
            const float av[4] = {a.x, a.y, a.z, a.w}, bv[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int j = 0; j < 4; j++) acc[i][j] = __builtin_fmaf(av[i], bv[j], acc[i][j]);
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int m = m0 + ty * 4 + i;
        if (m >= M) continue;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int n = n0 + tx * 4 + j;
            if (n < N) y[(int64_t)m * N + n] = bias ? acc[i][j] + bias[n] : acc[i][j];
        }
    }
}

// Whether k_dense_valu takes rows that k_dense_lds cannot read. It keeps a few
// waves on a CU waiting for one LDS buffer, whatever the shape: about 0.145 us a k
// up to 1024 workgroups, and 9 us to store 64 MB. k_dense_any has 16 times as many
// tiles and pays for each element it loads, twice that where the rows start at
// nearly the same place of the memory's lines (K one off a multiple of 32), and a
// quarter more where a 16-bit weight's odd rows start between dwords. Measured,
// us, valu / any, f32 weights unless stated, by workgroups here:
//    108 [333, K] x [1111, K]:  K 17 5.9/4.4  33 8.0/6.1  129 22.5/9.6
//    256 [1024, K] x [1024, K]: K 13 5.3/4.3  17 6.2/6.5  33 8.2/9.9  45 9.3/7.9  75 14.4/8.4
//                               129 22.7/17.0   f16: 33 8.5/10.0  63 11.7/13.3  129 23.0/22.1
//    480 [900, K] x [2000, K]:  K 21 7.8/10.8  45 10.5/12.1  99 18.5/11.8  129 22.8/27.8  299 46.9/29.3
//                               f16: 99 18.8/14.2  257 41.6/53.3  515 80/51
//    832 [1000, K] x [3300, K]: K 13 10.5/9.9  33 15.0/30.0  99 24.9/19.5  299 58/53  515 102/78
//                               f16: 299 62/65  450 93/66  515 102/92
//   1024 [1024, K] x [4096, K]: K 8 10.4/14.2  33 14.3/35.7  299 52/57  515 93/81   f16: 515 101/110
//   1760 [1000, K] x [7000, K]: K 13 15.7/17.6  129 40/98  299 77/107  1030 243/317
// Under eight steps the store is all there is (K 7, 1024 workgroups: 10.2/9.3).
// `lds`: rows that k_dense_lds reads. It loses where a workgroup has little more
// than one stage, most of it the last K % 16 steps (us, valu / lds, f32; f16 alike
// but for the last two):
//    480 [900, K] x [2000, K]:  K 16 6.8/8.4  24 8.0/11.5  40 10.0/11.8  48 10.7/9.3
//    640 [1000, K] x [2500, K]: K 16 8.8/9.1  24 10.2/12.1  32 10.8/9.8   f16: 16 8.9/6.6
//   1760 [1000, K] x [7000, K]: K 24 17.9/23.8  40 20.6/25.5  48 22.6/20.9   f16: 40 22.0/21.0
inline bool dense_valu(int64_t M, int64_t N, int64_t K, bool lds, bool f32) {
    const int64_t wgs = cdiv(M, DV_T) * cdiv(N, DV_T);
    if (wgs <= 128 || K < 8 || cdiv(N, DV_T) > WG_ROW) return false;  // (its grid has the features in x alone)
    if (lds) {
        if (wgs <= 256 || K >= 64) return false;
        if (wgs < 512) return K < 48;
        return wgs > 512 && (K < 32 ? f32 || K >= 24 : f32 && K % 16 && wgs > 1024);
    }
    const bool same = (K + 1) % 32 <= 2;
    if (wgs <= 256) return K >= 16 && K < (same ? 72 : 40);
    if (wgs <= 640) return K < 96 || same;
    return wgs > 1024 || K < 400 || same || (!f32 && K % 2);
}

template <int WT>
void launch_dense(hipStream_t st, const float* x, int64_t M, int64_t K, const void* w, int64_t N, const float* bias,
                  float* y) {
    constexpr int WS = WT == TN_F32 ? 4 : 2;
    const bool aligned = (reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w)) % 16 == 0 &&
                         K * WS % 16 == 0 && K % 4 == 0 && 64 * K * 4 <= INT32_MAX;
    const bool lds = aligned && K >= 16;
    if (dense_valu(M, N, K, lds, WS == 4)) {
        hipLaunchKernelGGL(k_dense_valu<WT>, dim3((unsigned)cdiv(N, DV_T), (unsigned)cdiv(M, DV_T)), dim3(DL_THREADS), 0,
                           st, x, (int)M, (int)K, w, (int)N, bias, y);
        return;
    }
    if (!lds) {
        const int64_t mt = cdiv(M, 16), nt = cdiv(N, 16), wgs = cdiv(mt * nt, DL_WAVES);
        hipLaunchKernelGGL(k_dense_any<WT>, wg_grid(wgs), dim3(DL_THREADS), 0, st, x, (int)M, (int)K, w, (int)N, bias, y,
                           (int)mt, (int)nt, (int)wgs);
        return;
    }
#define TN_DL(WM, WN, RT, CT, KS, NS)                                                                                \
    do {                                                                                                             \
        const int64_t mt = cdiv(M, 16 * RT * WM), wgs = mt * cdiv(N, 16 * CT * WN);                                 \
        hipLaunchKernelGGL((k_dense_lds<WT, WM, WN, RT, CT, KS, NS>), wg_grid(wgs), dim3(DL_THREADS), 0, st, x,     \
                           (int)M, (int)K, w, (int)N, bias, y, (int)mt, (int)wgs);                                  \
    } while (0)
    // one row tile: the four waves side by side over 64 columns (wider than
    // 16 rows would be padding); 64 x 64 once that gives every CU two
    // workgroups (half the LDS reads per product: [1024, 256] x [3200, 256] 25.2
    // us, 28 with 32 x 32); else 32 x 32, which spreads few outputs further
    if (M <= 16) TN_DL(1, 4, 1, 1, 64, 6);
    else if (cdiv(M, 64) * cdiv(N, 64) >= 512) TN_DL(2, 2, 2, 2, 32, 4);
    else TN_DL(2, 2, 1, 1, 64, 5);
#undef TN_DL
}

template <int WT>
__global__ void k_dense_store(const float* __restrict__ x, int64_t count, void* __restrict__ out) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < count; i += (int64_t)gridDim.x * blockDim.x) {
        if constexpr (WT == TN_F32) reinterpret_cast<float*>(out)[i] = x[i];
        else if constexpr (WT == TN_F16) reinterpret_cast<uint16_t*>(out)[i] = f16_out(x[i]);
        else reinterpret_cast<uint16_t*>(out)[i] = bf16_out(x[i]);
    }
}

template <int WT>
__global__ void k_dense_widen(const void* __restrict__ w, int64_t count, float* __restrict__ out) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < count; i += (int64_t)gridDim.x * blockDim.x)
        out[i] = widen_w<WT>(w, i);
}

tn_status dense_dtype(const char* op, int dtype) {
    if (dtype == TN_F32 || dtype == TN_F16 || dtype == TN_BF16) return TN_OK;
    return fail(TN_ENOTIMPL, std::string(op) + ": the dense formats are f32, f16 and bf16 (dtype code " +
                                 std::to_string(dtype) + " is none of them)");
}

unsigned stride_grid(int64_t count) { return (unsigned)std::min<int64_t>(cdiv(count, 256), 8192); }

}  // namespace
}  // namespace tn

using namespace tn;

extern "C" {

tn_status tn_dense_quantize(void* stream, const float* x, int64_t count, int dtype, void* out) {
    const char* op = "torch._C._quantize";
    TN_TRY(dense_dtype(op, dtype));
    if (count < 0) return fail(TN_EINVAL, std::string(op) + ": negative element count");
    if (count == 0) return TN_OK;
    if (!x || !out) return fail(TN_EVALUE, std::string(op) + ": null pointer");
    hipStream_t st = (hipStream_t)stream;
    if (dtype == TN_F32) hipLaunchKernelGGL(k_dense_store<TN_F32>, dim3(stride_grid(count)), dim3(256), 0, st, x, count, out);
    else if (dtype == TN_F16) hipLaunchKernelGGL(k_dense_store<TN_F16>, dim3(stride_grid(count)), dim3(256), 0, st, x, count, out);
    else hipLaunchKernelGGL(k_dense_store<TN_BF16>, dim3(stride_grid(count)), dim3(256), 0, st, x, count, out);
    TN_LAUNCHED();
    return TN_OK;
}

tn_status tn_dense_dequantize(void* stream, const void* w, int dtype, int64_t count, float* out) {
    const char* op = "torch._C._dequantize";
    TN_TRY(dense_dtype(op, dtype));
    if (count < 0) return fail(TN_EINVAL, std::string(op) + ": negative element count");
    if (count == 0) return TN_OK;
    if (!w || !out) return fail(TN_EVALUE, std::string(op) + ": null pointer");
    hipStream_t st = (hipStream_t)stream;
    if (dtype == TN_F32) hipLaunchKernelGGL(k_dense_widen<TN_F32>, dim3(stride_grid(count)), dim3(256), 0, st, w, count, out);
    else if (dtype == TN_F16) hipLaunchKernelGGL(k_dense_widen<TN_F16>, dim3(stride_grid(count)), dim3(256), 0, st, w, count, out);
    else hipLaunchKernelGGL(k_dense_widen<TN_BF16>, dim3(stride_grid(count)), dim3(256), 0, st, w, count, out);
    TN_LAUNCHED();
    return TN_OK;
}

tn_status tn_dense_linear(void* stream, const float* x, int64_t m, int64_t k, const void* w, int w_dtype,
                          int64_t n, const float* bias, float* y) {
    const char* op = "torch._C._quantized_linear";
    TN_TRY(dense_dtype(op, w_dtype));
    if (m < 0 || n < 0 || k < 1)
        return fail(TN_EINVAL, std::string(op) + ": mat1 and mat2 shapes cannot be multiplied ([" +
                                   std::to_string(m) + ", " + std::to_string(k) + "] and " + std::to_string(k) +
                                   "x" + std::to_string(n) + ")");
    if (m == 0 || n == 0) return TN_OK;
    if (!x || !w || !y) return fail(TN_EVALUE, std::string(op) + ": null pointer");
    if (m > INT32_MAX || n > INT32_MAX || k > INT32_MAX || cdiv(m, 64) > 65535 ||
        cdiv(m, 16) * cdiv(n, 16) / DL_WAVES >= INT32_MAX)
        return fail(TN_EVALUE, std::string(op) + ": shape too large");
    hipStream_t st = (hipStream_t)stream;
    if (w_dtype == TN_F32) launch_dense<TN_F32>(st, x, m, k, w, n, bias, y);
    else if (w_dtype == TN_F16) launch_dense<TN_F16>(st, x, m, k, w, n, bias, y);
    else launch_dense<TN_BF16>(st, x, m, k, w, n, bias, y);
    TN_LAUNCHED();
    return TN_OK;
}

}  // extern "C"
