// The q4_0 / q8_0 linear of more rows than the GEMV takes: batched decode,
// prompts.
//
// The reference's recurrence (see qlinear.hip), sumf += ((float)S_b * d_w) *
// d_x in block order, each step rounded on its own, with the exact integer
// block dots S_b from v_mfma_i32_16x16x32_i8: one product is one block of a
// 16 x 16 tile. A wave owns RT x CT tiles and all of K, so the order of the
// sum is kept without any exchange; what a call has to give it is many waves,
// operands that are there in time, and few other instructions.
//
// - q4_0 codes: with t = w ^ 0x88888888, the bytes t & 0xf0f0f0f0 and
//   (t << 4) & 0xf0f0f0f0 are 16 (nib - 8) as int8 (a nibble with its top bit
//   flipped is nib - 8 in two's complement), so four instructions make the
//   operand and no correction term is left: the product is 16 S_b. The
//   prepass stores d_x / 16; every value stays a power of two away from the
//   reference's until that cancels, so each rounding is the reference's
//   (|16 S_b| < 2^24; 16 S_b d_w does not overflow; d_x / 16, an f16 over 16, is
//   exact).
// - K-slot order: lane group g (lanes 16 g .. 16 g + 15) holds elements
//   4 g .. 4 g + 3 and 16 + 4 g .. 16 + 4 g + 3 of the block: dword g of a q4_0
//   block's low and high nibbles, dwords g and 4 + g of a q8_0 block. The
//   prepass writes the activation codes in that order, tile by tile, so that a
//   product's operand is 512 consecutive bytes.
// - A ring of NS stages of KB blocks in LDS, filled by loads that go straight
//   to LDS (a code plane that is not 16-byte aligned through registers, a stage
//   later: DMA false); one barrier per stage. Within a stage block t + 2 is read from LDS,
//   block t + 1's products are issued and block t's roundings done, in that
//   order, so that neither LDS nor the matrix core is waited for.
//
// What bounds it: the recurrence's 16 VALU instructions per tile and block
// (convert, two products, a sum, four elements each), issued every 4.3 cycles
// by a SIMD with several waves and every 8 by one with a single wave. 2 x 2 tiles
// take about 33 ns a tile and block on each SIMD, 78 cycles at 2.4 GHz, of which
// those 16 are 69 ([512, 4096] x [14336, 4096] in 124 us, 485 TFLOP/s, 5-7 of it the
// prepass). One tile a wave, alone on its SIMD, takes 110 ns, some 260 cycles (14.3
// of the 17.8 us at m = 16; the prepass is 4): 128 are the 16, the rest the scale's
// widening, the nibbles, the LDS reads and the waits, not measured one by one.
//
// Compared and not kept: two waves rounding two rows each of the same products
// (23 us at m = 16: the doubled reads cost what the halved roundings saved); 4 x 2
// tiles (72.4 against 78.2 us at m = 256, but 137 against 123 at 512 and 50-70%
// slower with fewer tiles); a ring of six or eight stages (no change).
#include <algorithm>

#include "attn_common.h"  // LdsDma, wait_vmcnt, f32x4
#include "qgemm.h"

namespace tn {
namespace {

constexpr int QG_WAVES = 4, QG_TH = 64 * QG_WAVES;
constexpr int QG_XCD = 8;

// Quantised rows (Q8_0): four lanes per (row, block), eight elements each. Rows past M get zero codes and scales.
//   xf  [row tile][block][64 lanes][8 bytes]  the operand of a product
//   dxf [row tile][block][16]                 d_x (over 16 for q4_0)
template <typename XT, int XM>
__global__ __launch_bounds__(256) void k_q8_frag(const XT* __restrict__ x, int M, int64_t blocks, int K, int nb,
                                                 uint8_t* __restrict__ xf, float* __restrict__ dxf, float unit, int hd) {
    const int64_t blk = (int64_t)blockIdx.x * (blockDim.x >> 2) + (threadIdx.x >> 2);
    const int part = threadIdx.x & 3;
    if (blk >= blocks) return;  // the four lanes of a block leave together
    const int row = (int)(blk / nb), b = (int)(blk - (int64_t)row * nb);
    float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (row < M) load_part<XT, XM>(x, row, M, K, b, part, hd, v);
    int q[8], s;
    float dx;
    q8_0_quad(v, q, &dx, &s);
    if (row >= M) dx = 0.0f;
    uint32_t w[2] = {0u, 0u};
#pragma unroll
    for (int e = 0; e < 8; e++) w[e >> 2] |= ((uint32_t)q[e] & 0xffu) << (8 * (e & 3));
    const int64_t tb = (int64_t)(row >> 4) * nb + b;
    // elements 8 part .. + 3 and + 4 .. + 7: lane groups g and g + 1, low or high dword
    const int g = 2 * (part & 1), half = part >> 1;
    uint8_t* o = xf + tb * 512 + (row & 15) * 8 + half * 4;
    *reinterpret_cast<uint32_t*>(o + g * 128) = w[0];
    *reinterpret_cast<uint32_t*>(o + (g + 1) * 128) = w[1];
    if (part == 0) dxf[tb * 16 + (row & 15)] = dx * unit;
}

typedef int i32x4 __attribute__((ext_vector_type(4)));

// WM x WN waves of RT x CT tiles; KB blocks a stage, NS stages.
template <int FMT, int RT, int CT, int WM, int WN, int KB, int NS>
struct QGeo {
    static_assert(WM * WN == QG_WAVES, "waves");
    static_assert(KB % 4 == 0, "the block registers rotate by four");
    static constexpr int CB = FMT == FMT_Q8_0 ? 32 : 16;    // code bytes per block
    static constexpr int RTT = RT * WM, BN = 16 * CT * WN;  // row tiles and columns of a workgroup
    // 64-lane loads of a stage: codes, activation codes, their scales (16 bytes
    // a lane), weight scales (2 bytes); each operand's dealt to the waves in turn
    static constexpr int IW = (BN * KB * CB / 16 + 63) / 64, IA = RTT * KB * 32 / 64, IX = (RTT * KB * 4 + 63) / 64,
                         ID = (BN * KB + 63) / 64;
    static_assert(IA * 64 == RTT * KB * 32, "whole row tiles");
    static constexpr int LW = (IW + 3) / 4, LA = (IA + 3) / 4, LX = (IX + 3) / 4, LD = (ID + 3) / 4;
    static constexpr int OW = 0, OA = OW + IW * 1024, OX = OA + IA * 1024, OD = OX + IX * 1024, STAGE = OD + ID * 256;
};

template <int FMT, int RT, int CT, int WM, int WN, int KB, int NS, bool DMA>
__global__ __launch_bounds__(QG_TH) void k_qgemm(const uint8_t* __restrict__ xf, const float* __restrict__ dxf, int M,
                                                 int mtiles, int nwg, int nb, const uint8_t* __restrict__ qs,
                                                 const uint16_t* __restrict__ dw, int N, const float* __restrict__ bias,
                                                 void* y, int y_bf16, const float* resid) {
    using G = QGeo<FMT, RT, CT, WM, WN, KB, NS>;
    constexpr int CB = G::CB, BN = G::BN, AHEAD = RT * CT < 4 ? 2 : 1;
    constexpr int PER_STAGE = (DMA ? G::LW : 0) + G::LA + G::LX + G::LD;
    static_assert((NS - 2) * PER_STAGE < 64, "loads in flight");
    // the ring, then 1 KB that takes the zeros of a wave with no load left to issue
    __shared__ __align__(16) uint8_t ring[NS * G::STAGE + 1024];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int i16 = lane & 15, g = lane >> 4;
    // tiles numbered down the rows first, consecutive numbers on one XCD
    const int mwg = (mtiles + G::RTT - 1) / G::RTT;
    const int id = wg_number();
    if (id >= nwg) return;
    const int wg = nwg % QG_XCD == 0 ? (id % QG_XCD) * (nwg / QG_XCD) + id / QG_XCD : id;
    const int t0 = wg % mwg * G::RTT, n0 = wg / mwg * BN;  // first row tile, first column
    const int wt = wave / WN * RT, wn = wave % WN * 16 * CT;

    const int ncols = min(BN, N - n0), ntl = min(G::RTT, mtiles - t0);
    const LdsDma rw(qs + (int64_t)n0 * nb * CB, (uint32_t)(ncols * nb * CB));
    const LdsDma ra(xf + (int64_t)t0 * nb * 512, (uint32_t)(ntl * nb * 512));
    const LdsDma rx(dxf + (int64_t)t0 * nb * 16, (uint32_t)(ntl * nb * 64));
    const LdsDma rd(dw + (int64_t)n0 * nb, (uint32_t)(ncols * nb * 2));
    // offsets of this thread's pieces in the first stage (load i of a wave is
    // the operand's load 4 i + wave). Codes lie in 64-byte granules,
    // [granule][column], 16-byte chunk c of a column's granule at place
    // c ^ (column / 2 mod 4): quads of lanes load 64 consecutive bytes and the
    // 16 columns of an operand cover every LDS bank.
    uint32_t vw[G::LW], va[G::LA], vx[G::LX], vd[G::LD];
#pragma unroll
    for (int i = 0; i < G::LW; i++) {
        const int p = (4 * i + wave) * 64 + lane, gran = p / (4 * BN), r = p % (4 * BN) / 4, c = (p & 3) ^ ((r >> 1) & 3);
        vw[i] = gran * 64 < KB * CB ? (uint32_t)(r * nb * CB + gran * 64 + c * 16) : BUF_OOB;
    }
#pragma unroll
    for (int i = 0; i < G::LA; i++) {
        const int p = (4 * i + wave) * 64 + lane;
        va[i] = p < G::IA * 64 ? (uint32_t)(p / (KB * 32) * nb * 512 + p % (KB * 32) * 16) : BUF_OOB;
    }
#pragma unroll
    for (int i = 0; i < G::LX; i++) {
        const int p = (4 * i + wave) * 64 + lane;
        vx[i] = p < G::RTT * KB * 4 ? (uint32_t)(p / (KB * 4) * nb * 64 + p % (KB * 4) * 16) : BUF_OOB;
    }
#pragma unroll
    for (int i = 0; i < G::LD; i++) {
        // scale of (block, column) at dword (block / 4) 4 BN + 4 column + block % 4
        const int p = (4 * i + wave) * 64 + lane, b = p / (4 * BN) * 4 + (p & 3), c = p % (4 * BN) / 4;
        vd[i] = b < KB ? (uint32_t)(c * nb + b) * 2u : BUF_OOB;
    }
    // the codes of the last issued stage on their way through registers, and its slot
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    [[maybe_unused]] u32x4 pend[G::LW];
    [[maybe_unused]] int pslot = 0;
    auto flush = [&]() __attribute__((always_inline)) {
        if constexpr (!DMA) {
#pragma unroll
            for (int i = 0; i < G::LW; i++)
                if (4 * i + wave < G::IW)
                    *reinterpret_cast<u32x4*>(ring + pslot * G::STAGE + G::OW + (4 * i + wave) * 1024 + lane * 16) = pend[i];
        }
    };
    auto issue = [&](int st, int slot) __attribute__((always_inline)) {
        uint8_t* const s = ring + slot * G::STAGE;
        uint8_t* const spare = ring + NS * G::STAGE;
        if constexpr (DMA) {
#pragma unroll
            for (int i = 0; i < G::LW; i++)
                rw.load16(vw[i] + (uint32_t)(st * KB * CB), 4 * i + wave < G::IW ? s + G::OW + (4 * i + wave) * 1024 : spare);
        } else {
            typedef u32x4 anywhere __attribute__((aligned(1)));
            const uint32_t bytes = (uint32_t)(ncols * nb * CB);
#pragma unroll
            for (int i = 0; i < G::LW; i++) {
                // (past the end: the first codes again, unused)
                const uint32_t o = vw[i] + (uint32_t)(st * KB * CB);
                pend[i] = *reinterpret_cast<const anywhere*>(qs + (int64_t)n0 * nb * CB + (o < bytes ? o : 0u));
            }
            pslot = slot;
        }
#pragma unroll
        for (int i = 0; i < G::LA; i++)
            ra.load16(va[i] + (uint32_t)(st * KB * 512), 4 * i + wave < G::IA ? s + G::OA + (4 * i + wave) * 1024 : spare);
#pragma unroll
        for (int i = 0; i < G::LX; i++)
            rx.load16(vx[i] + (uint32_t)(st * KB * 64), 4 * i + wave < G::IX ? s + G::OX + (4 * i + wave) * 1024 : spare);
#pragma unroll
        for (int i = 0; i < G::LD; i++)
            rd.load2(vd[i] + (uint32_t)(st * KB * 2), 4 * i + wave < G::ID ? s + G::OD + (4 * i + wave) * 256 : spare);
    };

    // the operands of one block
    constexpr int WD = CB / 16;
    struct Block {
        uint32_t w[CT][WD];
        long a[RT];
        f32x4 dx[RT];
    };
    const int rsw = (i16 >> 1) & 3;
    uint32_t pw[4];
#pragma unroll
    for (int c = 0; c < 4; c++) pw[c] = (uint32_t)(G::OW + (wn + i16) * 64 + (c ^ rsw) * 16 + g * 4);
    const uint32_t pa = (uint32_t)(G::OA + wt * KB * 512 + lane * 8), px = (uint32_t)(G::OX + wt * KB * 64 + g * 16),
                   pd = (uint32_t)(G::OD + (wn + i16) * 16);
    auto lread = [&](const uint8_t* s, int b, Block& t) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < CT; j++) {
#pragma unroll
            for (int h = 0; h < WD; h++)
                t.w[j][h] = *reinterpret_cast<const uint32_t*>(s + pw[(b * WD + h) & 3] + (b * WD / 4) * BN * 64 + j * 1024);
        }
#pragma unroll
        for (int i = 0; i < RT; i++) {
            t.a[i] = *reinterpret_cast<const long*>(s + pa + i * KB * 512 + b * 512);
            t.dx[i] = *reinterpret_cast<const f32x4*>(s + px + i * KB * 64 + b * 64);
        }
    };
    // the weight scales of four blocks at once (the dword's low half)
    struct Scales {
        u32x4 d[CT];
    };
    auto dread = [&](const uint8_t* s, int b, Scales& t) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < CT; j++) t.d[j] = *reinterpret_cast<const u32x4*>(s + pd + (b >> 2) * BN * 16 + j * 256);
    };
    f32x4 acc[RT][CT];
#pragma unroll
    for (int i = 0; i < RT; i++)
#pragma unroll
        for (int j = 0; j < CT; j++) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
    auto products = [&](const Block& t, i32x4 (&sv)[RT][CT]) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < CT; j++) {
            uint32_t lo, hi;
            if constexpr (FMT == FMT_Q8_0) {
                lo = t.w[j][0], hi = t.w[j][WD - 1];
            } else {
                const uint32_t f = t.w[j][0] ^ 0x88888888u;
                lo = (f << 4) & 0xf0f0f0f0u, hi = f & 0xf0f0f0f0u;
            }
            const long b = (long)(((uint64_t)hi << 32) | lo);
#pragma unroll
            for (int i = 0; i < RT; i++)
                sv[i][j] = __builtin_amdgcn_mfma_i32_16x16x32_i8(t.a[i], b, (i32x4){0, 0, 0, 0}, 0, 0, 0);
        }
    };
    auto roundings = [&](const Block& t, const Scales& d, int b, const i32x4 (&sv)[RT][CT]) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < CT; j++) {
            const float dwf = f16_bits_hw((uint16_t)d.d[j][b & 3]);
#pragma unroll
            for (int i = 0; i < RT; i++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    float v = (float)sv[i][j][r] * dwf;
                    v = v * t.dx[i][r];
                    acc[i][j][r] = acc[i][j][r] + v;
                }
        }
    };

    const int nst = (nb + KB - 1) / KB;
    // stage st has landed for every wave, and every wave has read stage st - 1
    auto landed = [&](int st) __attribute__((always_inline)) {
        if (st + NS - 2 < nst) wait_vmcnt<(NS - 2) * PER_STAGE>();
        else wait_vmcnt<0>();
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    for (int st = 0; st < min(NS - 1, nst); st++) {
        if (st > 0) flush();
        issue(st, st);
    }
    // Registers of block t: blk[t mod 2 AHEAD], products sv[t mod AHEAD]. Few
    // tiles: block t + 2 is read and t + 1's products issued ahead of t's
    // roundings. Four and more hide a product's latency by themselves: one
    // block ahead, half the registers.
    Block blk[2 * AHEAD];
    i32x4 sv[AHEAD][RT][CT];
    flush();
    landed(0);
    if (NS - 1 < nst) issue(NS - 1, NS - 1);
    lread(ring, 0, blk[0]);
    if constexpr (AHEAD == 2) {
        lread(ring, 1, blk[1]);
        products(blk[0], sv[0]);
    }
    Scales dn[2];  // of the four blocks at hand, and the next four
    dread(ring, 0, dn[0]);
    int slot = 0, st = 0;
    // The first `left` blocks of a stage. Whole stages with one behind them
    // have no branch within.
    auto stage = [&](auto whole, int left) __attribute__((always_inline)) {
        constexpr bool WHOLE = decltype(whole)::value;
        const uint8_t* const s = ring + slot * G::STAGE;
        const int next = slot + 1 < NS ? slot + 1 : 0;
        const uint8_t* const sn = ring + next * G::STAGE;
#pragma unroll
        for (int b = 0; b < KB; b++) {
            if (!WHOLE && b >= left) break;
            if (WHOLE && b == KB - AHEAD) {
                // every read of this stage has been issued: its slot takes
                // stage st + NS once all waves are here (and stage st - 1's
                // slot, free since the barrier before, the codes issued there)
                if (st + NS - 1 < nst) flush();
                landed(st + 1);
                if (st + NS < nst) issue(st + NS, slot);
            }
            // (past the last block these read stale LDS, unused)
            lread(b + AHEAD < KB ? s : sn, (b + AHEAD) % KB, blk[(b + AHEAD) % (2 * AHEAD)]);
            if (b % 4 == 0 && b + 4 < KB) dread(s, b + 4, dn[(b / 4 + 1) & 1]);
            if (KB > 4 && b == KB - 1) dread(sn, 0, dn[0]);
            products(blk[(b + AHEAD - 1) % (2 * AHEAD)], sv[(b + AHEAD - 1) % AHEAD]);
            __builtin_amdgcn_sched_barrier(0);
            roundings(blk[b % (2 * AHEAD)], dn[(b / 4) & 1], b, sv[b % AHEAD]);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (KB == 4) dread(sn, 0, dn[0]);
        slot = next;
    };
    for (; st + 1 < nst; st++) stage(std::true_type{}, KB);
    stage(std::false_type{}, nb - st * KB);

#pragma unroll
    for (int i = 0; i < RT; i++) {
#pragma unroll
        for (int j = 0; j < CT; j++) {
            const int n = n0 + wn + 16 * j + i16;
            if (n >= N) continue;
            const float bv = bias ? bias[n] : 0.0f;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int m = (t0 + wt + i) * 16 + 4 * g + r;
                if (m >= M) continue;
                float v = acc[i][j][r];
                if (bias) v = v + bv;
                if (resid) v = resid[(int64_t)m * N + n] + v;  // resid + y, tn_add's operation; resid may be y
                if (y_bf16)
                    reinterpret_cast<uint16_t*>(y)[(int64_t)m * N + n] = bf16_out(v);
                else
                    reinterpret_cast<float*>(y)[(int64_t)m * N + n] = v;
            }
        }
    }
}

template <int FMT, int RT, int CT, int WM, int WN, int KB, int NS, bool DMA = true>
void launch(hipStream_t st, const QGemmArgs& a, const uint8_t* xf, const float* dxf, int mt, int nb) {
    using G = QGeo<FMT, RT, CT, WM, WN, KB, NS>;
    const int64_t wgs = cdiv(mt, G::RTT) * cdiv(a.n, G::BN);
    hipLaunchKernelGGL((k_qgemm<FMT, RT, CT, WM, WN, KB, NS, DMA>), wg_grid(wgs), dim3(QG_TH), 0, st, xf, dxf, (int)a.m, mt, (int)wgs, nb,
                       a.qs, a.d, (int)a.n, a.bias, a.y, a.y_bf16, a.resid);
}

// The tile shapes, by how many 16 x 16 tiles there are for the 1024 SIMDs
// (measured, us; [m, 4096] x [14336, 4096] q4_0 unless stated; the 128 x 128
// tile kernel this one replaced in the last column):
//                                             1x1 64 wide  1x1 KB 8  1x1 KB 4  2x2    before
//   m 16   (one row tile)                         17.9        18.6     22.2   35.6     73.3
//   m 32   (1792 tiles)                           20.1        18.8     22.4   37.0     74.2
//   m 64   (3584)                                 34.5        31.6     31.2   37.3     74.5
//   m 128  (7168)                                 58.2        46.7     48.4   43.3     74.9
//   m 512  (28672)                                204         156      159    123      150
//   q8_0 [200, 1536] x [5000, 1536] (4069)        37.7        24.6     21.7   23.4     61.9
//   q8_0 m 512                                    383         201      164    151      160
// One row tile: four waves side by side (a second row tile would be padding).
// Few tiles: one to a wave, long stages (KB 8) while every SIMD has one or two
// waves; short stages (KB 4) leave LDS for five workgroups on a CU. Many: 2 x 2
// tiles to a wave share their operands' reads.
template <int FMT>
void launch_fmt(hipStream_t st, const QGemmArgs& a, const uint8_t* xf, const float* dxf, int mt, int nb) {
    const int64_t tiles = mt * cdiv(a.n, 16);
    // a code plane off 16 bytes: loads straight to LDS need whole granules ([m, 4096]
    // x [14336, 4096] q4_0, m 16, 128, 512, us: 24.4, 44.9, 126.4; aligned 17.9,
    // 44.5, 123.0)
    if (reinterpret_cast<uintptr_t>(a.qs) % 16 != 0) {
        if (tiles <= 6144) launch<FMT, 1, 1, 2, 2, 4, 4, false>(st, a, xf, dxf, mt, nb);
        else launch<FMT, 2, 2, 2, 2, 4, 3, false>(st, a, xf, dxf, mt, nb);
        return;
    }
    if (mt == 1) launch<FMT, 1, 1, 1, 4, 8, FMT == FMT_Q8_0 ? 3 : 4>(st, a, xf, dxf, mt, nb);
    else if (tiles <= 2560) launch<FMT, 1, 1, 2, 2, 8, 3>(st, a, xf, dxf, mt, nb);
    else if (tiles <= 6144) launch<FMT, 1, 1, 2, 2, 4, 4>(st, a, xf, dxf, mt, nb);
    else launch<FMT, 2, 2, 2, 2, 4, 3>(st, a, xf, dxf, mt, nb);
}

}  // namespace

tn_status qgemm_launch(hipStream_t st, const QGemmArgs& a) {
    // row and tile counts as int, a workgroup's operands under 2^31 bytes
    if (a.m > INT32_MAX - 15 || a.n > INT32_MAX || a.k > INT32_MAX || 4 * (a.k / QK) * 512 > INT32_MAX)
        return fail(TN_EVALUE, "torch._C._quantized_linear: shape too large");
    const int nb = (int)(a.k / QK);
    const int mt = (int)cdiv(a.m, 16);
    const int64_t blocks = (int64_t)mt * 16 * nb;
    if (mt * cdiv(a.n, 32) > INT32_MAX || cdiv(blocks, 64) > INT32_MAX)
        return fail(TN_EVALUE, "torch._C._quantized_linear: shape too large");
    void* ws = nullptr;
    const size_t xbytes = (size_t)blocks * 32;
    TN_TRY(workspace(st, qgemm_workspace(a), &ws));
    uint8_t* xf = static_cast<uint8_t*>(ws);
    float* dxf = reinterpret_cast<float*>(xf + xbytes);
    const float unit = a.fmt == FMT_Q4_0 ? 0.0625f : 1.0f;
    const dim3 grid((unsigned)cdiv(blocks, 64));
#define TN_PRE(XT, XM)                                                                                               \
    hipLaunchKernelGGL((k_q8_frag<XT, XM>), grid, dim3(256), 0, st, static_cast<const XT*>(a.x), (int)a.m, blocks,  \
                       (int)a.k, nb, xf, dxf, unit, a.hd)
    if (a.xm == XM_GLU) TN_PRE(float, XM_GLU);
    else if (a.xm == XM_HEADS) TN_PRE(float, XM_HEADS);
    else if (a.x_bf16) TN_PRE(uint16_t, XM_ROWS);
    else TN_PRE(float, XM_ROWS);
#undef TN_PRE
    TN_LAUNCHED();
    if (a.fmt == FMT_Q4_0) launch_fmt<FMT_Q4_0>(st, a, xf, dxf, mt, nb);
    else launch_fmt<FMT_Q8_0>(st, a, xf, dxf, mt, nb);
    TN_LAUNCHED();
    return TN_OK;
}

}  // namespace tn
