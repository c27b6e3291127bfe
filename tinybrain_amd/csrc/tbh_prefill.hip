// tbh_prefill.hip -- the prefill route (bf16 x of any row count, and fp32 x
// from a per-weight row count): the GEMM of tbh_gemm.h, and the
// register-staged bf16 MFMA GEMM here, gemm_bf16, for few rows of fp32 x or of
// runtime-layout INT4 (use_gemm), for products of few full tiles
// (keep_gemm_bf16) and where the other has no scratch (capture) or rows too
// long for it (gemm_supported).
//
// y[M, N] = x[M, K] (bf16) . dequantize(W)[K, N], fp32 accumulation, for the
// repacked K-contiguous row layout.  This is the one dense contraction of the
// path: the reference runs it as dequantize() + cblas_sgemm on the CPU
// (Sources/TinyBrainRuntime/QuantizedTensor.swift:640-642,
// Tensor.swift:839-861) or as the MSL dequant kernels one output per thread
// (Shaders/Dequant.metal:49-79, DequantINT4.metal:95-137).
//
// A block of four or eight waves owns a BM x BN output tile; its waves, as
// 2 x (waves / 2), own (BM/2) x (BN/(waves/2)) each, as TM x TN tiles of
// v_mfma_f32_16x16x32_bf16 (eight waves: two per SIMD from one block).  Per
// K step of 64 (128 for unsplit INT4 128 x 128 tiles of fp32 x) the block
// stages x (bf16, as given, or its pieces) and the dequantized weight tile in
// LDS; global loads of step t+1 are in flight while step t's MFMAs run.  Weight
// operands are exact:
//   * INT8 (one scale per row): q - zp is an integer of magnitude <= 255,
//     exact in bf16; the row scale multiplies the fp32 result once.
//   * INT4 K-groups: groups are whole multiples of 32 along K, so each
//     32-deep MFMA K-slice lies in one group.  The slice's MFMA takes the
//     integer 16 (q - zp) (exact in bf16) into a zeroed accumulator, and the
//     group scale multiplies that partial product once before it is added
//     to the tile's accumulator; the epilogue multiplies by 1/16.  Scaling
//     every operand of a sum by a power of two commutes with fp32 rounding,
//     so the outputs are those of the unscaled products.
// Accumulation is fp32.
#include "tbh_internal.h"

#include <algorithm>
#include <cstdlib>
#include <type_traits>

namespace tbh {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

constexpr int kBK = 64;           // K per staged step (two MFMA K-steps of 32) unless a launch takes 128
// bf16 of padding per LDS row (32 bytes): rows of 160 (K steps of 64) or 288
// (of 128) bytes.  The MFMA fragment reads (lane l: row l % 16, 16-byte
// column l / 16) measured conflict-free with these strides on gfx950 and
// 2-way conflicted with 144 / 272-byte rows (16 bytes of padding), which
// cost 1-6 % per launch (rocprofv3 SQ_LDS_BANK_CONFLICT per LDS
// instruction 2.98 -> 1.02 on INT8 M = 2048).
constexpr int kRowPad = 16;
constexpr int kDepth = 2;         // K steps whose global loads are in flight at once

struct PParams {
    const uint16_t *x;   // bf16 bits, [M][ldx]
    const float *xf;     // fp32 mode: x as fp32 [Mout][ldx], row r of the product = piece r % 4 of row r / 4
    int64_t ldx;
    float *y;            // [M][ldy]; with split-K, split z writes y + z * split_stride
    int64_t ldy;
    int64_t split_stride;
    int32_t split_steps; // K steps per split (a multiple of kDepth)
    const uint8_t *data;
    int64_t row_bytes;
    const float *scales;
    const int8_t *zp;
    int32_t M, K, N, Np;
    int32_t Mout;    // output rows: M, or M / 4 in fp32 mode
    int32_t chunks;  // 16-byte chunks per row
    int32_t G;       // INT4 K-groups per row
    int32_t cpg;     // chunks per K-group
    int32_t rpn;     // runtime-layout INT4: rows per N-block (scales: [nbk][chunks * 32])
    int32_t nbk;     // runtime-layout INT4: N-blocks
};

__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Two fp32 values -> one dword of two bf16 (upper halves; exact when the low
// halves are zero, else truncation).
__device__ __forceinline__ uint32_t pack_hi16(float lo_elem, float hi_elem) {
    return __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, hi_elem),
                                 __builtin_bit_cast(uint32_t, lo_elem), 0x07060302u);
}

// One 16x16x32 MFMA of eight bf16 operands per lane.
__device__ __forceinline__ f32x4 mfma16(bf16x8 a, bf16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// A 32-bit word as fp32.  By value: __builtin_bit_cast applied directly to
// an element of an ext_vector_type value (v[1]) reads element 0.
__device__ __forceinline__ float as_f32(uint32_t u) { return __builtin_bit_cast(float, u); }

// An fp32 value split exactly into three bf16 values, x = p[0] + p[1] + p[2]:
// p[0] keeps the upper 16 bits of x, p[1] the upper 16 bits of the exact
// remainder x - p[0] (at most 16 significant bits), p[2] the rest (at most 8
// significant bits, so exact in bf16).  Non-finite x stays in p[0].
__device__ __forceinline__ void split3(float x, float (&p)[3]) {
    const uint32_t b = __builtin_bit_cast(uint32_t, x);
    p[0] = __builtin_bit_cast(float, b & 0xFFFF0000u);
    const float r1 = (b & 0x7F800000u) != 0x7F800000u ? x - p[0] : 0.0f;
    p[1] = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, r1) & 0xFFFF0000u);
    p[2] = r1 - p[1];
}

// Byte J of w, read as a signed byte, as fp32 (one sign-extending byte
// select of v_cvt_f32_i32).
template <int J>
__device__ __forceinline__ float sbyte(uint32_t w) {
    return (float)(int8_t)(uint8_t)(w >> (8 * J));
}

// XF = 1 (fp32 x): product row r is piece r % 4 of x row r / 4 (split3;
// piece 3 is zero), so the four rows a lane holds in each 16 x 16
// accumulator tile are the pieces of one x row, and the epilogue adds them
// into that row's output.  XF = 2: the same from bf16 x (widened exactly).
//
// NC > 0: INT4 in the runtime layout (groups along N: one scale per
// (N-block of rpn rows, k)).  The scale varies along K inside an MFMA, so it
// goes on the x side: the tile's NC N-blocks each get their own LDS copy of
// x, copy c holding split3(fl(x[k] * s[nb0 + c][k])) (fp32 product, split
// exactly into three bf16 pieces), and an MFMA of output columns in N-block
// c reads copy c against the exact integers 16 q.  Each term differs from the
// reference's x * fl(q * s) only in which fp32 product is rounded.
//
// Eight-wave blocks with K steps of 64 are held to four waves per SIMD
// (two blocks per CU) where that fits: not the INT4 128 x 128 tiles (about
// 180 VGPRs) nor runtime-layout tiles holding two or more x copies (their
// LDS allows one block per CU).
template <int PREC, int BM, int BN, int WV, int BK, int NC>
constexpr bool kFourWavesPerSimd = WV == 8 && BK == 64 && NC <= 1 && !(PREC == 4 && BM == 128 && BN == 128);

template <int PREC, int BM, int BN, bool ZP, int WV, int BK, int XF, int NC>
__global__ __launch_bounds__(64 * WV) __attribute__((amdgpu_waves_per_eu(kFourWavesPerSimd<PREC, BM, BN, WV, BK, NC> ? 4 : 1)))
void gemm_bf16(const PParams p) {
    static_assert(NC == 0 || (PREC == 4 && XF != 0 && !ZP), "runtime-layout INT4 stages split x, no zero points");
    static_assert(XF != 2 || NC > 0, "bf16 x is split only for runtime-layout scales");
    constexpr int XP = 4;                                   // product rows per x row (split x)
    constexpr int NCC = NC > 0 ? NC : 1;                    // copies of x in LDS
    // Steps wholly inside K and the N tile run an unmasked loop form, except
    // in INT4 blocks with K steps of 128 (256 VGPRs), which run every step
    // masked: with the second form their spilled registers went from 2 to 14-17.
    constexpr bool kTwoForm = !(PREC == 4 && BK == 128);
    constexpr int kLdsRow = BK + kRowPad;
    constexpr int NT = 64 * WV;                   // threads; waves as 2 x (WV / 2)
    constexpr int WC = WV / 2;
    constexpr int CE = PREC == 8 ? 16 : 32;       // elements per chunk
    constexpr int CPR = BK / CE;                 // chunks per row per step
    constexpr int WCH = BN * CPR;                 // weight chunks per step
    constexpr int WPT = (WCH + NT - 1) / NT;      // per thread (last may idle)
    constexpr int XSEG = BM * (BK / 8);          // 16-byte x segments per step
    constexpr int XPT = XSEG / NT;
    constexpr int WM = BM / 2, WN = BN / WC;
    constexpr int TM = WM / 16, TN = WN / 16;
    static_assert(XSEG % NT == 0 && TN >= 1, "tile too small for the waves");

    // two LDS buffers: step t + 1 is staged while step t's MFMAs read
    __shared__ __attribute__((aligned(16))) uint16_t xs[2][NCC][BM * kLdsRow];
    __shared__ __attribute__((aligned(16))) uint16_t ws[2][BN * kLdsRow];
    __shared__ float ssc[2][PREC == 4 && NC == 0 ? BN * CPR : 1];   // INT4 K-groups: scale of each (row, K-slice)

    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int wm = wave / WC, wn = wave % WC;
    const int kpart = blockIdx.z;
    const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
    const int nsteps = (p.chunks * CE + BK - 1) / BK;
    // This block's K steps [t_begin, t_end); x past kend reads as zero, so
    // the padded steps at a split's end add nothing.
    const int t_begin = kpart * p.split_steps;
    const int t_end = min(nsteps, t_begin + p.split_steps);
    const int kend = min(p.K, t_end * BK);

    // INT8 row scales of this lane's output columns, loaded before the K loop;
    // INT4 weights are staged as 16 (q - zp)
    float scn[TN];
#pragma unroll
    for (int b = 0; b < TN; ++b)
        scn[b] = PREC == 8 ? p.scales[min(n0 + wn * WN + b * 16 + (lane & 15), p.Np - 1)] : 0.0625f;

    // ---- global -> registers for one step, into register stage d of kDepth:
    // the loads of steps t+1 .. t+kDepth-1 are in flight while step t runs
    // split x: a segment is 8 elements of one x row (two 16-byte loads of
    // fp32, one of bf16), staged as the four product rows of its pieces; with
    // runtime-layout scales an item is a (segment, copy) pair and also loads
    // the copy's 8 scales
    constexpr int XSEGF = (BM / XP) * (BK / 8);
    constexpr int XPTF = XF ? (XSEGF * NCC + NT - 1) / NT : 1;
    constexpr int XPTL = XF ? XPTF : XPT;
    u32x4 xr[kDepth][XPTL][XF == 1 ? 2 : 1];
    u32x4 xsc[kDepth][NC > 0 ? XPTL : 1][2];
    bool xin[kDepth][XPTL];   // segment within K, applied at the LDS store
    u32x4 wr[kDepth][WPT];
    float sr[kDepth][WPT];
    int8_t zq[kDepth][WPT];
    // Only addresses are computed here; everything that uses a loaded value
    // (masks, conversions) happens in store_step, kDepth - 1 steps later.
    // full (std::true_type): step t lies wholly inside this block's K range
    // and the block's N tile inside the weight, so no address is clamped and
    // no segment masked (the K loop takes this form for all but its last
    // iterations).
    auto load_step = [&](int t, int d, auto full) {
        constexpr bool FULL = decltype(full)::value && !XF && kTwoForm;
        const int k0 = t * BK;
        if constexpr (XF) {
#pragma unroll
            for (int j = 0; j < XPTF; ++j) {
                const int i = min(tid + NT * j, XSEGF * NCC - 1);   // threads past the last item repeat it
                const int s = NCC == 1 ? i : i % XSEGF;
                const int qrow = s / (BK / 8), kq = s % (BK / 8);
                const int m = min(m0 / XP + qrow, p.Mout - 1), k = k0 + 8 * kq;
                const int kk = k < p.K ? k : 0;
                xin[d][j] = k < kend;
                if constexpr (XF == 1) {
                    const float *src = p.xf + (int64_t)m * p.ldx + kk;
                    xr[d][j][0] = *(const u32x4 *)src;
                    xr[d][j][1] = *(const u32x4 *)(src + 4);
                } else {
                    xr[d][j][0] = *(const u32x4 *)(p.x + (int64_t)m * p.ldx + kk);
                }
                if constexpr (NC > 0) {
                    // copy i / XSEGF: N-block n0 / rpn + copy (clamped; tiles
                    // past the last N-block store nothing)
                    const int nb = min(n0 / p.rpn + i / XSEGF, p.nbk - 1);
                    const float *sp = p.scales + (int64_t)nb * (p.chunks * CE) + kk;
                    xsc[d][j][0] = *(const u32x4 *)sp;
                    xsc[d][j][1] = *(const u32x4 *)(sp + 4);
                }
            }
        } else {
#pragma unroll
            for (int j = 0; j < XPT; ++j) {
                const int s = tid + NT * j;
                const int row = s / (BK / 8), kq = s % (BK / 8);
                const int m = min(m0 + row, p.M - 1), k = k0 + 8 * kq;
                // K % 8 == 0: a segment is all in or out.  Rows past M read row
                // M-1 (finite values; their outputs are never stored).
                xin[d][j] = FULL || k < kend;
                xr[d][j][0] = *(const u32x4 *)(p.x + (int64_t)m * p.ldx + (FULL || k < p.K ? k : 0));
            }
        }
#pragma unroll
        for (int j = 0; j < WPT; ++j) {
            const int s = tid + NT * j;
            const int row = s / CPR, c = t * CPR + s % CPR;
            const int n = n0 + row;
            // (the INT4 128-deep kernel keeps the run-time s < WCH test here and in
            // store_step: with it folded, that kernel's register allocation
            // spilled 6-11 more registers)
            const bool in = ((kTwoForm && WCH % NT == 0) || s < WCH) && (FULL || (n < p.Np && c < p.chunks));
            // Out-of-range chunks read a valid chunk: rows past N are never
            // stored and K padding meets x = 0, so the values do not matter.
            const int64_t nn = in ? n : 0, cc = in ? c : 0;
            wr[d][j] = __builtin_nontemporal_load((const u32x4 *)(p.data + nn * p.row_bytes + cc * 16));
            if constexpr (PREC == 4 && NC == 0) {
                const int64_t gi = kgroup_index(nn, cc / p.cpg, p.G);
                sr[d][j] = p.scales[gi];
                if (ZP) zq[d][j] = p.zp[gi];
            } else if constexpr (ZP) {
                zq[d][j] = p.zp[nn];
            }
        }
    };

    // ---- registers -> LDS (x as is; weights dequantized to bf16 pieces)
    auto store_step = [&](int d, int bb, auto full) {
        constexpr bool FULL = decltype(full)::value && !XF && kTwoForm;
        if constexpr (XF) {
            // segment (quad row qrow, kq) of copy i / XSEGF -> product rows
            // 4 qrow + piece
#pragma unroll
            for (int j = 0; j < XPTF; ++j) {
                const int i = tid + NT * j;
                if (i < XSEGF * NCC) {
                    const int s = NCC == 1 ? i : i % XSEGF;
                    const int qrow = s / (BK / 8), kq = s % (BK / 8);
                    float pc[8][3];
#pragma unroll
                    for (int h = 0; h < 8; ++h) {
                        const int e = 4 * (h % 2) + h / 2;   // 0, 4, 1, 5, ...: the two loads' elements alternate
                        float v;
                        if constexpr (XF == 1) {
                            v = as_f32(xr[d][j][e / 4][e % 4]);
                        } else {   // bf16 element e: low half of word e / 2 when e is even
                            const uint32_t wv = xr[d][j][0][e / 2];
                            v = as_f32(e % 2 ? wv & 0xFFFF0000u : wv << 16);
                        }
                        if constexpr (NC > 0) v *= as_f32(xsc[d][j][e / 4][e % 4]);
                        split3(xin[d][j] ? v : 0.0f, pc[e]);
                    }
                    uint16_t *dst = &xs[bb][NCC == 1 ? 0 : i / XSEGF][(4 * qrow) * kLdsRow + 8 * kq];
#pragma unroll
                    for (int piece = 0; piece < 3; ++piece) {
                        uint32_t o[4];
#pragma unroll
                        for (int e = 0; e < 4; ++e) o[e] = pack_hi16(pc[2 * e][piece], pc[2 * e + 1][piece]);
                        *(u32x4 *)(dst + piece * kLdsRow) = u32x4{o[0], o[1], o[2], o[3]};
                    }
                    *(u32x4 *)(dst + 3 * kLdsRow) = u32x4{0, 0, 0, 0};
                }
            }
        } else {
#pragma unroll
            for (int j = 0; j < XPT; ++j) {
                const int s = tid + NT * j;
                const int row = s / (BK / 8), kq = s % (BK / 8);
                *(u32x4 *)&xs[bb][0][row * kLdsRow + 8 * kq] = FULL || xin[d][j] ? xr[d][j][0] : u32x4{0, 0, 0, 0};
            }
        }
#pragma unroll
        for (int j = 0; j < WPT; ++j) {
            const int s = tid + NT * j;
            if ((kTwoForm && WCH % NT == 0) || s < WCH) {
                const int row = s / CPR, cl = s % CPR;
                uint16_t *dst = &ws[bb][row * kLdsRow + cl * CE];
                if (PREC == 8) {
                    // bytes {0,2,1,3} of each word are k+{0,1,2,3}, each stored as
                    // u = q + 128: flipping the top bit of every byte leaves q as a
                    // signed byte.  Value q - zp.
                    const float zf = ZP ? (float)zq[d][j] : 0.0f;
                    uint32_t o[8];
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const uint32_t w = wr[d][j][q] ^ 0x80808080u;
                        const float f0 = sbyte<0>(w) - zf;
                        const float f1 = sbyte<2>(w) - zf;
                        const float f2 = sbyte<1>(w) - zf;
                        const float f3 = sbyte<3>(w) - zf;
                        o[2 * q] = pack_hi16(f0, f1);
                        o[2 * q + 1] = pack_hi16(f2, f3);
                    }
                    *(u32x4 *)dst = u32x4{o[0], o[1], o[2], o[3]};
                    *(u32x4 *)(dst + 8) = u32x4{o[4], o[5], o[6], o[7]};
                } else {
                    // nibble of k % 8 at bit {0,16,4,20,8,24,12,28}, stored as
                    // u = q + 8: flipping the top bit of every nibble leaves q as a
                    // 4-bit two's complement value.  Moved into the upper half of
                    // its byte (high nibbles masked in place, low nibbles shifted
                    // up), a nibble reads as the signed byte 16 q.  Value 16 (q - zp).
                    const float zf = ZP ? 16.0f * (float)zq[d][j] : 0.0f;
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const uint32_t w = wr[d][j][q] ^ 0x88888888u;
                        const uint32_t hi = w & 0xF0F0F0F0u;          // bytes: k + {2, 6, 3, 7}
                        const uint32_t lo = (w << 4) & 0xF0F0F0F0u;   // bytes: k + {0, 4, 1, 5}
                        uint32_t o[4];
                        o[0] = pack_hi16(sbyte<0>(lo) - zf, sbyte<2>(lo) - zf);
                        o[1] = pack_hi16(sbyte<0>(hi) - zf, sbyte<2>(hi) - zf);
                        o[2] = pack_hi16(sbyte<1>(lo) - zf, sbyte<3>(lo) - zf);
                        o[3] = pack_hi16(sbyte<1>(hi) - zf, sbyte<3>(hi) - zf);
                        *(u32x4 *)(dst + 8 * q) = u32x4{o[0], o[1], o[2], o[3]};
                    }
                    if constexpr (NC == 0) ssc[bb][s] = sr[d][j];
                }
            }
        }
    };

    f32x4 acc[TM][TN];
#pragma unroll
    for (int a = 0; a < TM; ++a)
#pragma unroll
        for (int b = 0; b < TN; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};

    // runtime-layout scales: copy c serves the tile's columns [c, c + 1) * BN / NC
    constexpr int kColsPerCopy = BN / NCC;
    constexpr bool kWaveOneCopy = kColsPerCopy >= WN;   // all of a wave's columns in one copy
    static_assert(kColsPerCopy % 16 == 0, "an MFMA's 16 columns lie in one N-block");
    auto compute = [&](int bb) {
#pragma unroll
        for (int ks = 0; ks < BK / 32; ++ks) {
            const int kofs = ks * 32 + 8 * (lane >> 4);
            bf16x8 af[TM];
            if constexpr (kWaveOneCopy) {
                const int cw = NCC == 1 ? 0 : (wn * WN) / kColsPerCopy;
#pragma unroll
                for (int a = 0; a < TM; ++a)
                    af[a] = *(const bf16x8 *)&xs[bb][cw][(wm * WM + a * 16 + (lane & 15)) * kLdsRow + kofs];
            }
#pragma unroll
            for (int b = 0; b < TN; ++b) {
                const int wrow = wn * WN + b * 16 + (lane & 15);
                const bf16x8 bfr = *(const bf16x8 *)&ws[bb][wrow * kLdsRow + kofs];
                if constexpr (!kWaveOneCopy) {
                    const int cb = (wn * WN + b * 16) / kColsPerCopy;
#pragma unroll
                    for (int a = 0; a < TM; ++a)
                        af[a] = *(const bf16x8 *)&xs[bb][cb][(wm * WM + a * 16 + (lane & 15)) * kLdsRow + kofs];
                }
                if (PREC == 8 || NC > 0) {
#pragma unroll
                    for (int a = 0; a < TM; ++a)
                        acc[a][b] = mfma16(af[a], bfr, acc[a][b]);
                } else {
                    const float sc = ssc[bb][wrow * CPR + ks];
#pragma unroll
                    for (int a = 0; a < TM; ++a) {
                        const f32x4 part = mfma16(af[a], bfr, f32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
                        for (int e = 0; e < 4; ++e) acc[a][b][e] = __builtin_fmaf(part[e], sc, acc[a][b][e]);
                    }
                }
            }
        }
    };

    // Register ring slot s holds a step's global loads; LDS buffer t % 2 holds
    // step t.  Each iteration stages step t + 1 from its slot into the other
    // buffer, refills that slot with step t + 3, computes step t, and ends with
    // the one barrier of the step (step t + 1 visible, step t's reads done).
    // Steps are padded to a multiple of kDepth and every iteration loads and
    // computes unconditionally: steps past K read clamped addresses and meet
    // x = 0, so they add nothing, and the loop body has no branches at which
    // the compiler would have to wait for every load in flight.  (Rings of
    // four steps measured slower: INT8 5632x2048 at M = 2048 76.2 -> 84.7 us,
    // M = 512 31.6 -> 32.4 us; six steps for split launches, INT8 M = 64
    // 14.7 -> 18.6 us.)
    // The iterations whose four steps t0 + 1 .. t0 + 4 all lie below t_full
    // (inside K, in a full N tile) run without clamps or masks.
    static_assert(kDepth == 2, "two register slots, two LDS buffers");
    const int t_stop = t_begin + ((t_end - t_begin + kDepth - 1) / kDepth) * kDepth;
    const std::false_type part;
    load_step(t_begin, 0, part);
    load_step(t_begin + 1, 1, part);
    store_step(0, 0, part);
    lds_barrier();
    load_step(t_begin + 2, 0, part);
    // A step is staged before the one before it is computed: the other order
    // spills the INT4 kernels' registers (M = 128 17.9 -> 27.3 us) and the
    // fp32-x form's (M = 128 31.2 -> 32.2 us).
    auto iteration = [&](int t0, auto full) {
        store_step(1, 1, full);        // step t0 + 1
        load_step(t0 + 3, 1, full);
        compute(0);                    // step t0
        lds_barrier();
        store_step(0, 0, full);        // step t0 + 2
        load_step(t0 + 4, 0, full);
        compute(1);                    // step t0 + 1
        lds_barrier();
    };
    if constexpr (kTwoForm) {
        const int t_full = n0 + BN <= p.Np ? kend / BK : 0;
        int t0 = t_begin;
        for (; t0 < t_stop && t0 + 4 < t_full; t0 += 2) iteration(t0, std::true_type{});
        for (; t0 < t_stop; t0 += 2) iteration(t0, part);
    } else {
        // the same iteration written out (measured 1-2 % faster than the
        // lambda call in this kernel: INT4 2048x5632 at M = 2048 84.8 against
        // 86.6 us)
        for (int t0 = t_begin; t0 < t_stop; t0 += 2) {
            store_step(1, 1, part);
            load_step(t0 + 3, 1, part);
            compute(0);
            lds_barrier();
            store_step(0, 0, part);
            load_step(t0 + 4, 0, part);
            compute(1);
            lds_barrier();
        }
    }

    // ---- epilogue: lane holds C[4 (lane / 16) + e][lane % 16] of each tile
    float *out = p.y + (int64_t)blockIdx.z * p.split_stride;
    const int mrow = m0 + wm * WM + 4 * (lane >> 4), ncol = n0 + wn * WN + (lane & 15);
    if constexpr (XF) {
        // the lane's four rows are the pieces of x row (mrow + 16 a) / 4
#pragma unroll
        for (int b = 0; b < TN; ++b) {
            const int n = ncol + b * 16;
            if (n >= p.N) continue;
#pragma unroll
            for (int a = 0; a < TM; ++a) {
                const int m = (mrow + a * 16) >> 2;
                const float v = ((acc[a][b][0] + acc[a][b][1]) + acc[a][b][2]) + acc[a][b][3];
                if (m < p.Mout) out[(int64_t)m * p.ldy + n] = v * scn[b];
            }
        }
        return;
    }
    if (m0 + BM <= p.M && n0 + BN <= p.N) {
        // whole tile in range: no per-element branches
#pragma unroll
        for (int b = 0; b < TN; ++b)
#pragma unroll
            for (int a = 0; a < TM; ++a)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    out[(int64_t)(mrow + a * 16 + e) * p.ldy + ncol + b * 16] = acc[a][b][e] * scn[b];
    } else {
#pragma unroll
        for (int b = 0; b < TN; ++b) {
            const int n = ncol + b * 16;
            if (n >= p.N) continue;
#pragma unroll
            for (int a = 0; a < TM; ++a)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int m = mrow + a * 16 + e;
                    if (m < p.M) out[(int64_t)m * p.ldy + n] = acc[a][b][e] * scn[b];
                }
        }
    }
}

// y = sum over splits of the partial tiles, in split order (deterministic).
// S > 0: exactly S splits, loaded together before they are added, so a sum
// costs one memory round trip; S = 0: any number, kSumBatch at a time (clamped
// addresses, selected afterwards).
constexpr int kSumBatch = 16;

template <class V, int S>
__global__ __launch_bounds__(256) void split_sum(const V *__restrict__ part, int64_t stride, int splits,
                                                 V *__restrict__ y, int64_t n) {
    constexpr int E = sizeof(V) / sizeof(float), B = S > 0 ? S - 1 : kSumBatch;
    auto add = [](V &v, const V &u) {
#pragma unroll
        for (int c = 0; c < E; ++c) ((float *)&v)[c] += ((const float *)&u)[c];
    };
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        V v = part[i];
        for (int z0 = 1; z0 < (S > 0 ? 2 : splits); z0 += B) {
            V u[B];
#pragma unroll
            for (int j = 0; j < B; ++j) u[j] = part[(S > 0 ? 1 + j : min(z0 + j, splits - 1)) * stride + i];
#pragma unroll
            for (int j = 0; j < B; ++j)
                if (S > 0 || z0 + j < splits) add(v, u[j]);
        }
        y[i] = v;
    }
}

template <class V>
void sum_splits(const float *part, int splits, float *y, int64_t n, int64_t cus, hipStream_t s) {
    // blocks of one wave while those do not fill the chip: a block per CU
    // needs 16384 threads, where blocks of four waves would leave most idle
    const int64_t threads = n <= 16 * 64 * cus ? 64 : 256;
    const dim3 grid((unsigned)std::min(16 * cus, (n + threads - 1) / threads)), block((unsigned)threads);
    const V *p = (const V *)part;
    V *o = (V *)y;
    switch (splits) {
    case 2: hipLaunchKernelGGL((split_sum<V, 2>), grid, block, 0, s, p, n, splits, o, n); break;
    case 3: hipLaunchKernelGGL((split_sum<V, 3>), grid, block, 0, s, p, n, splits, o, n); break;
    case 4: hipLaunchKernelGGL((split_sum<V, 4>), grid, block, 0, s, p, n, splits, o, n); break;
    case 5: hipLaunchKernelGGL((split_sum<V, 5>), grid, block, 0, s, p, n, splits, o, n); break;
    case 6: hipLaunchKernelGGL((split_sum<V, 6>), grid, block, 0, s, p, n, splits, o, n); break;
    case 7: hipLaunchKernelGGL((split_sum<V, 7>), grid, block, 0, s, p, n, splits, o, n); break;
    case 8: hipLaunchKernelGGL((split_sum<V, 8>), grid, block, 0, s, p, n, splits, o, n); break;
    default: hipLaunchKernelGGL((split_sum<V, 0>), grid, block, 0, s, p, n, splits, o, n); break;
    }
}

template <int PREC, int BM, int BN, int BK, int NC>
hipError_t launch_tile(const PParams &p, int splits, hipStream_t s) {
    static const int waves = [] {   // 4 or 8 forces the waves per block
        const char *v = std::getenv("TBH_PREFILL_WAVES");
        return v && *v ? std::atoi(v) : 0;
    }();
    const dim3 grid((unsigned)((p.Np + BN - 1) / BN), (unsigned)((p.M + BM - 1) / BM), (unsigned)splits);
    if constexpr (NC > 0) {   // runtime-layout INT4: split x (fp32, or bf16 widened)
        constexpr int WVN = BM == 128 ? 8 : 4;
        if (p.xf) hipLaunchKernelGGL((gemm_bf16<4, BM, BN, false, WVN, BK, 1, NC>), grid, dim3(64 * WVN), 0, s, p);
        else hipLaunchKernelGGL((gemm_bf16<4, BM, BN, false, WVN, BK, 2, NC>), grid, dim3(64 * WVN), 0, s, p);
    } else if (p.xf) {   // fp32 x as three bf16 pieces and a zero row
        const bool w8 = waves == 8 || (waves != 4 && BN == 128 && (p.M >= 256 || PREC == 4));
        if (p.zp) {
            if (w8) hipLaunchKernelGGL((gemm_bf16<PREC, BM, BN, true, 8, BK, 1, 0>), grid, dim3(512), 0, s, p);
            else hipLaunchKernelGGL((gemm_bf16<PREC, BM, BN, true, 4, BK, 1, 0>), grid, dim3(256), 0, s, p);
        } else {
            if (w8) hipLaunchKernelGGL((gemm_bf16<PREC, BM, BN, false, 8, BK, 1, 0>), grid, dim3(512), 0, s, p);
            else hipLaunchKernelGGL((gemm_bf16<PREC, BM, BN, false, 4, BK, 1, 0>), grid, dim3(256), 0, s, p);
        }
    } else if constexpr (BN == 128 && BK == kBK && (PREC == 4 || BM == 128)) {   // bf16 x
        if (p.zp) hipLaunchKernelGGL((gemm_bf16<PREC, BM, BN, true, 8, BK, 0, 0>), grid, dim3(512), 0, s, p);
        else hipLaunchKernelGGL((gemm_bf16<PREC, BM, BN, false, 8, BK, 0, 0>), grid, dim3(512), 0, s, p);
    } else {
        return hipErrorInvalidValue;   // launch_prec takes bf16 x to no other tile
    }
    return hipGetLastError();
}

// Blocks a split-K launch aims for, per CU: `dflt` unless
// TBH_PREFILL_BLOCKS_PER_CU is set (0 disables split-K).
int blocks_per_cu(int dflt) {
    static const int v = [] {
        const char *e = std::getenv("TBH_PREFILL_BLOCKS_PER_CU");
        return e ? std::max(0, std::atoi(e)) : -1;
    }();
    return v >= 0 ? v : dflt;
}

constexpr int kMinSplitK = 256;  // K a split keeps at least

}  // namespace

// y[0, n) = the sum of `splits` partial arrays part + z n, in split order.
hipError_t launch_split_sum(const float *part, int splits, float *y, int64_t n, int64_t cus, hipStream_t s) {
    if (n % 4 == 0 && ((uintptr_t)y & 15) == 0) sum_splits<float4>(part, splits, y, n / 4, cus, s);
    else sum_splits<float>(part, splits, y, n, cus, s);
    return hipGetLastError();
}

namespace {

// K is split over blocks when there are fewer than bpc blocks per CU.  BK:
// K per staged step (64 or 128).
template <int PREC, int BM, int BN, int BK = kBK, int NC = 0>
hipError_t launch_split(const tbh_weight &w, PParams p, int64_t tiles, int bpc, hipStream_t s,
                        const Scratch &scr) {
    const int nsteps = (int)((p.chunks * (PREC == 8 ? kInt8ChunkElems : kInt4ChunkElems) + BK - 1) / BK);
    const int64_t cus = std::max(1, w.dev->cu_count);
    int splits = 1, sps = nsteps;
    bpc = blocks_per_cu(bpc);
    if (tiles < bpc * cus && p.ldy == p.N) {
        const int64_t want = (bpc * cus + tiles - 1) / tiles;
        sps = (int)std::max<int64_t>(kMinSplitK / BK, (nsteps + want - 1) / want);
        sps = (sps + kDepth - 1) / kDepth * kDepth;
        splits = (nsteps + sps - 1) / sps;
    }
    float *const y = p.y;
    const int64_t n = (int64_t)p.Mout * p.N;
    float *part = nullptr;
    if (splits > 1) {
        part = (float *)scr.get(s, (size_t)(splits * n) * sizeof(float));
        if (!part && scr.is_fixed()) return hipErrorOutOfMemory;
        if (!part) {          // no workspace (graph capture before any eager call): one pass
            splits = 1;
            sps = nsteps;
        }
    }
    p.split_steps = sps;
    if (splits > 1) {
        p.y = part;
        p.split_stride = n;
    }
    hipError_t e = launch_tile<PREC, BM, BN, BK, NC>(p, splits, s);
    if (e != hipSuccess || splits == 1) return e;
    return launch_split_sum(part, splits, y, n, cus, s);
}

template <int PREC>
hipError_t launch_prec(const tbh_weight &w, const PParams &p, hipStream_t s, const Scratch &scr) {
    const int64_t cus = std::max(1, w.dev->cu_count);
    const int64_t t128 = ((p.Np + 127) / 128) * ((p.M + 127) / 128);
    const int64_t t64x128 = ((p.Np + 127) / 128) * ((p.M + 63) / 64);
    const int64_t t64 = ((p.Np + 63) / 64) * ((p.M + 63) / 64);
    // bf16 x, eight waves a block, split along K to a block per CU: INT4 of few
    // full tiles (keep_gemm_bf16), 64 x 128 below 256 rows (2048x5632: M = 64
    // 16.9 -> 14.9 us, M = 128 22.2 -> 18.5 us; 128 x 128 there 18.1 -> 20.4), and
    // rows too long for launch_gemm
    if (!p.xf) {
        if constexpr (PREC == 4) {
            if (p.M < 256) return launch_split<PREC, 64, 128>(w, p, t64x128, 1, s, scr);
        }
        return launch_split<PREC, 128, 128>(w, p, t128, 1, s, scr);
    }
    static const int force = [] {   // fp32 x: 1: 64 x 64, 2: 64 x 128, 3: 128 x 128 tiles
        const char *v = std::getenv("TBH_PREFILL_TILE");
        return v && *v ? std::atoi(v) : 0;
    }();
    if (force == 1) return launch_split<PREC, 64, 64>(w, p, t64, 2, s, scr);
    if (force == 2) return launch_split<PREC, 64, 128>(w, p, t64x128, 1, s, scr);
    if (force == 3) return launch_split<PREC, 128, 128>(w, p, t128, 1, s, scr);
    // fp32 x, four product rows per x row: up to 64 x rows, or any number that
    // finds no scratch for launch_gemm.
    if (p.M >= 256) {
        // Timestamps inside the kernel showed a block with one wave per SIMD
        // spending three quarters of each K step on global-load waits,
        // dequantization, LDS traffic and barriers that nothing overlaps;
        // two blocks on a CU took 1.2x the time of one.  So: 128 x 128 tiles
        // as 8-wave blocks (two waves per SIMD) when they give every CU a
        // block; else, for INT8, 64 x 64 tiles when they give two blocks per
        // CU without a K split (64 x 128 tiles never do here: there are at
        // most twice as many as 128 x 128 tiles, which are fewer than the
        // CUs); else 128 x 128 split along K to a block per CU.
        // INT4 128 x 128 tiles without a K split stage K steps of 128 (half
        // the barriers and loop trips per flop; its group scale per MFMA
        // makes each step's VALU work larger: 2048x5632 at 2048 product rows
        // 90.4 -> 84.1 us; INT8 79.0 -> 79.9).
        if (t128 >= cus)
            return PREC == 4 ? launch_split<PREC, 128, 128, 128>(w, p, t128, 1, s, scr)
                             : launch_split<PREC, 128, 128>(w, p, t128, 1, s, scr);
        if (PREC == 8 && t64 >= 2 * cus) return launch_split<PREC, 64, 64>(w, p, t64, 2, s, scr);
        return launch_split<PREC, 128, 128>(w, p, t128, 1, s, scr);
    }
    // Fewer rows (HBM-bound).  INT4, whose K steps carry a group scale per
    // MFMA: 128 x 128 tiles from 32 x rows (2048x5632 at 32 rows 16.6 -> 14.8
    // us), else 64 x 128, as 8-wave blocks, split along K to a block per CU.
    // INT8: the largest tile that still gives every CU a block; below that, 64
    // x 64 tiles split along K until there are two blocks per CU (a 64 x 64
    // block does little work per K step, so one per CU leaves its latency
    // exposed).
    if (PREC == 4 && p.M >= 128) return launch_split<PREC, 128, 128>(w, p, t128, 1, s, scr);
    if (PREC == 4) return launch_split<PREC, 64, 128>(w, p, t64x128, 1, s, scr);
    if (t128 >= cus) return launch_split<PREC, 128, 128>(w, p, t128, 1, s, scr);
    if (t64x128 >= cus) return launch_split<PREC, 64, 128>(w, p, t64x128, 1, s, scr);
    return launch_split<PREC, 64, 64>(w, p, t64, 2, s, scr);
}

// Copies of x a 64-column tile of a runtime-layout INT4 weight needs (its
// N-blocks), or 0 when the N-blocks do not tile the 64 columns evenly.
int ng_copies(const tbh_weight &w) {
    const int64_t rpn = w.rows_per_nblock;
    if (rpn >= w.Np || rpn % 64 == 0) return 1;
    if (rpn == 32) return 2;
    if (rpn == 16) return 4;
    return 0;
}

// Runtime-layout INT4 (one scale per (N-block, k)) with x given as p.x (bf16)
// or p.xf (fp32), p.M = 4 * x rows: 64 x 64 tiles (16 x rows by 64 outputs,
// four waves) or 128 x 64 tiles (32 x rows, eight waves), split along K when
// the tiles are fewer than the CUs.
hipError_t launch_ngroup(const tbh_weight &w, PParams p, hipStream_t s, const Scratch &scr) {
    p.rpn = w.rows_per_nblock;
    p.nbk = (int32_t)((w.Np + w.rows_per_nblock - 1) / w.rows_per_nblock);
    const int64_t tiles = ((p.Np + 63) / 64) * ((p.M + 63) / 64);
    // past 16 x rows (64 product rows): 128 x 64 tiles as 8-wave blocks,
    // which re-read the weights half as often (2048x5632, N-blocks of 32, us
    // per call 64 / 128 product rows: M = 64 28.1 / 24.6, M = 128 49.2 /
    // 41.0, M = 512 160.1 / 133.9, M = 2048 598 / 508); with four copies of
    // x the 128-row tile does not fit the LDS
    if (p.M > 64) {
        const int64_t t128 = ((p.Np + 63) / 64) * ((p.M + 127) / 128);
        switch (ng_copies(w)) {
        case 1: return launch_split<4, 128, 64, kBK, 1>(w, p, t128, 1, s, scr);
        case 2: return launch_split<4, 128, 64, kBK, 2>(w, p, t128, 1, s, scr);
        default: break;
        }
    }
    switch (ng_copies(w)) {
    case 1: return launch_split<4, 64, 64, kBK, 1>(w, p, tiles, 2, s, scr);
    case 2: return launch_split<4, 64, 64, kBK, 2>(w, p, tiles, 2, s, scr);
    case 4: return launch_split<4, 64, 64, kBK, 4>(w, p, tiles, 2, s, scr);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace

bool prefill_supported(const tbh_weight &w) {
    if (w.mfma_tiles) return false;
    if (w.path == Path::Int4NGroup) return !w.ng_pairs && !w.zp && ng_copies(w) > 0;
    return w.path == Path::Int8Row || w.path == Path::Int4KGroup;
}

static PParams prefill_params(const tbh_weight &w, int64_t ldx, float *y, int64_t ldy) {
    PParams p{};
    p.ldx = ldx;
    p.y = y;
    p.ldy = ldy;
    p.data = w.data;
    p.row_bytes = w.row_bytes;
    p.scales = w.scales;
    p.zp = w.zp;
    p.K = (int32_t)w.K;
    p.N = (int32_t)w.N;
    p.Np = (int32_t)w.Np;
    const bool int8 = w.precision == TBH_PREC_INT8;
    p.chunks = (int32_t)(w.Kp / (int8 ? kInt8ChunkElems : kInt4ChunkElems));
    p.G = (int32_t)w.groups_per_row;
    p.cpg = w.chunks_per_group;
    return p;
}

// Rows of x per GEMM launch.  The grid's second dimension counts row tiles,
// and the fp32 and runtime-layout forms run up to four product rows per x
// row in 32-bit row indices; longer x is taken in chunks of this many rows, one
// launch (and split sum) after the other on the caller's stream.
constexpr int64_t kGemmRowsPerLaunch = (int64_t)1 << 18;

static hipError_t launch_rows(const tbh_weight &w, PParams &p, hipStream_t s, const Scratch &scr) {
    if (w.path == Path::Int4NGroup) return launch_ngroup(w, p, s, scr);
    return w.precision == TBH_PREC_INT8 ? launch_prec<8>(w, p, s, scr) : launch_prec<4>(w, p, s, scr);
}

// Whether `rows` rows of fp32 x (or of bf16 x on a runtime-layout weight) go
// to launch_gemm, whose extra pass over x (2.5-3 us) and 64-row tiles lose to
// gemm_bf16 on few rows of a small weight.  Runtime-layout weights go from 65
// rows: launch_gemm holds both x and weights to 22 bits, where gemm_bf16 splits
// fl(x * s) exactly.  us per call of fp32 x, gemm_bf16 / launch_gemm: INT4
// 2048x2048 63 rows 12.2 / 14.8, 80 17.4 / 15.2; 5632x2048 16 rows 12.4 / 14.6,
// 20 18.7 / 15.7; 2048x5632 24 rows 16.2 / 17.0, 48 20.8 / 18.0; 1024x8192 48
// rows 16.9 / 17.8; 11008x4096 16 rows 30.3 / 27.5; INT8 5632x2048 24 rows 14.8 /
// 20.8; 4096x11008 16 rows 22.3 / 30.6, 24 39.0 / 30.8.
static bool use_gemm(const tbh_weight &w, int64_t rows) {
    const int64_t nk = w.N * w.K;
    if (rows > 64) return true;
    if (w.path == Path::Int4NGroup) return false;
    if (w.path == Path::Int8Row) return rows > 16 && nk >= (int64_t)32 << 20;
    return nk >= (int64_t)32 << 20 || (nk >= (int64_t)10 << 20 && rows > (w.N >= 4096 ? 16 : 32));
}

// Whether `rows` rows of bf16 x on an INT4 K-group weight stay on gemm_bf16:
// its 128 x 128 tiles, split along K, take a long-K product of a small output
// in one full round of blocks, where a block's step is bound by unpacking,
// scales and MFMA alike in both kernels and launch_gemm's longer pipeline only
// adds its start.  us, gemm_bf16 / launch_gemm on 256 CUs:
//   64 tiles (four K parts): 2048x5632 512 rows 30.4 / 33.2, 4096x4096 256 28.7 /
//     32.3, 1024x4096 1024 25.3 / 28.8, 1024x8192 1024 39.5 / 38.4
//   32 tiles (eight): 1024x8192 512 rows 27.6 / 30.6, 2048x8192 256 27.7 / 30.7,
//     1024x4096 512 19.6 / 19.5, 2048x5632 256 23.8 / 23.9
//   128 tiles (two): K of 4096 as above (4096x4096 512 rows 37.4 / 40.2, 2048x4096
//     1024 39.2 / 40.7, 1024x4096 2048 37.9 / 40.2), but each part's steps beyond
//     that are slower (1024x4800 2048 47.6 / 46.5, 2048x5632 1024 46.9 / 45.8,
//     1024x8192 2048 64.8 / 56.8)
//   16 tiles: 2048x5632 128 rows 17.9 / 17.2, 1024x4096 256 19.1 / 14.9; 256
//     (unsplit): 4096x4096 1024 60.3 / 55.5
//   other counts leave a part-filled round: 2048x5632 384 rows 34.1 / 27.9,
//     3072x4096 512 46.2 / 37.2, 1536x6144 512 40.2 / 30.3
// Shorter or larger products are launch_gemm's: 2048x2048 512 rows 22.6 / 20.3,
// 4096x11008 256 54.3 / 50.2.
static bool keep_gemm_bf16(const tbh_weight &w, int64_t rows) {
    const int64_t cus = std::max(1, w.dev->cu_count), tiles = ((w.N + 127) / 128) * ((rows + 127) / 128);
    return w.path == Path::Int4KGroup && w.K >= 4096 && w.N * w.K <= (int64_t)16 << 20 &&
           (8 * tiles == cus || 4 * tiles == cus || (2 * tiles == cus && w.K < 4608));
}

// x [M][ldx] (fp32, or bf16) through launch_gemm, in calls whose pieces take
// kPiecesBytes at most (or 64 rows).  The calls share the rows evenly: a short
// last one would run a small product's plan behind a large one's.
// hipErrorNotReady, with nothing enqueued, when scratch is not to be had.
constexpr size_t kPiecesBytes = (size_t)128 << 20;
static hipError_t gemm_rows(const tbh_weight &w, const void *x, bool f32, int64_t ldx, int64_t M, float *y, int64_t ldy,
                            hipStream_t s, const Scratch &scr) {
    const int pieces = gemm_pieces(w, f32, M);
    int64_t most = kGemmRowsPerLaunch;
    if (pieces > 0) {
        const int64_t per64 = (int64_t)(64 * pieces * 2) * ((w.K + 63) / 64 * 64);
        most = std::min(most, std::max<int64_t>(1, (int64_t)kPiecesBytes / per64) * 64);
    }
    const int64_t calls = (M + most - 1) / most;
    const int64_t rows = ((M + calls - 1) / calls + 63) / 64 * 64;
    for (int64_t m0 = 0; m0 < M; m0 += rows) {
        const int64_t mc = std::min(rows, M - m0);
        const hipError_t e = launch_gemm(w, (const char *)x + m0 * ldx * (f32 ? 4 : 2), f32, pieces, ldx, mc,
                                         y + m0 * ldy, ldy, s, scr);
        if (e != hipSuccess) return m0 > 0 && e == hipErrorNotReady ? hipErrorOutOfMemory : e;
    }
    return hipSuccess;
}

hipError_t launch_prefill_f32(const tbh_weight &w, const float *x, int64_t ldx, int64_t M, float *y,
                              int64_t ldy, hipStream_t s, const Scratch &scr) {
    if (!prefill_supported(w) || M < 1 || w.K % 8 != 0 || ldx % 4 != 0 || ((uintptr_t)x & 15) != 0)
        return hipErrorInvalidValue;
    // launch_gemm: every x row as two f16 pieces scaled by a power of two per
    // row, or as three bf16 pieces up to 64 rows; gemm_bf16 (three bf16 pieces
    // and a zero row) for few rows or when scratch is not to be had (graph
    // capture before any eager call).
    // (16 rows of pieces fit the no-allocation entry's scratch, so that its
    // results are the device entry's)
    if (gemm_supported(w) && use_gemm(w, M) && gemm_pieces_bytes(w, 3, 16) <= kNoAllocScratchBytes) {
        const hipError_t e = gemm_rows(w, x, true, ldx, M, y, ldy, s, scr);
        if (e != hipErrorNotReady) return e;
    }
    for (int64_t m0 = 0; m0 < M; m0 += kGemmRowsPerLaunch) {
        const int64_t mc = std::min(kGemmRowsPerLaunch, M - m0);
        PParams p = prefill_params(w, ldx, y + m0 * ldy, ldy);
        p.xf = x + m0 * ldx;
        p.M = (int32_t)(4 * mc);
        p.Mout = (int32_t)mc;
        const hipError_t e = launch_rows(w, p, s, scr);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

hipError_t launch_prefill(const tbh_weight &w, const uint16_t *x, int64_t ldx, int64_t M, float *y,
                          int64_t ldy, hipStream_t s, const Scratch &scr) {
    if (!prefill_supported(w) || M < 1 || w.K % 8 != 0 || ldx % 8 != 0 || ((uintptr_t)x & 15) != 0)
        return hipErrorInvalidValue;
    // INT8 rows and INT4 K-groups take bf16 x as it is; runtime-layout INT4
    // takes it as one scaled f16 piece, or (few rows, or no scratch) as three
    // bf16 pieces of fl(x * s).
    const bool ng = w.path == Path::Int4NGroup;
    if (gemm_supported(w) && (ng ? use_gemm(w, M) : !keep_gemm_bf16(w, M))) {
        const hipError_t e = gemm_rows(w, x, false, ldx, M, y, ldy, s, scr);
        if (e != hipErrorNotReady) return e;
    }
    for (int64_t m0 = 0; m0 < M; m0 += kGemmRowsPerLaunch) {
        const int64_t mc = std::min(kGemmRowsPerLaunch, M - m0);
        PParams p = prefill_params(w, ldx, y + m0 * ldy, ldy);
        p.x = x + m0 * ldx;
        p.M = (int32_t)((ng ? 4 : 1) * mc);
        p.Mout = (int32_t)mc;
        const hipError_t e = launch_rows(w, p, s, scr);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace tbh
