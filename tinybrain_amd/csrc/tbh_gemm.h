// tbh_gemm.h -- the prefill GEMM kernel y[M, N] = x[M, K] . dequantize(W)[K, N]
// (K-contiguous row layout of the weights, 16-bit x in one or two pieces) and
// its launcher; instantiated per weight kind in tbh_gemm_*.hip.
//
// A block of eight waves owns BM = 16 TM rows of x and BN = 128 TN outputs;
// every wave takes all BM rows of its own 16 TN outputs, so each weight is
// unpacked by exactly one wave per block, and x, which all waves read, is the
// only operand shared.  Per K step of 64, x (16-bit) and the packed weights
// with their scales go from memory straight into LDS (buffer loads with the
// LDS bit: no registers, no VALU work), NB - 1 steps ahead of their use; a
// wave reads its weights as packed integers, unpacks them in registers into
// MFMA operands and multiplies them by the x fragments.  LDS rows of x are
// 128 bytes with the 16-byte segment index XORed with row % 8: the fragment
// reads (16 rows x 4 consecutive segments) are conflict-free (measured 475
// B/ns per CU, the same as 160-byte rows; unswizzled 151).
//
// Why waves side by side along N, not in a 2 x 4 grid: unpacking (INT8 7
// VALU instructions per four weights, INT4 9-16 per eight, runtime-layout
// INT4 about 90 per eight) is then done once per block instead of twice, and
// the LDS read rate (2 TM KiB per wave and 32-deep slice) stays under half of
// the LDS's for TN = 2.
//
// Operands: A = weights, B = x, so lane l holds outputs 4 (l / 16) + e, e =
// 0..3, of x row l % 16 in each 16 x 16 accumulator tile: four neighbouring
// outputs, one 16-byte store.
#pragma once

#include "tbh_internal.h"

#include <algorithm>
#include <cstdint>
#include <type_traits>

namespace tbh {
namespace gemm {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

// Weight kinds: INT8 rows, INT4 with scales along K, runtime-layout INT4
// (scales per N-block and k).
enum Kind { W8 = 0, W4K = 1, W4N = 2 };

constexpr int kBK = 64;             // K per step
constexpr int kWaves = 8;
// Every buffer holds less than 2^30 bytes; offsets past it read as zero.  A
// lane's offset kFar and a step's offset kDead do not wrap together.
constexpr uint32_t kFar = 0x80000000u, kDead = 0x40000000u;

struct Args {
    const uint16_t *x;       // [XP][rows][ldx]: bf16 (XP = 1; XP = 3, exact pieces) or f16 (W4N; XP = 2)
    int64_t ldx;             // elements
    int64_t piece_stride;    // elements between two pieces
    float *y;                // [M][ldy]; split z writes y + z * split_stride
    int64_t ldy;
    int64_t split_stride;
    const uint8_t *data;
    int64_t row_bytes;
    const float *scales;     // W8 [Np]; W4K [Np / 4][G][4]; W4N [nbk][kp] scaled by 2^(8 - e_b)
    int64_t scale_bytes;
    const int8_t *zp;        // W8 [Np]; W4K as scales; or NULL
    const int32_t *row_exp;  // f16 pieces: per x row e with |x| < 2^e
    const int32_t *nb_exp;   // W4N: per N-block e_b
    int32_t M, K, N, Np;
    int32_t xk;              // elements of an x row that may be read (K; padded rows: their length)
    int32_t chunks;          // 16-byte weight chunks per row
    int32_t G;               // W4K: groups per row
    uint64_t cpg_magic;      // W4K: 2^32 / chunks per group, rounded up
    int32_t rpn, kp;         // W4N: rows per N-block, padded K
    int32_t nsteps, split_steps;
    int32_t tiles_m, tiles_n;
    int32_t n_fast;          // tile order: neighbouring tiles share x rows (1) or weight rows (0)
    // blocks [0, main_blocks) take whole (tile, split) items; the rest are the
    // tail: tile tail_first + q / tail_parts over K steps [j tail_steps, ..),
    // j = q % tail_parts, written to tail_part[j][q / tail_parts][BM][BN]
    int32_t main_blocks, tail_first, tail_parts, tail_steps, tail_n;
    float *tail_part;
    int32_t vec;             // y rows take 16-byte stores
    // One part at a time without partial tiles (seq): the tiles of tile rows
    // [seq_tm, seq_tm + seq_tms), whose x rows [row_base, row_end) the pieces
    // hold, over K steps [seq_part * seq_steps, ..); only the tail's tiles
    // (seq_tail) or only the others, the rest return.  add: y += the part, so
    // that part after part gives the bits of their sum in part order.
    int32_t seq, seq_tm, seq_tms, seq_part, seq_steps, seq_tail, add;
    int32_t row_base, row_end;
};

__device__ __forceinline__ i32x4 make_rsrc(const void *p, int bytes) {
    const uint64_t a = (uint64_t)p;
    const int n = max(bytes, 0);
    // base (48 bits, stride 0: raw buffer), size, 32-bit data format
    return i32x4{__builtin_amdgcn_readfirstlane((int)(uint32_t)a),
                 __builtin_amdgcn_readfirstlane((int)((uint32_t)(a >> 32) & 0xFFFFu)),
                 __builtin_amdgcn_readfirstlane(n), 0x00020000};
}

// 16 (or 4) bytes per active lane from buffer offset `off` + `soff` to LDS
// byte lds + 16 (4) * lane; offsets past the buffer's size write zeros.  No
// register receives the load; completion is waited for by dma_wait.  (One
// wait state between the write of M0 and the load that reads it.  M0 is a
// reserved register, which the compiler neither allocates nor takes as a
// clobber; the built kernels use it in these statements only.)
__device__ __forceinline__ void dma16(uint32_t lds, i32x4 r, uint32_t off, uint32_t soff) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(lds), "v"(off), "s"(r),
                 "s"(soff) : "memory");
}
// The same from the lanes of `mask` alone, 16 or 4 bytes a lane (called with
// every lane active, as EXEC is left, and without a branch that would end the
// basic block the surrounding instructions are scheduled in).
template <int BYTES>
__device__ __forceinline__ void dma_lanes(uint32_t lds, i32x4 r, uint32_t off, uint32_t soff, uint64_t mask) {
    if constexpr (BYTES == 16)
        asm volatile("s_mov_b32 m0, %0\n\ts_mov_b64 exec, %4\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds\n\t"
                     "s_mov_b64 exec, -1" ::"s"(lds), "v"(off), "s"(r), "s"(soff), "s"(mask) : "memory");
    else
        asm volatile("s_mov_b32 m0, %0\n\ts_mov_b64 exec, %4\n\tbuffer_load_dword %1, %2, %3 offen lds\n\t"
                     "s_mov_b64 exec, -1" ::"s"(lds), "v"(off), "s"(r), "s"(soff), "s"(mask) : "memory");
}

// Waits until at most LEFT of the wave's loads are in flight, then meets the
// block's other waves.  LDS reads may still be in flight: the callers place
// the barrier where those read buffers that are refilled only after the next
// one.
template <int LEFT>
__device__ __forceinline__ void dma_wait() {
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"i"(LEFT) : "memory");
}

__device__ __forceinline__ uint32_t lds_addr(const void *p) {
    return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const char *)p;
}

__device__ __forceinline__ uint32_t pack_hi16(float lo_elem, float hi_elem) {
    return __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, hi_elem), __builtin_bit_cast(uint32_t, lo_elem),
                                 0x07060302u);
}

template <int J>
__device__ __forceinline__ float sbyte(uint32_t w) {
    return (float)(int8_t)(uint8_t)(w >> (8 * J));
}

__device__ __forceinline__ f16x2 as_h2(uint32_t u) { return __builtin_bit_cast(f16x2, u); }
__device__ __forceinline__ uint32_t as_u(f16x2 h) { return __builtin_bit_cast(uint32_t, h); }

// Dword I (weights 2 I, 2 I + 1) of eight INT8 weights (two words, bytes of
// k + {0, 2, 1, 3}, stored q + 128) as q - zp in bf16 (sign-extending byte
// conversions, upper halves packed) or f16 (0x6400 | u is 1024 + u; one
// packed add leaves q - zp, all exact).
template <bool F16, bool ZP, int I>
__device__ __forceinline__ uint32_t unpack8(u32x2 w, float zf) {
    const uint32_t u = w[I / 2];
    if constexpr (F16) {
        const _Float16 off = (_Float16)(ZP ? -1152.0f - zf : -1152.0f);   // integers: exact
        // one byte permutation: {u byte, 0x64, u byte, 0x64}
        const uint32_t m = __builtin_amdgcn_perm(0x64646464u, u, I % 2 ? 0x04030401u : 0x04020400u);
        return as_u(as_h2(m) + f16x2{off, off});
    } else {
        const uint32_t v = u ^ 0x80808080u;
        const float z = ZP ? zf : 0.0f;
        return pack_hi16(sbyte<I % 2>(v) - z, sbyte<2 + I % 2>(v) - z);
    }
}

// Dword I of eight INT4 weights (one word, nibble of k % 8 at bit {0, 16, 4,
// 20, 8, 24, 12, 28}, stored q + 8) as 16 (q - zp) in bf16, or q - zp in f16
// (nibbles left in place at bits 0 and 4: 1024 + u, and 1024 + 16 u taken
// through one fma by 1/16; exact).
// m0, m1: 0x000F000F and 0x00F000F0 held in registers, so that mask and
// merge are one v_and_or_b32.
template <bool F16, bool ZP, int I>
__device__ __forceinline__ uint32_t unpack4(uint32_t w, float zf, uint32_t m0, uint32_t m1) {
    if constexpr (F16) {
        const uint32_t v = I / 2 ? w >> 8 : w;
        if constexpr (I % 2 == 0) {
            const _Float16 c = (_Float16)(ZP ? -1032.0f - zf : -1032.0f);
            return as_u(as_h2((v & m0) | 0x64006400u) + f16x2{c, c});
        } else {
            const _Float16 c = (_Float16)(ZP ? -72.0f - zf : -72.0f);
            return as_u(__builtin_elementwise_fma(as_h2((v & m1) | 0x64006400u),
                                                  f16x2{(_Float16)0.0625f, (_Float16)0.0625f}, f16x2{c, c}));
        }
    } else {
        const float z = ZP ? 16.0f * zf : 0.0f;
        const uint32_t v = w ^ 0x88888888u;
        const uint32_t b = I % 2 ? v & 0xF0F0F0F0u : (v << 4) & 0xF0F0F0F0u;   // bytes: k + {2, 6, 3, 7}, {0, 4, 1, 5}
        return pack_hi16(sbyte<I / 2>(b) - z, sbyte<2 + I / 2>(b) - z);
    }
}

// The low f16 piece of a weight w' whose high piece was rounded toward zero
// (r = w' - hi, exact; NaN for a non-finite w', which hi holds): r, but at
// least 2^-24 in magnitude and with w's sign unless w' = 0, so that an
// infinite x meets two pieces of one sign (inf * w' as one product: +-inf,
// or NaN for w' = 0) and never inf * 0 = NaN from an empty low piece.  The
// scale table keeps every nonzero |w'| at 2^-24 or more.
__device__ __forceinline__ float lo_piece(float w, float r) {
    return w == 0.0f ? 0.0f : __builtin_copysignf(__builtin_fmaxf(__builtin_fabsf(r), 0x1p-24f), w);
}

// Dword I of eight runtime-layout INT4 weights against their scales (times
// 2^(8 - e_b)): w' = 16 q * s' as two f16 pieces, hi rounded toward zero.
template <int I>
__device__ __forceinline__ void unpack4n(uint32_t w0, float sa, float sb, uint32_t &ph, uint32_t &pl) {
    const uint32_t w = w0 ^ 0x88888888u;
    const uint32_t v = I % 2 ? w & 0xF0F0F0F0u : (w << 4) & 0xF0F0F0F0u;
    const float a = sbyte<I / 2>(v) * sa, b = sbyte<2 + I / 2>(v) * sb;
    const f16x2 h = __builtin_bit_cast(f16x2, __builtin_amdgcn_cvt_pkrtz(a, b));
    const f32x2 hb = __builtin_convertvector(h, f32x2);
    ph = as_u(h);
    pl = as_u(__builtin_convertvector(f32x2{lo_piece(a, a - hb[0]), lo_piece(b, b - hb[1])}, f16x2));
}

template <bool F16>
__device__ __forceinline__ f32x4 mfma(u32x4 a, u32x4 b, f32x4 c) {
    if constexpr (F16)
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0,
                                                      0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                       0, 0, 0);
}

// LDS bytes of one step: x, packed weights, scales, zero points.
constexpr int x_bytes(int xp, int tm) { return xp * tm * 2048; }
constexpr int w_bytes(int kind, int tn) { return kind == W8 ? tn * 8192 : tn * 4096; }
constexpr int s_bytes(int kind, int tn) { return kind == W8 ? 0 : kind == W4K ? tn * 1024 : tn * 2048; }
constexpr int z_bytes(int kind, int tn) { return kind == W4K ? tn * 256 : 0; }
constexpr int step_bytes(int kind, int xp, int tm, int tn) {
    return x_bytes(xp, tm) + w_bytes(kind, tn) + s_bytes(kind, tn) + z_bytes(kind, tn);
}
// Step buffers of a tile: four where they fit the 160 KiB (three left INT8
// 128 x 128 tiles waiting for memory: 0.51 -> 0.43 us a step on 160 CUs; more
// than four changed nothing), else three; the kernel needs three.
constexpr int step_bufs(int kind, int xp, int tm, int tn) {
    return 4 * step_bytes(kind, xp, tm, tn) <= 160 * 1024 ? 4 : 160 * 1024 / step_bytes(kind, xp, tm, tn);
}
// (runtime-layout tiles over 16 x 16 MFMA tiles per wave spill registers; its
// 64 x 256 tile of one piece is never the cheapest: 0 of 34000 drawn products)
constexpr bool tile_fits(int kind, int xp, int tm, int tn) {
    if (xp == 3 && (kind == W4N || tm != 4)) return false;   // few rows of x only
    if (kind == W4N && (tm * tn > 16 || (xp == 1 && tm == 4 && tn == 2))) return false;
    return step_bufs(kind, xp, tm, tn) >= 3;
}

template <int KIND, int XP, int TM, int TN>
struct Lds {
    static constexpr int x = x_bytes(XP, TM), w = w_bytes(KIND, TN), s = s_bytes(KIND, TN), z = z_bytes(KIND, TN);
    static constexpr int step = step_bytes(KIND, XP, TM, TN);
    static constexpr int bufs = step_bufs(KIND, XP, TM, TN);
};

// Tile of linear index t: rows of tiles along N (n_fast) or columns along M.
struct Tile {
    int tm, tn;
};
__device__ __forceinline__ Tile tile_of(const Args &p, int t) {
    const int d = p.n_fast ? p.tiles_n : p.tiles_m, q = t / d, r = t % d;
    return p.n_fast ? Tile{q, r} : Tile{r, q};
}

template <int KIND, int XP, bool ZP, int TM, int TN>
__global__ __launch_bounds__(64 * kWaves) void gemm(const Args p) {
    using L = Lds<KIND, XP, TM, TN>;
    constexpr bool F16 = XP == 2 || KIND == W4N;
    constexpr int BM = 16 * TM, BN = 128 * TN, NB = L::bufs;
    constexpr int NX = XP * TM * 2 / kWaves;                       // x loads per wave and step
    constexpr int NW = KIND == W8 ? TN : 1;
    constexpr int NLOADS = NX + NW + (KIND != W8 ? 1 : 0) + (KIND == W4K && ZP ? 1 : 0);
    static_assert(TM * 2 % kWaves == 0, "a piece's x loads divide over the waves");

    __shared__ __attribute__((aligned(1024))) char sm[NB * L::step];

    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r16 = lane & 15, kb = lane >> 4;

    // ---- which tile and K range
    Tile tile;
    int kpart = 0, tr = -1, steps = p.split_steps;
    {
        const int bid = blockIdx.x;
        if (p.seq) {
            tile = Tile{p.seq_tm + bid % p.seq_tms, bid / p.seq_tms};
            const int at = p.n_fast ? tile.tm * p.tiles_n + tile.tn : tile.tn * p.tiles_m + tile.tm;
            if ((p.tail_parts > 0 && at >= p.tail_first) != (p.seq_tail != 0)) return;
            kpart = p.seq_part;
            steps = p.seq_steps;
        } else if (bid < p.main_blocks) {
            // consecutive blocks go to the eight XCDs in turn: give each XCD a
            // contiguous range of items, so its L2 holds the rows they share
            const int q = p.main_blocks / 8, rem = p.main_blocks % 8, xcd = bid % 8;
            const int item = xcd * q + min(xcd, rem) + bid / 8;
            const int tiles = p.tail_parts ? p.tail_first : p.tiles_m * p.tiles_n;
            kpart = item / tiles;
            tile = tile_of(p, item % tiles);
        } else {
            const int q = bid - p.main_blocks;
            tr = q / p.tail_parts;
            kpart = q % p.tail_parts;
            steps = p.tail_steps;
            tile = tile_of(p, p.tail_first + tr);
        }
    }
    const int m0 = p.row_base + (tile.tm - p.seq_tm) * BM, n0 = tile.tn * BN, wn0 = n0 + wave * 16 * TN;
    const int x_row = m0 - p.row_base;   // row of the pieces
    const int t_begin = kpart * steps, t_end = min(p.nsteps, t_begin + steps);

    // ---- values the epilogue needs, loaded before the step loads begin (the
    // loop's waits count every load of the wave)
    f32x4 osc[TN];          // W8: row scales
    float zf8[TN];          // W8 zero points of the lane's weight rows
#pragma unroll
    for (int b = 0; b < TN; ++b) {
        osc[b] = f32x4{1.f, 1.f, 1.f, 1.f};
        zf8[b] = 0.0f;
        if constexpr (KIND == W8) {
            osc[b] = *(const f32x4 *)(p.scales + min(wn0 + b * 16 + 4 * kb, p.Np - 4));
            if constexpr (ZP) zf8[b] = (float)p.zp[min(wn0 + b * 16 + r16, p.Np - 1)];
        }
    }

    // ---- step loads: each lane's buffer offsets, the same for every step
    // (the step's own offset is the scalar one), and what the step that
    // reaches past the rows' end adds to them
    const int xlast = p.xk / kBK * kBK, wlast = (KIND == W4K ? p.chunks / 2 : p.kp / kBK);
    // x load i of this wave: LDS rows 8 j .. 8 j + 7 of the pieces' stacked
    // rows, j = i * kWaves + wave; lane -> row lane / 8, segment lane % 8
    uint32_t xoff[NX], xfar[NX];   // xfar: set in the lanes past an x row's end in its last step
#pragma unroll
    for (int i = 0; i < NX; ++i) {
        const int row = (i * kWaves + wave) * 8 + (lane >> 3), seg = (lane & 7) ^ (row & 7);
        xoff[i] = (uint32_t)((row % BM) * (int)(p.ldx * 2) + seg * 16);
        xfar[i] = xlast + 8 * seg < p.xk ? 0 : kFar;
    }
    uint32_t woff[NW], soff = 0, sdelta = 0, sfar = 0;
    constexpr uint64_t kScaleLanes = KIND == W4K ? (1ull << (8 * TN)) - 1 : (1ull << (16 * TN)) - 1;
    int64_t q0 = 0;   // W4K: byte of the wave's first scale
    if constexpr (KIND == W8) {
#pragma unroll
        for (int i = 0; i < NW; ++i)   // 16 rows x 64 bytes, 16-byte segment index ^ (row / 4) % 4
            woff[i] = (uint32_t)((16 * i + (lane >> 2)) * (int)p.row_bytes + ((lane & 3) ^ ((lane >> 4) & 3)) * 16);
    } else {
        // 16 TN rows x 32 bytes, segment index ^ (row / 8) % 2
        woff[0] = (uint32_t)((lane >> 1) * (int)p.row_bytes + ((lane & 1) ^ ((lane >> 4) & 1)) * 16);
        if constexpr (KIND == W4K) {
            // [4 TN quads][2 chunks] x 16 bytes (four rows' scales): the
            // step's second chunk lies in its first one's group or the next;
            // a chunk past the row takes scale 0
            q0 = (int64_t)(wn0 >> 2) * p.G * 16;
            soff = (uint32_t)((lane >> 1) * p.G * 16);
            sdelta = (lane & 1) * 16;
            sfar = lane & 1 ? kFar : 0;
        } else {
            // [TN tiles][64 k] fp32: tile b's N-block
            const int nb = min(wn0 + 16 * (lane >> 4), p.Np - 1) / p.rpn;
            soff = (uint32_t)(nb * p.kp * 4 + (lane & 15) * 16);
            sfar = wlast * kBK + (lane & 15) * 4 < p.kp ? 0 : kFar;
        }
    }
    const uint32_t sm0 = lds_addr(sm);
    const int xbytes = (int)((int64_t)min(BM, p.row_end - m0) * p.ldx * 2);
    i32x4 xrs[XP], wrs, srs{}, zrs{};
#pragma unroll
    for (int q = 0; q < XP; ++q) xrs[q] = make_rsrc(p.x + q * p.piece_stride + (int64_t)x_row * p.ldx, xbytes);
    wrs = make_rsrc(p.data + (int64_t)wn0 * p.row_bytes, (int)((int64_t)max(0, min(16 * TN, p.Np - wn0)) * p.row_bytes));
    if constexpr (KIND != W8)
        srs = make_rsrc((const char *)p.scales + q0, (int)max((int64_t)0, min(p.scale_bytes - q0, (int64_t)kDead - 1)));
    if constexpr (KIND == W4K && ZP)
        zrs = make_rsrc(p.zp + q0 / 4, (int)max((int64_t)0, min((p.scale_bytes - q0) / 4, (int64_t)kDead - 1)));
    // What the loads of step t share.  Steps past the block's range read
    // nothing (zeros into a buffer that is not used again).
    struct Step {
        uint32_t lds, xo, wo, so, zo;
        bool x_part, s_part, s_next;
    };
    auto step_of = [&](int t, int buf) {
        Step st;
        const bool live = t < t_end;
        st.lds = sm0 + buf * L::step;
        st.xo = live ? (uint32_t)t * (kBK * 2) : kDead;
        st.wo = live ? (uint32_t)t * (KIND == W8 ? kBK : kBK / 2) : kDead;
        st.x_part = (t + 1) * kBK > p.xk;
        st.s_part = st.s_next = false;
        st.so = st.zo = 0;
        if constexpr (KIND == W4K) {
            // group of chunk c: c / cpg (c cpg_magic / 2^32, exact for c cpg < 2^32)
            const uint32_t g0 = (uint32_t)((uint32_t)(2 * t) * p.cpg_magic >> 32);
            const uint32_t g1 = (uint32_t)((uint32_t)(2 * t + 1) * p.cpg_magic >> 32);
            st.so = live ? g0 * 16 : kDead;
            st.zo = live ? g0 * 4 : kDead;
            st.s_part = 2 * t + 1 >= p.chunks;
            st.s_next = g1 != g0;
        } else if constexpr (KIND == W4N) {
            st.so = live ? (uint32_t)t * (kBK * 4) : kDead;
            st.s_part = t >= wlast;
        }
        return st;
    };
    auto load_one = [&](const Step &st, int i) {   // load i of this wave
        if (i < NX) {
            const int j = i * kWaves + wave;
            // padded rows (pieces) end with a whole step
            const uint32_t off = F16 || XP > 1 ? xoff[i] : xoff[i] | (st.x_part ? xfar[i] : 0u);
            dma16(__builtin_amdgcn_readfirstlane(st.lds + j * 1024), xrs[i / (TM / 4)], off, st.xo);   // 2 TM loads a piece
        } else if (i < NX + NW) {
            const uint32_t wb = __builtin_amdgcn_readfirstlane(st.lds + L::x + wave * (L::w / kWaves) + (i - NX) * 1024);
            if constexpr (KIND == W8 || TN == 2) dma16(wb, wrs, woff[i - NX], st.wo);
            else dma_lanes<16>(wb, wrs, woff[0], st.wo, 0xFFFFFFFFull);
        } else if (i == NX + NW) {
            const uint32_t sb = __builtin_amdgcn_readfirstlane(st.lds + L::x + L::w + wave * (L::s / kWaves));
            const uint32_t off = (soff + (st.s_next ? sdelta : 0u)) | (st.s_part ? sfar : 0u);
            dma_lanes<16>(sb, srs, off, st.so, kScaleLanes);
        } else {
            const uint32_t zb = __builtin_amdgcn_readfirstlane(st.lds + L::x + L::w + L::s + wave * (L::z / kWaves));
            const uint32_t off = ((soff + (st.s_next ? sdelta : 0u)) / 4) | (st.s_part ? sfar : 0u);
            dma_lanes<4>(zb, zrs, off, st.zo, kScaleLanes);
        }
    };

    // Products with a low piece (2^-11 of the others) sum apart: added to the
    // same accumulator they would round it twice as often (INT8 fp32 x at K =
    // 2048: error against float64 3.8e-7 in one accumulator, 2.5e-7 in two).
    // W4K's pieces meet in the group's partial product, which is small.
    constexpr bool kLow = KIND == W4N || (KIND == W8 && XP > 1);
    f32x4 acc[TM][TN], low[kLow ? TM : 1][TN];
#pragma unroll
    for (int a = 0; a < TM; ++a)
#pragma unroll
        for (int b = 0; b < TN; ++b) {
            acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
            if constexpr (kLow) low[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
        }

    // lane's byte offset of x fragment (row r16, segment 4 ks + kb) in a tile
    const int xfr = r16 * 128 + ((kb ^ (r16 & 7)) * 16);
    // and of its eight packed weights of slice 0 in a column tile: 8 bytes of
    // row r16's 64 (W8) or 4 of its 32, segments permuted so that the 16 rows
    // cover all banks (in row order the reads of a tile cost 56 conflict
    // cycles each, 900 a step at TN = 2)
    const int wfr = KIND == W8 ? r16 * 64 + ((kb >> 1) ^ (r16 >> 2)) * 16 + (kb & 1) * 8
                               : r16 * 32 + (r16 >> 3) * 16 + kb * 4;
    // ---- the K loop, pipelined across steps.  Step t's buffer is t % NB.  The
    // step's 2 TM x fragments (slice ks = f / TM, rows 16 (f % TM)) are read
    // kAhead slots before their MFMAs, the last slots reading the next step's
    // first ones, and the next step's weights are read and its first slice
    // unpacked in the second half, so that no step starts by waiting for the
    // LDS (0.4 us a step when it did).  The one barrier stands in the middle of
    // the step, where every operand of the next slots is already in registers:
    // it says that step t + 1 has landed (each wave has waited for its own
    // loads) and that every wave is done with step t - 1, whose buffer the
    // loads of step t + NB - 1, spread over the second half, then fill.  The
    // fences between slots keep the compiler from moving reads to their uses.
    constexpr int NF = 2 * TM;
    constexpr int kRing = TN == 1 && XP == 1 && TM >= 8 ? 8 : 4, kAhead = kRing == 8 ? 6 : 3;
    static_assert(kAhead <= TM, "the next step is read behind the barrier only");
    static_assert(NF % kRing == 0, "fragment f of every step has the same ring place");
    uint32_t nib0 = 0x000F000Fu, nib1 = 0x00F000F0u;
    asm volatile("" : "+v"(nib0), "+v"(nib1));
    u32x4 xf[kRing][XP];
    u32x2 raw8[2][TN];
    uint32_t raw4[2][TN];
    f32x4 sc[2][TN], sc_next[TN], sn[2][TN][2];
    float zf[2][TN];
    u32x4 wf[2][TN], wl[2][TN];
    f32x4 part[2][TN];
    auto load_x = [&](uint32_t bo, int f) {
        const char *xb = sm + bo + (xfr ^ ((f / TM) * 64)) + (f % TM) * 2048;
#pragma unroll
        for (int q = 0; q < XP; ++q) xf[f % kRing][q] = *(const u32x4 *)(xb + q * TM * 2048);
    };
    // packed weights, zero points and scales of slice ks (W4K: its scales into sd)
    auto load_w = [&](uint32_t bo, int ks, f32x4 *sd) {
        const char *wb = sm + bo + L::x + wave * (L::w / kWaves);
        const char *sb = sm + bo + L::x + L::w + wave * (L::s / kWaves);
        const char *zb = sm + bo + L::x + L::w + L::s + wave * (L::z / kWaves);
#pragma unroll
        for (int b = 0; b < TN; ++b) {
            if constexpr (KIND == W8) {
                raw8[ks][b] = *(const u32x2 *)(wb + b * 1024 + (wfr ^ (ks * 32)));
            } else {
                raw4[ks][b] = *(const uint32_t *)(wb + b * 512 + (wfr ^ (ks * 16)));
                if constexpr (KIND == W4K) {
                    if constexpr (ZP) zf[ks][b] = (float)*(const int8_t *)(zb + b * 32 + ((r16 >> 2) * 2 + ks) * 4 + (r16 & 3));
                    else zf[ks][b] = 0.0f;
                    sd[b] = *(const f32x4 *)(sb + b * 128 + (kb * 2 + ks) * 16);
                } else {
                    const char *sp = sb + b * 256 + (ks * 32 + kb * 8) * 4;
                    sn[ks][b][0] = *(const f32x4 *)sp;
                    sn[ks][b][1] = *(const f32x4 *)(sp + 16);
                }
            }
        }
    };
    // dword i of the operand of slice ks, column tile b
    auto unpack = [&](int ks, int b, auto ic) {
        constexpr int i = decltype(ic)::value;
        if constexpr (KIND == W8) {
            wf[ks][b][i] = unpack8<F16, ZP, i>(raw8[ks][b], zf8[b]);
        } else if constexpr (KIND == W4K) {
            wf[ks][b][i] = unpack4<F16, ZP, i>(raw4[ks][b], zf[ks][b], nib0, nib1);
        } else {
            uint32_t h, l;
            unpack4n<i>(raw4[ks][b], sn[ks][b][i / 2][2 * (i % 2)], sn[ks][b][i / 2][2 * (i % 2) + 1], h, l);
            wf[ks][b][i] = h;
            wl[ks][b][i] = l;
        }
    };
    auto unpack_part = [&](int ks, int part) {   // parts 0 .. 4 TN - 1
        const int b = part / 4;
        switch (part % 4) {
        case 0: unpack(ks, b, std::integral_constant<int, 0>{}); break;
        case 1: unpack(ks, b, std::integral_constant<int, 1>{}); break;
        case 2: unpack(ks, b, std::integral_constant<int, 2>{}); break;
        default: unpack(ks, b, std::integral_constant<int, 3>{}); break;
        }
    };
    auto add_part = [&](int f, int b, int e0, int e1) {
#pragma unroll
        for (int e = e0; e < e1; ++e)
            acc[f % TM][b][e] = __builtin_fmaf(part[f % 2][b][e], sc[f / TM][b][e], acc[f % TM][b][e]);
    };
    static_assert(NB >= 3, "a step's loads are issued one step before the barrier that waits for them");

    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
    for (int j = 0; j < NB - 1; ++j) {
        const Step st = step_of(t_begin + j, j);
#pragma unroll
        for (int i = 0; i < NLOADS; ++i) load_one(st, i);
    }
    dma_wait<(NB - 2) * NLOADS>();
    load_w(0, 0, sc[0]);
    load_w(0, 1, sc[1]);
#pragma unroll
    for (int f = 0; f < kAhead; ++f) load_x(0, f);
#pragma unroll
    for (int i = 0; i < 4 * TN; ++i) unpack_part(0, i);
    int buf = 0;
    for (int t = t_begin; t < t_end; ++t) {
        const int next = buf + 1 == NB ? 0 : buf + 1, last = buf == 0 ? NB - 1 : buf - 1;
        const uint32_t bo = (uint32_t)(buf * L::step), no = (uint32_t)(next * L::step);
        const Step st = step_of(t + NB - 1, last);
#pragma unroll
        for (int f = 0; f < NF; ++f) {
            __builtin_amdgcn_sched_barrier(0);
            const int ks = f / TM, a = f % TM;
            if (f == TM) {
                dma_wait<(NB - 3) * NLOADS>();
                __builtin_amdgcn_sched_barrier(0);
            }
            if (f >= TM) {
#pragma unroll
                for (int i = 0; i < NLOADS; ++i)
                    if (TM + i * TM / NLOADS == f) load_one(st, i);
            }
            if (f + kAhead < NF) load_x(bo, f + kAhead);
            else load_x(no, f + kAhead - NF);
            // per column tile: its MFMAs, each followed by VALU work that does
            // not wait for them (the waves of a SIMD run in step, and the
            // matrix core idles through a run of VALU instructions): W4K's
            // scaled sums of the previous slot, and pieces of the unpacking of
            // the second slice and then (behind the barrier) of the next
            // step's first
#pragma unroll
            for (int b = 0; b < TN; ++b) {
                if (b) __builtin_amdgcn_sched_barrier(0);
                const bool add = KIND == W4K && f > 0;
#pragma unroll
                for (int q = 0; q < XP; ++q) {
                    const u32x4 xv = xf[f % kRing][q];
                    if constexpr (KIND == W4K) {
                        part[f % 2][b] = mfma<F16>(wf[ks][b], xv, q == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : part[f % 2][b]);
                        __builtin_amdgcn_sched_barrier(0);
                        if (add) add_part(f - 1, b, q * 4 / XP, (q + 1) * 4 / XP);
                    } else {
                        if (q == 0) acc[a][b] = mfma<F16>(wf[ks][b], xv, acc[a][b]);
                        else low[kLow ? a : 0][b] = mfma<F16>(wf[ks][b], xv, low[kLow ? a : 0][b]);
                        if constexpr (KIND == W4N) low[a][b] = mfma<F16>(wl[ks][b], xv, low[a][b]);
                    }
                }
#pragma unroll
                for (int i = 0; i < 4 * TN; ++i) {
                    // part i in slot-and-tile unit i * units / (4 TN)
                    if (i * (TM * TN) / (4 * TN) == f * TN + b) unpack_part(1, i);
                    if ((TM + 2) * TN + i * ((TM - 2) * TN) / (4 * TN) == f * TN + b) unpack_part(0, i);
                }
            }
            if (f == TM) {
                load_w(no, 0, sc[0]);   // sc[0] was last used above
                load_w(no, 1, sc_next);
            }
        }
        if constexpr (KIND == W4K) {
#pragma unroll
            for (int b = 0; b < TN; ++b) {
                add_part(NF - 1, b, 0, 4);
                sc[1][b] = sc_next[b];
            }
        }
        buf = next;
    }
    // the loads past the range have still to land in this block's LDS
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

    // ---- epilogue: lane holds outputs 4 kb + e of x row r16 of each tile
    float *out = p.y + (p.seq ? 0 : (int64_t)kpart * p.split_stride);
#pragma unroll
    for (int a = 0; a < TM; ++a) {
        const int m = m0 + a * 16 + r16;
        int re = 0;
        if constexpr (F16) re = p.row_exp[min(m, p.row_end - 1) - p.row_base];
#pragma unroll
        for (int b = 0; b < TN; ++b) {
            const int n = wn0 + b * 16 + 4 * kb;
            f32x4 v = acc[a][b];
            if constexpr (kLow) {
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] += low[a][b][e];
            }
            if constexpr (KIND == W4N) {
                const int eb = p.nb_exp[min(n, p.Np - 1) / p.rpn] - 27;
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = __builtin_ldexpf(v[e], eb + re);
            } else if constexpr (F16) {
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = __builtin_ldexpf(v[e], re - 15) * osc[b][e];
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] *= KIND == W8 ? osc[b][e] : 0.0625f;
            }
            if (tr >= 0) {
                // a tail part: the whole tile into its slot
                *(f32x4 *)(p.tail_part + ((int64_t)(kpart * p.tail_n + tr) * BM + a * 16 + r16) * BN + (n - n0)) = v;
                continue;
            }
            if (m >= p.row_end || n >= p.N) continue;
            float *o = out + (int64_t)m * p.ldy + n;
            if (p.add) {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (n + e < p.N) v[e] = o[e] + v[e];
            }
            if (p.vec && n + 3 < p.N) {
                *(f32x4 *)o = v;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (n + e < p.N) o[e] = v[e];
            }
        }
    }
}

template <int KIND, int XP, bool ZP, int TM, int TN>
hipError_t launch_tile(const Args &a, unsigned blocks, hipStream_t s) {
    if constexpr (tile_fits(KIND, XP, TM, TN)) {
        hipLaunchKernelGGL((gemm<KIND, XP, ZP, TM, TN>), dim3(blocks), dim3(64 * kWaves), 0, s, a);
        return hipGetLastError();
    } else {
        return hipErrorInvalidValue;   // three steps do not fit the LDS
    }
}

template <int KIND, int XP, bool ZP>
hipError_t launch(const Args &a, int tm, int tn, unsigned blocks, hipStream_t s) {
#define TBH_GEMM(TM)                                                       \
    case TM: return tn == 1 ? launch_tile<KIND, XP, ZP, TM, 1>(a, blocks, s) \
                            : launch_tile<KIND, XP, ZP, TM, 2>(a, blocks, s);
    if constexpr (XP == 3) {
        if (tm != 4) return hipErrorInvalidValue;
        return tn == 1 ? launch_tile<KIND, XP, ZP, 4, 1>(a, blocks, s) : launch_tile<KIND, XP, ZP, 4, 2>(a, blocks, s);
    }
    switch (tm) {
        TBH_GEMM(4)
        TBH_GEMM(8)
        TBH_GEMM(12)
        TBH_GEMM(16)
    default: return hipErrorInvalidValue;
    }
#undef TBH_GEMM
}

hipError_t launch_w8(const Args &a, int xp, bool zp, int tm, int tn, unsigned blocks, hipStream_t s);
hipError_t launch_w4k(const Args &a, int xp, bool zp, int tm, int tn, unsigned blocks, hipStream_t s);
hipError_t launch_w4n(const Args &a, int xp, bool zp, int tm, int tn, unsigned blocks, hipStream_t s);

}  // namespace gemm
}  // namespace tbh
