// tbh_gemm.hip -- host side of the prefill GEMM (tbh_gemm.h): the pass that
// turns fp32 x (or bf16 x of runtime-layout weights) into 16-bit pieces, the
// choice of tile and K split, and the sums of split launches.
#include "tbh_gemm.h"

namespace tbh {
namespace {

using namespace gemm;

// One x row per block of 256 threads: e = the least e with |x| < 2^e for
// every finite element of the row (0 for a row of zeros, -126 when the
// largest is subnormal), then the row times 2^(15 - e) as f16: hi = f16(x'),
// and for fp32 x lo = f16(x' - hi) in the second piece (the difference exact
// in fp32; 0 for a non-finite x', which hi holds).  bf16 x is exact in hi.
// Columns [K, ldp) of the pieces are zero.  R > 0: the row's 16-byte segments
// stay in registers between the two passes (R per thread); R = 0 reads the
// row twice.  Rows 16-byte aligned, K a multiple of the segment.
template <bool F32, int R>
__global__ __launch_bounds__(256) void x_pieces(const void *__restrict__ xv, int64_t ldx, int32_t K,
                                                int32_t *__restrict__ e_out, uint16_t *__restrict__ out,
                                                int64_t ldp, int64_t piece_stride) {
    constexpr int EPS = F32 ? 4 : 8;   // elements per 16-byte segment
    __shared__ uint32_t wmax[4];
    const int64_t r = blockIdx.x;
    const int tid = threadIdx.x;
    const u32x4 *src = (const u32x4 *)((const char *)xv + r * ldx * (F32 ? 4 : 2));
    const int nseg = K / EPS, npad = (int)(ldp / EPS);
    u32x4 v[R > 0 ? R : 1];
    uint32_t mx = 0;   // largest finite |x| as bits (magnitudes order as their bits)
    auto scan = [&](u32x4 s) {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            if constexpr (F32) {
                const uint32_t a = s[c] & 0x7FFFFFFFu;
                mx = max(mx, a < 0x7F800000u ? a : 0u);
            } else {
                const uint32_t lo = s[c] & 0x7FFFu, hi = (s[c] >> 16) & 0x7FFFu;
                mx = max(mx, max(lo < 0x7F80u ? lo : 0u, hi < 0x7F80u ? hi : 0u));
            }
        }
    };
    if constexpr (R > 0) {
#pragma unroll
        for (int i = 0; i < R; ++i) {
            const int j = tid + 256 * i;
            v[i] = j < nseg ? src[j] : u32x4{0, 0, 0, 0};
        }
#pragma unroll
        for (int i = 0; i < R; ++i) scan(v[i]);
    } else {
#pragma unroll 4
        for (int j = tid; j < nseg; j += 256) scan(src[j]);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) mx = max(mx, (uint32_t)__shfl_xor((int)mx, o));
    if ((tid & 63) == 0) wmax[tid >> 6] = mx;
    __syncthreads();
    mx = max(max(wmax[0], wmax[1]), max(wmax[2], wmax[3]));
    const int E = (int)(mx >> (F32 ? 23 : 7));   // exponent field
    const int e = mx == 0 ? 0 : (E == 0 ? -126 : E - 126);
    if (tid == 0) e_out[r] = e;
    const int sh = 15 - e;
    uint16_t *dst = out + r * ldp;
    auto emit = [&](int j, u32x4 s) {
        if constexpr (F32) {
            uint32_t hi[2], lo[2];
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const uint32_t ua = s[2 * q], ub = s[2 * q + 1];
                const float a = __builtin_ldexpf(__builtin_bit_cast(float, ua), sh);
                const float b = __builtin_ldexpf(__builtin_bit_cast(float, ub), sh);
                const f16x2 h = __builtin_convertvector(f32x2{a, b}, f16x2);
                const f32x2 hb = __builtin_convertvector(h, f32x2);
                const float ra = a - hb[0], rb = b - hb[1];
                hi[q] = as_u(h);
                lo[q] = as_u(__builtin_convertvector(
                    f32x2{__builtin_isnan(ra) ? 0.0f : ra, __builtin_isnan(rb) ? 0.0f : rb}, f16x2));
            }
            *(u32x2 *)(dst + 4 * j) = u32x2{hi[0], hi[1]};
            *(u32x2 *)(dst + piece_stride + 4 * j) = u32x2{lo[0], lo[1]};
        } else {
            u32x4 o;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint32_t w = s[q];
                const float a = __builtin_bit_cast(float, w << 16), b = __builtin_bit_cast(float, w & 0xFFFF0000u);
                o[q] = as_u(__builtin_convertvector(f32x2{__builtin_ldexpf(a, sh), __builtin_ldexpf(b, sh)}, f16x2));
            }
            *(u32x4 *)(dst + 8 * j) = o;
        }
    };
    if constexpr (R > 0) {
#pragma unroll
        for (int i = 0; i < R; ++i) {
            const int j = tid + 256 * i;
            if (j < npad) emit(j, v[i]);
        }
    } else {
        for (int j = tid; j < npad; j += 256) emit(j, j < nseg ? src[j] : u32x4{0, 0, 0, 0});
    }
}

// fp32 x as three bf16 pieces, exactly: p0 the upper 16 bits of x, p1 those of
// the remainder, p2 the rest (at most 8 significant bits); non-finite x stays
// in p0.  One thread per four elements of a row of ldp (zeros past K).
__global__ __launch_bounds__(256) void x_split3(const float *__restrict__ x, int64_t ldx, int32_t K, int64_t rows,
                                                uint16_t *__restrict__ out, int64_t ldp, int64_t piece_stride) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x, q4 = ldp / 4;
    if (i >= rows * q4) return;
    const int64_t r = i / q4, k = 4 * (i % q4);
    u32x4 v = u32x4{0, 0, 0, 0};
    if (k < K) v = *(const u32x4 *)(x + r * ldx + k);
    uint32_t p[3][4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const uint32_t b = v[c];
        const float f = __builtin_bit_cast(float, b), p0 = __builtin_bit_cast(float, b & 0xFFFF0000u);
        const float r1 = (b & 0x7F800000u) != 0x7F800000u ? f - p0 : 0.0f;
        const uint32_t b1 = __builtin_bit_cast(uint32_t, r1) & 0xFFFF0000u;
        p[0][c] = b;
        p[1][c] = b1;
        p[2][c] = __builtin_bit_cast(uint32_t, r1 - __builtin_bit_cast(float, b1));
    }
#pragma unroll
    for (int j = 0; j < 3; ++j)
        *(u32x2 *)(out + j * piece_stride + r * ldp + k) =
            u32x2{__builtin_amdgcn_perm(p[j][1], p[j][0], 0x07060302u), __builtin_amdgcn_perm(p[j][3], p[j][2], 0x07060302u)};
}

template <bool F32>
hipError_t launch_pieces(const void *x, int64_t ldx, int32_t K, int64_t rows, int32_t *e, uint16_t *out, int64_t ldp,
                         int64_t piece_stride, hipStream_t s) {
    const int64_t per = (ldp / (F32 ? 4 : 8) + 255) / 256;   // segments per thread
    const dim3 grid((unsigned)rows), block(256);
    if (per <= 2) hipLaunchKernelGGL((x_pieces<F32, 2>), grid, block, 0, s, x, ldx, K, e, out, ldp, piece_stride);
    else if (per <= 6) hipLaunchKernelGGL((x_pieces<F32, 6>), grid, block, 0, s, x, ldx, K, e, out, ldp, piece_stride);
    else if (per <= 12) hipLaunchKernelGGL((x_pieces<F32, 12>), grid, block, 0, s, x, ldx, K, e, out, ldp, piece_stride);
    else hipLaunchKernelGGL((x_pieces<F32, 0>), grid, block, 0, s, x, ldx, K, e, out, ldp, piece_stride);
    return hipGetLastError();
}

// The pieces of `rows` rows: xp = 3 three exact bf16 pieces, else f16 ones
// (two of fp32 x, one of bf16 x) and the rows' exponents.
hipError_t launch_split_x(const void *x, bool f32, int xp, int64_t ldx, int32_t K, int64_t rows, int32_t *e, uint16_t *out,
                          int64_t ldp, int64_t piece_stride, hipStream_t s) {
    if (xp == 3) {
        const int64_t n = rows * (ldp / 4);
        hipLaunchKernelGGL(x_split3, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, (const float *)x, ldx, K, rows,
                           out, ldp, piece_stride);
        return hipGetLastError();
    }
    return f32 ? launch_pieces<true>(x, ldx, K, rows, e, out, ldp, piece_stride, s)
               : launch_pieces<false>(x, ldx, K, rows, e, out, ldp, piece_stride, s);
}

// The tail's sums: element e of tail tile r (four at a time) = tail_part[0]
// [r][e] + tail_part[1][r][e] + ..., in part order, written where the tile
// lies inside the output.
__global__ __launch_bounds__(256) void tail_sum(const Args p, int bm, int bn) {
    const int64_t q = (int64_t)bm * bn / 4, total = (int64_t)p.tail_n * q;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
        const int r = (int)(i / q), e = 4 * (int)(i % q);
        const Tile tile = tile_of(p, p.tail_first + r);
        const int m = tile.tm * bm + e / bn, n = tile.tn * bn + e % bn;
        if (m >= p.M || n >= p.N) continue;
        f32x4 acc = *(const f32x4 *)(p.tail_part + (int64_t)r * bm * bn + e);
        for (int j = 1; j < p.tail_parts; ++j) {
            const f32x4 v = *(const f32x4 *)(p.tail_part + (int64_t)(j * p.tail_n + r) * bm * bn + e);
#pragma unroll
            for (int c = 0; c < 4; ++c) acc[c] += v[c];
        }
        float *o = p.y + (int64_t)m * p.ldy + n;
        if (p.vec && n + 3 < p.N) {
            *(f32x4 *)o = acc;
        } else {
            for (int c = 0; c < 4 && n + c < p.N; ++c) o[c] = acc[c];
        }
    }
}

constexpr int kMinSplitSteps = 4;   // K steps a split keeps at least

struct Plan {
    int tm = 8, tn = 1;
    int splits = 1, sps = 0;       // K splits and steps per split
    int tail_r = 0, tail_parts = 0, tail_steps = 0;
    double us = 0;
};

// Expected times, in us.  One K step of a block: s0 + s1 TM + s2 TN + s3 TM TN
// (barrier, x reads, weight unpacking, MFMA and scales), 1 + c times that when
// all CUs run a block (shared L2 and clock); the output's bytes, `out` times
// what they take at 4.6 TB/s; for a split the launch that sums, `sum`, and the
// partial tiles' bytes, written and read, at `part` times what they take.
// Least-squares fits over 534 shapes (rows 48 .. 2048, 1024x2048 ..
// 32000x2048) of every tile and 1 .. 16 splits, near-best plans weighted: the
// plan of least expected time takes 1.0-1.6 % more than the best one measured
// on average (a model from instruction counts, with 1.5 us a block and splits
// at their bytes: 5.6-9 %; INT8 bf16 x 5632x2048 at 333 rows 27.5 -> 19.3 us,
// INT4 4096x4096 at 128 rows 26.8 -> 19.3).
struct Cost {
    double s0, s1, s2, s3, c, out, sum, part;
};
constexpr Cost kCost[3][2] = {
    {{0.000, 0.011, 0.099, 0.021, 0.225, 1.30, 1.7, 1.6}, {0.055, 0.025, 0.091, 0.037, 0.308, 1.76, 1.9, 2.1}},   // W8
    {{0.133, 0.013, 0.078, 0.046, 0.000, 0.98, 0.3, 1.85}, {0.062, 0.040, 0.204, 0.042, 0.142, 1.50, 2.0, 2.0}},  // W4K
    {{0.000, 0.016, 0.496, 0.048, 0.004, 1.60, 2.8, 2.2}, {0.000, 0.041, 0.471, 0.067, 0.180, 2.00, 2.1, 2.3}},   // W4N
};

// The tile and K split of least expected time; a split is over all tiles, or
// over the R tiles of a last, part-filled round (the tail).  Tiles higher than
// the rows need are not looked at: the choice itself takes host time on every
// call.  Three pieces (xp = 3) cost 1.5 times two.
Plan choose(int kind, int xp, int64_t M, int64_t N, int nsteps, int64_t cus64, bool can_split) {
    const Cost &k = kCost[kind][xp > 1];
    const double more = xp == 3 ? 1.5 : 1.0;
    constexpr double kBytesPerUs = 4.6e6;
    Plan best;
    best.us = 1e30;
    const double out_us = 4.0 * (double)M * (double)N / kBytesPerUs;
    const int cus = (int)cus64;
    for (int tm : {4, 8, 12, 16}) {
        if (tm > 4 && 16 * (tm - 4) >= M) break;
        for (int tn : {1, 2}) {
            if (!tile_fits(kind, xp, tm, tn)) continue;
            const int64_t tiles64 = ((M + 16 * tm - 1) / (16 * tm)) * ((N + 128 * tn - 1) / (128 * tn));
            const double st = k.s0 + k.s1 * more * tm + k.s2 * tn + k.s3 * more * tm * tn;
            auto step = [&](int64_t blocks) { return st * (1.0 + k.c * std::min(1.0, (double)blocks / cus)); };
            auto rounds = [&](int64_t blocks) { return (double)((blocks + cus - 1) / cus); };
            Plan p;
            p.tm = tm;
            p.tn = tn;
            p.sps = nsteps;
            p.us = rounds(tiles64) * nsteps * step(tiles64) + k.out * out_us;
            if (p.us < best.us) best = p;
            if (!can_split || tiles64 > INT32_MAX / 64) continue;
            const int tiles = (int)tiles64;
            for (int sp = 2; sp <= 32 && tiles * sp <= 2 * cus; ++sp) {
                const int sps = (nsteps + sp - 1) / sp;
                if (sps < kMinSplitSteps) break;
                if ((nsteps + sps - 1) / sps != sp) continue;
                p.us = rounds(tiles * sp) * sps * step(tiles * sp) + (k.out + k.part * sp) * out_us + k.sum;
                p.splits = sp;
                p.sps = sps;
                if (p.us < best.us) best = p;
            }
            p.splits = 1;
            p.sps = nsteps;
            if (tiles <= cus || tiles % cus == 0) continue;
            const int R = tiles % cus;
            const double tile_us = 4.0 * 16 * tm * 128 * tn / kBytesPerUs;
            for (int P = 2; P <= 8; ++P) {
                const int ts = (nsteps + P - 1) / P;
                if (ts < kMinSplitSteps) break;
                if ((nsteps + ts - 1) / ts != P) continue;
                p.us = (double)(tiles / cus) * nsteps * step(cus) + rounds(R * P) * ts * step(R * P) +
                       k.out * out_us + k.sum + k.part * P * R * tile_us;
                p.tail_r = R;
                p.tail_parts = P;
                p.tail_steps = ts;
                if (p.us < best.us) best = p;
            }
        }
    }
    return best;
}

}  // namespace

// Whether the GEMM takes this weight: the bytes a tile reads of x, weights or
// scales stay under 2^30 (buffer offsets), and runtime-layout N-blocks are
// whole 16-output MFMA tiles.
bool gemm_supported(const tbh_weight &w) {
    if (w.mfma_tiles || w.K % 8 != 0 || w.Kp >= (int64_t)kDead / 1024) return false;
    if (w.path == Path::Int8Row || w.path == Path::Int4KGroup) return true;
    return w.path == Path::Int4NGroup && !w.ng_pairs && !w.zp && w.ng_scaled != nullptr &&
           (w.rows_per_nblock % 16 == 0 || w.rows_per_nblock >= w.Np) &&
           w.n_scales_dev * (int64_t)sizeof(float) < (int64_t)kDead;
}

// 16-bit pieces per x row that a product of M rows writes to scratch: none of
// bf16 x on INT8 rows and INT4 K-groups (read as given), one of bf16 x on
// runtime-layout INT4; fp32 x two f16 pieces (22 bits of x) past 64 rows, three
// bf16 pieces (all of it, as the GEMV kernels read x) up to 64, where the third
// costs little: the weights' bytes are the bound.  M is the whole product's:
// its parts (gemm_rows) are all of one form.
int gemm_pieces(const tbh_weight &w, bool f32, int64_t M) {
    if (!f32) return w.path == Path::Int4NGroup ? 1 : 0;
    return M > 64 ? 2 : 3;
}

// Bytes of scratch that `rows` rows of x take as pieces, with their row
// exponents ahead of them.
size_t gemm_pieces_bytes(const tbh_weight &w, int pieces, int64_t rows) {
    if (pieces == 0) return 0;
    const int64_t ldp = (w.K + kBK - 1) / kBK * kBK;
    const size_t eb = ((size_t)rows * sizeof(int32_t) + 255) / 256 * 256;
    return eb + ((size_t)(pieces * rows * ldp) * 2 + 255) / 256 * 256;
}

static hipError_t launch_kind(const Args &a, int kind, int xp, const Plan &pl, int64_t blocks, hipStream_t s) {
    const bool zp = a.zp != nullptr;
    if (kind == W8) return launch_w8(a, xp, zp, pl.tm, pl.tn, (unsigned)blocks, s);
    if (kind == W4K) return launch_w4k(a, xp, zp, pl.tm, pl.tn, (unsigned)blocks, s);
    return launch_w4n(a, xp, zp, pl.tm, pl.tn, (unsigned)blocks, s);
}

// The plan `pl` in a fixed scratch that does not hold its pieces and partial
// tiles at once (the no-allocation entry, whose results are those of the
// device entry bit for bit): the pieces of as many rows as fit at a time, and
// the K parts one launch after the other, each added to y.
static hipError_t launch_seq(Args a, int kind, int xp, const Plan &pl, const void *x, bool f32, int64_t ldx, int64_t M,
                             hipStream_t s, const Scratch &scr) {
    const int64_t bm = 16 * pl.tm, ldp = (a.K + kBK - 1) / kBK * kBK;
    const size_t room = scr.fixed_bytes - std::min(scr.fixed_bytes, scr.offset);
    const size_t per16 = 16 * (sizeof(int32_t) + (size_t)xp * ldp * 2) + 512;   // two paddings at most
    const int64_t fit = (int64_t)(room / per16) * 16;
    if (fit < 16) {
        scr.shortfall = scr.offset + per16;
        return hipErrorNotReady;
    }
    const int parts = pl.splits > 1 ? pl.splits : 1;
    a.seq = 1;
    a.tail_parts = pl.tail_parts;
    a.tail_first = a.tiles_m * a.tiles_n - pl.tail_r;
    a.ldx = a.xk = (int32_t)ldp;
    for (int64_t r0 = 0; r0 < M;) {
        const int64_t tm = r0 / bm;
        int64_t r1 = std::min(M, r0 + fit);
        if (r1 < M) r1 = r1 / bm > tm ? r1 / bm * bm : r1;   // whole tile rows, or a piece of one
        if (r0 % bm) r1 = std::min(r1, (tm + 1) * bm);
        const int64_t rows = r1 - r0;
        const size_t eb = ((size_t)rows * sizeof(int32_t) + 255) / 256 * 256;
        char *buf = (char *)scr.get(s, eb + (size_t)(xp * rows * ldp) * 2);
        if (!buf) return hipErrorOutOfMemory;
        int32_t *re = (int32_t *)buf;
        uint16_t *xq = (uint16_t *)(buf + eb);
        a.piece_stride = rows * ldp;
        const char *src = (const char *)x + r0 * ldx * (f32 ? 4 : 2);
        hipError_t e = launch_split_x(src, f32, xp, ldx, a.K, rows, re, xq, ldp, a.piece_stride, s);
        if (e != hipSuccess) return e;
        a.row_exp = re;
        a.x = xq;
        a.row_base = (int32_t)r0;
        a.row_end = (int32_t)r1;
        a.seq_tm = (int32_t)tm;
        a.seq_tms = (int32_t)((r1 - 1) / bm - tm + 1);
        const int64_t blocks = (int64_t)a.seq_tms * a.tiles_n;
        for (int j = 0; j < parts + pl.tail_parts; ++j) {
            a.seq_tail = j >= parts;
            a.seq_part = a.seq_tail ? j - parts : j;
            a.seq_steps = a.seq_tail ? pl.tail_steps : pl.splits > 1 ? pl.sps : a.nsteps;
            a.add = a.seq_part > 0;
            e = launch_kind(a, kind, xp, pl, blocks, s);
            if (e != hipSuccess) return e;
        }
        r0 = r1;
    }
    return hipSuccess;
}

// hipErrorNotReady, before anything is enqueued, when the pieces' scratch is
// not to be had; hipErrorInvalidConfiguration, likewise, for pieces that no
// tile of the weight's kind takes (three on runtime-layout INT4, which
// prefill's rule never asks for).
hipError_t launch_gemm(const tbh_weight &w, const void *x, bool f32, int nx, int64_t ldx, int64_t M, float *y,
                       int64_t ldy, hipStream_t s, const Scratch &scr) {
    const int kind = w.path == Path::Int8Row ? W8 : w.path == Path::Int4KGroup ? W4K : W4N;
    const int xp = std::max(nx, 1);
    const int64_t cus = std::max(1, w.dev->cu_count);
    Args a{};
    a.y = y;
    a.ldy = ldy;
    a.data = w.data;
    a.row_bytes = w.row_bytes;
    a.scales = kind == W4N ? w.ng_scaled : w.scales;
    a.scale_bytes = w.n_scales_dev * (int64_t)sizeof(float);
    a.zp = w.zp;
    a.nb_exp = w.ng_sexp;
    a.M = (int32_t)M;
    a.K = (int32_t)w.K;
    a.N = (int32_t)w.N;
    a.Np = (int32_t)w.Np;
    a.chunks = (int32_t)(w.Kp / (kind == W8 ? kInt8ChunkElems : kInt4ChunkElems));
    a.G = (int32_t)w.groups_per_row;
    a.cpg_magic = (((uint64_t)1 << 32) + w.chunks_per_group - 1) / w.chunks_per_group;
    a.rpn = w.rows_per_nblock;
    a.kp = (int32_t)w.Kp;
    a.nsteps = (int32_t)((w.K + kBK - 1) / kBK);
    a.vec = ldy % 4 == 0 && ((uintptr_t)y & 15) == 0;

    // scratch: the pieces of x, then the partial tiles
    Plan pl = choose(kind, xp, M, w.N, a.nsteps, cus, ldy == w.N);
    if (pl.sps == 0) return hipErrorInvalidConfiguration;
    const size_t pieces = gemm_pieces_bytes(w, nx, M);
    const int64_t n = M * w.N;
    size_t part_bytes = pl.splits > 1 ? (size_t)(pl.splits * n) * sizeof(float)
                                      : (size_t)pl.tail_parts * pl.tail_r * (16 * pl.tm) * (128 * pl.tn) * sizeof(float);
    char *buf = pieces + part_bytes ? (char *)scr.get(s, pieces + part_bytes) : nullptr;
    auto set_tiles = [&] {
        a.tiles_m = (int32_t)((M + 16 * pl.tm - 1) / (16 * pl.tm));
        a.tiles_n = (int32_t)((w.N + 128 * pl.tn - 1) / (128 * pl.tn));
    };
    set_tiles();
    // neighbouring tiles share the operand that is the larger in memory
    a.n_fast = (double)M * (double)w.K * 2 * xp > (double)w.N * (double)w.row_bytes;
    if (!buf && pieces && scr.is_fixed()) return launch_seq(a, kind, xp, pl, x, f32, ldx, M, s, scr);
    if (!buf && part_bytes) {   // no room for partial tiles: one pass
        pl = choose(kind, xp, M, w.N, a.nsteps, cus, false);
        set_tiles();
        part_bytes = 0;
        buf = pieces ? (char *)scr.get(s, pieces) : nullptr;
    }
    if (pieces && !buf) return hipErrorNotReady;
    if (pieces) {
        const size_t eb = ((size_t)M * sizeof(int32_t) + 255) / 256 * 256;
        int32_t *re = (int32_t *)buf;
        uint16_t *xq = (uint16_t *)(buf + eb);
        a.ldx = (w.K + kBK - 1) / kBK * kBK;
        a.xk = (int32_t)a.ldx;
        a.piece_stride = M * a.ldx;
        const hipError_t e = launch_split_x(x, f32, xp, ldx, a.K, M, re, xq, a.ldx, a.piece_stride, s);
        if (e != hipSuccess) return e;
        a.row_exp = re;
        a.x = xq;
    } else {
        a.x = (const uint16_t *)x;
        a.ldx = ldx;
        a.xk = a.K;
    }
    float *part = part_bytes ? (float *)(buf + pieces) : nullptr;

    const int64_t bm = 16 * pl.tm, bn = 128 * pl.tn;
    const int64_t tiles = (int64_t)a.tiles_m * a.tiles_n;
    int64_t blocks = tiles;
    a.split_steps = a.nsteps;
    if (pl.splits > 1) {
        a.split_steps = pl.sps;
        a.y = part;
        a.split_stride = n;
        a.vec = w.N % 4 == 0;
        blocks = tiles * pl.splits;
        a.main_blocks = (int32_t)blocks;
    } else if (pl.tail_parts) {
        a.tail_part = part;
        a.tail_parts = pl.tail_parts;
        a.tail_steps = pl.tail_steps;
        a.tail_n = pl.tail_r;
        a.tail_first = (int32_t)(tiles - pl.tail_r);
        a.main_blocks = a.tail_first;
        blocks = a.tail_first + (int64_t)pl.tail_r * pl.tail_parts;
    } else {
        a.main_blocks = (int32_t)tiles;
    }
    a.row_end = (int32_t)M;
    const hipError_t e = launch_kind(a, kind, xp, pl, blocks, s);
    if (e != hipSuccess) return e;
    if (pl.splits > 1) return launch_split_sum(part, pl.splits, y, n, cus, s);
    if (pl.tail_parts) {
        const int64_t n4 = (int64_t)pl.tail_r * bm * bn / 4;
        hipLaunchKernelGGL(tail_sum, dim3((unsigned)std::min<int64_t>(4 * cus, (n4 + 255) / 256)), dim3(256), 0, s, a,
                           (int)bm, (int)bn);
        return hipGetLastError();
    }
    return hipSuccess;
}

}  // namespace tbh
