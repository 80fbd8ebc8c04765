// Prompt-sized projections with the f64 contract on the int8 matrix cores.
//
// The contract is that of model_ops.hip: y = f32(sum_k f64(w[n][k]) * f64(h[m][k])), the
// reference CPU model's matvec (engine/src/ops.rs:17-32), with RMSNorm, residual and SwiGLU
// fused. linear_gemm_kernel runs it on the f64 MFMA, whose rate (64 MACs per CU and cycle)
// bounds it; the int8 MFMA does 4096. So the operands are written as sums of signed 8-bit
// digits, every digit product is an exact int8 GEMM with int32 sums, and the sums join in
// f64 at the end:
//   - a weight is a whole multiple of 2^-24 (fp16's smallest step): w = 2^-24 sum_j w_j
//     256^(2-j), 3 digits for |w| < 0.498, a 4th (j = -1) up to |w| <= 127;
//   - a row of activations is scaled by a power of two to |X| < 2^46 and rounded to a whole
//     number: X = sum_i x_i 256^(5-i), 6 digits. An f32 within 2^22 of its row's largest
//     value keeps every bit; what the rounding of a smaller one drops is listed, up to 16
//     elements a row, and multiplied in f64 with the sums (of rows of 768 N(0,1) values about
//     one in three thousand has such an element, of SwiGLU outputs one in thirty);
//   - digit products of equal weight, s = i + j, share an accumulator: 18 products (i, j)
//     in 8 accumulators (a ninth with the fourth weight digit), 15 where the last activation
//     digit is zero over 32 rows and 32 keys: it holds bits only of elements 2^14 below their
//     row's largest (about one in twelve such pieces of N(0,1) rows of 768 has any).
// So every product is exact, and the sums are joined in f64. Rows that this does not fit (a
// non-finite value, a largest value outside 2^-60 .. 2^22, more than 16 rounded elements) and
// columns with a weight over 127 or not finite take plain f64 sums instead, 32 x 32 outputs at
// a time.
//
// Two launches: digits_kernel writes the digit planes of both operands into the caller's
// workspace in MFMA operand order, digits_gemm_kernel multiplies them.
//
// Included by model_ops.hip, whose floating-point contraction setting (off) it relies on.
#pragma once

#include "common.hpp"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace crucible {
namespace {

enum DigitMode { kDigitPlain = 0, kDigitResidual = 1, kDigitSwiGLU = 2 };

constexpr int kDecodeRows = 32;  // batches up to here keep the decode tilings
constexpr int64_t kWideOutputs = 16 * 1024;  // decode tilings: several column blocks a workgroup

struct DigitLinear {
    const float* x;
    int64_t ldx;
    const float* norm_w;  // fused RMSNorm weight, or nullptr
    double eps;
    const half_t* w;      // [n_out][k_in]; the gate rows when w2 is set
    const half_t* w2;     // SwiGLU: the up rows
    const float* resid;
    float* out;
    int64_t ldo;
    int rows;
    int n_out;
    int k_in;
};

typedef double double4_t __attribute__((ext_vector_type(4)));
typedef int32_t i32x4_t __attribute__((ext_vector_type(4)));
typedef int32_t i32x16_t __attribute__((ext_vector_type(16)));

constexpr int kXDigits = 6;
constexpr int kWDigits = 4;         // the last one is zero for |w| < 0.498
constexpr int kBlk = 32;            // rows (columns) of an operand block
constexpr int kStep = 32;           // K of one MFMA
constexpr int kFrag = kBlk * kStep; // bytes of one digit of an operand block: 1 KiB
constexpr int kXBlk = kXDigits * kFrag;
constexpr int kWBlk = kWDigits * kFrag;
constexpr int kPart = 128;          // K range of one weight workgroup
constexpr int kWgRows = 8;          // rows of one activation workgroup
constexpr int kRowWgs = kBlk / kWgRows;
constexpr int kMaxK = 16384;        // 4 products of 2^14 a key stay below 2^31
constexpr int kRests = 16;          // listed elements of a row

// What the digits of element k leave of it, in units of X.
struct Rest {
    int k;
    float r;
};

// Workspace: the planes' blocks first (1 KiB aligned), then the rows' scales and rests, then
// flags (rows: 1 f64 sums, 2 some row has rests; columns: 1 a fourth digit, 2 f64 sums; a byte
// for 8 rows and 32 keys: their last digit holds something).
//   x planes [row block][K / 32][6][1024], w planes [column block][K / 32][4][1024]
struct Layout {
    int64_t row_blks, col_blks, parts;
    int64_t w_off, scale_off, norm_off, rest_off, count_off, last_off, xflag_off, wflag_off, bytes;
};

Layout make_layout(int64_t rows, int64_t cols, int64_t k_in) {
    Layout l;
    const int64_t steps = k_in / kStep;
    // 64-row and 64-column tiles: both blocks of the last tile exist
    l.row_blks = (rows + 63) / 64 * 2;
    l.col_blks = (cols + 63) / 64 * 2;
    l.parts = (k_in + kPart - 1) / kPart;
    l.w_off = l.row_blks * steps * kXBlk;
    l.scale_off = l.w_off + l.col_blks * steps * kWBlk;
    l.norm_off = l.scale_off + l.row_blks * kBlk * 8;
    l.rest_off = l.norm_off + l.row_blks * kBlk * 8;
    l.count_off = l.rest_off + l.row_blks * kBlk * kRests * (int64_t)sizeof(Rest);
    l.last_off = l.count_off + l.row_blks * kBlk * 4;
    l.xflag_off = l.last_off + l.row_blks * steps * kRowWgs;
    l.wflag_off = l.xflag_off + l.row_blks * kRowWgs * 4;
    l.bytes = l.wflag_off + l.col_blks * l.parts * 4;
    return l;
}

struct DigitArgs {
    DigitLinear p;
    unsigned char* ws;
    Layout l;
    int row_wgs;    // digits_kernel: workgroups of the activations
    int row_tiles;  // 64 x 64 output tiles
    int col_tiles;
    int per_xcd;
};

// The weight row behind column c of the product. SwiGLU interleaves 16 gate columns with
// the up columns of the same outputs, so one 32-column block holds both halves.
__device__ __forceinline__ const half_t* weight_row(const DigitLinear& p, int c, bool& ok) {
    if (p.w2) {
        const int n = (c >> 5) * 16 + (c & 15);
        ok = n < p.n_out;
        return ((c & 16) ? p.w2 : p.w) + (int64_t)(ok ? n : 0) * p.k_in;
    }
    ok = c < p.n_out;
    return p.w + (int64_t)(ok ? c : 0) * p.k_in;
}

// Byte b of four words as one word (v_perm_b32 selects bytes of {first = 7..4, second = 3..0}).
__device__ __forceinline__ uint32_t bytes_of(uint32_t a0, uint32_t a1, uint32_t a2, uint32_t a3,
                                             int b) {
    const uint32_t lo = __builtin_amdgcn_perm(a1, a0, 0x0c0c0400u + 0x0101u * b);
    const uint32_t hi = __builtin_amdgcn_perm(a3, a2, 0x04000c0cu + 0x01010000u * b);
    return lo | hi;
}

// ---------------------------------------------------------------- digit planes

constexpr int kDigitThreads = 256;

// Memory-bound: 4 B read and 6 written per activation, 2 and 4 per weight. A thread
// handles groups of 16 consecutive K of a row, the 16 bytes one lane supplies to an MFMA for
// each digit; 8 neighbouring lanes hold 8 rows, so a digit's stores are 128-byte runs (8 rows
// a workgroup against 16: 4,713 x 2048 22.4 -> 19.4 us, 1,003 x 768 12.6 -> 11.4). The digits
// need the row's norm and largest value first: with G > 0 (k_in <= 512 G) a thread's groups wait
// in registers, loaded at once; G = 0 reads the row twice.
template <int G, bool NORM>
__global__ __launch_bounds__(kDigitThreads) void digits_kernel(DigitArgs a) {
    __shared__ double s_ss[32][kWgRows];
    __shared__ uint32_t s_mx[32][kWgRows];
    __shared__ Rest s_rest[kWgRows][kRests];
    __shared__ int s_rests[kWgRows];
    __shared__ int s_flag;
    const DigitLinear& p = a.p;
    const int tid = threadIdx.x;
    const int steps = p.k_in / kStep;
    const int r = tid & 7, kg = tid >> 3;  // row (of 8), group of 16 K (of 32)

    if ((int)blockIdx.x >= a.row_wgs) {
        // ---- weights: 32 rows x kPart
        const int id = blockIdx.x - a.row_wgs;
        const int blk = id / (int)a.l.parts, part = id - blk * (int)a.l.parts;
        if (tid == 0) s_flag = 0;
        __syncthreads();
        const int row = tid & 31;
        const int k = part * kPart + (tid >> 5) * 16;
        if (k < p.k_in) {
            bool ok;
            const half_t* src = weight_row(p, blk * kBlk + row, ok) + k;
            half8_t v[2];
            v[0] = *reinterpret_cast<const half8_t*>(src);
            v[1] = *reinterpret_cast<const half8_t*>(src + 8);
            uint32_t wv[16];
            int flag = 0;
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const float f = ok ? (float)v[e >> 3][e & 7] : 0.0f;
                const bool fits = fabsf(f) <= 127.0f;  // false for NaN
                const int wi = fits ? (int)(f * 16777216.0f) : 0;
                wv[e] = ((uint32_t)wi + 0x808080u) ^ 0x808080u;
                flag |= fits ? ((wv[e] >> 24) != 0 ? 1 : 0) : 2;
            }
            unsigned char* dst = a.ws + a.l.w_off + ((int64_t)blk * steps + k / kStep) * kWBlk +
                                 ((k & 16) ? 512 : 0) + row * 16;
#pragma unroll
            for (int j = 0; j < kWDigits; ++j) {  // digit j: bytes 2, 1, 0, then 3
                const int b = j < 3 ? 2 - j : 3;
                u32x4_t o;
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    o[q] = bytes_of(wv[4 * q], wv[4 * q + 1], wv[4 * q + 2], wv[4 * q + 3], b);
                *reinterpret_cast<u32x4_t*>(dst + j * kFrag) = o;
            }
            if (flag) atomicOr(&s_flag, flag);
        }
        __syncthreads();
        if (tid == 0) reinterpret_cast<int*>(a.ws + a.l.wflag_off)[id] = s_flag;
        return;
    }

    // ---- activations: 8 rows, all of K
    const int row = blockIdx.x * kWgRows + r;
    const bool ok = row < p.rows;
    const float* src = p.x + (int64_t)(ok ? row : 0) * p.ldx;
    const int groups = p.k_in / 16;
    struct Group {
        float4_t x[4], nw[NORM ? 4 : 1];
    };
    auto load = [&](int g, Group& v) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            v.x[q] = *reinterpret_cast<const float4_t*>(src + g * 16 + 4 * q);
            if constexpr (NORM)
                v.nw[q] = *reinterpret_cast<const float4_t*>(p.norm_w + g * 16 + 4 * q);
        }
    };
    // first pass: the f64 sum of squares and a bound of the largest |h|, as float bits (an
    // infinity or a NaN is the largest)
    double ss = 0.0;
    uint32_t mx = 0;
    auto measure = [&](const Group& v) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float m = v.x[q][e];
                if constexpr (NORM) {
                    const double d = (double)m;
                    ss += d * d;
                    m *= v.nw[q][e];
                }
                mx = max(mx, __builtin_bit_cast(uint32_t, m) & 0x7fffffffu);
            }
    };
    Group held[G > 0 ? G : 1];
    if constexpr (G > 0) {
        // a group past the row's end re-reads the last one: its digits are not written
#pragma unroll
        for (int i = 0; i < G; ++i) load(min(kg + 32 * i, groups - 1), held[i]);
#pragma unroll
        for (int i = 0; i < G; ++i)
            if (kg + 32 * i < groups) measure(held[i]);
    } else {
        for (int g = kg; g < groups; g += 32) {
            load(g, held[0]);
            measure(held[0]);
        }
    }
    s_ss[kg][r] = ss;
    s_mx[kg][r] = mx;
    if (tid < kWgRows) s_rests[tid] = 0;
    if (tid == 0) s_flag = 0;
    __syncthreads();
    double tot = 0.0;
    mx = 0;
#pragma unroll
    for (int i = 0; i < 32; ++i) {
        tot += s_ss[i][r];
        mx = max(mx, s_mx[i][r]);
    }
    const double scale = NORM ? 1.0 / sqrt(tot / (double)p.k_in + p.eps) : 1.0;
    // |h| <= bound (1 + 2^-18 covers the roundings of h, unless x * scale is subnormal: those
    // rows are found by their values below), so |h| 2^(21 - e) < 2^22 with e the exponent of
    // 2^e > bound / 2
    const float bound = (float)((double)__builtin_bit_cast(float, mx) * scale * 1.00001);
    const int e = (int)((__builtin_bit_cast(uint32_t, bound) >> 23) & 255) - 127;
    // Usual magnitudes only: every power of two below is a normal f32, and the scaling up exact.
    // x * norm_w below the normal range bounds nothing: the row's scale may lift h out of it.
    const bool usual = mx >= 0x00800000u && mx < 0x7f800000u && e >= -60 && e <= 21;  // up >= 1
    // a zero row stays one unless eps lets its scale be infinite
    const bool zero = mx == 0 && (!NORM || (tot == 0.0 && scale < (double)INFINITY));
    const float up = usual ? __builtin_bit_cast(float, (uint32_t)(21 - e + 127) << 23) : 0.0f;
    unsigned char* blk = a.ws + (int64_t)(row >> 5) * steps * kXBlk + (row & 31) * 16;
    auto write = [&](int g, const Group& v) {
        uint32_t hi[16], lo[16], rounded = 0;
        auto scaled = [&](int e) {
            float h = v.x[e >> 2][e & 3];
            if constexpr (NORM) h = (float)((double)h * scale) * v.nw[e >> 2][e & 3];
            return ok && usual ? h * up : 0.0f;                     // exact
        };
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float t = scaled(4 * q + i);
                if constexpr (NORM)
                    if (fabsf(t) >= 4194304.0f) s_flag = 1;
                const float th = rintf(t);
                const float tl = (t - th) * 16777216.0f;            // exact, |tl| <= 2^23
                const float tr = rintf(tl);                         // rounds below 2^-22 of the largest
                const uint32_t l = (uint32_t)((int)tr + 0x808080);  // 25 bits, carry on top
                rounded |= tl != tr ? 1u << (4 * q + i) : 0u;
                hi[4 * q + i] = ((uint32_t)((int)th + (int)(l >> 24) + 0x808080)) ^ 0x808080u;
                lo[4 * q + i] = l ^ 0x808080u;
            }
        if (rounded) {
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                if (!(rounded >> i & 1)) continue;
                const float t = scaled(i), tl = (t - rintf(t)) * 16777216.0f;
                const int at = atomicAdd(&s_rests[r], 1);
                if (at < kRests) s_rest[r][at] = {g * 16 + i, tl - rintf(tl)};  // exact
            }
        }
        uint32_t last = 0;
#pragma unroll
        for (int i = 0; i < 16; ++i) last |= lo[i];
        // 16 neighbouring lanes hold the 8 rows' 32 keys
        const uint64_t some = __ballot((last & 255u) != 0) >> (tid & 48);
        if ((tid & 15) == 0)
            a.ws[a.l.last_off + ((int64_t)(row >> 5) * steps + (g >> 1)) * kRowWgs + (blockIdx.x & (kRowWgs - 1))] =
                (some & 0xffffu) != 0;
        unsigned char* dst = blk + (int64_t)(g >> 1) * kXBlk + ((g & 1) ? 512 : 0);
#pragma unroll
        for (int i = 0; i < kXDigits; ++i) {
            u32x4_t o;
#pragma unroll
            for (int q = 0; q < 4; ++q)
                o[q] = i < 3 ? bytes_of(hi[4 * q], hi[4 * q + 1], hi[4 * q + 2], hi[4 * q + 3], 2 - i)
                             : bytes_of(lo[4 * q], lo[4 * q + 1], lo[4 * q + 2], lo[4 * q + 3], 5 - i);
            *reinterpret_cast<u32x4_t*>(dst + i * kFrag) = o;
        }
    };
    if constexpr (G > 0) {
#pragma unroll
        for (int i = 0; i < G; ++i)
            if (kg + 32 * i < groups) write(kg + 32 * i, held[i]);
    } else {
        for (int g = kg; g < groups; g += 32) {
            load(g, held[0]);
            write(g, held[0]);
        }
    }
    __syncthreads();
    const int n_rest = s_rests[r];
    if (kg == 0) {
        // 2^(e - 45) per unit of X, 2^-24 per unit of W
        reinterpret_cast<double*>(a.ws + a.l.scale_off)[row] =
            usual ? __builtin_bit_cast(double, (uint64_t)(e - 69 + 1023) << 52) : 0.0;
        reinterpret_cast<double*>(a.ws + a.l.norm_off)[row] = scale;
        reinterpret_cast<int*>(a.ws + a.l.count_off)[row] = min(n_rest, kRests);
        if (ok && !zero && (!usual || n_rest > kRests)) atomicOr(&s_flag, 1);
        if (n_rest > 0) atomicOr(&s_flag, 2);
    }
    // in the order of k, whatever order the threads came in
    if (kg < min(n_rest, kRests)) {
        const Rest mine = s_rest[r][kg];
        int rank = 0;
        for (int i = 0; i < min(n_rest, kRests); ++i) rank += s_rest[r][i].k < mine.k;
        reinterpret_cast<Rest*>(a.ws + a.l.rest_off)[(int64_t)row * kRests + rank] = mine;
    }
    __syncthreads();
    if (tid == 0) reinterpret_cast<int*>(a.ws + a.l.xflag_off)[blockIdx.x] = s_flag;
}

// ---------------------------------------------------------------- digit products

constexpr int kDigitGemmThreads = 256;
constexpr int kGroups = 9;                 // s = i + j = -1 .. 7
constexpr int kStageK = 64;                // K of a stage: two MFMA steps
constexpr int kStageX = 2 * 2 * kXBlk;     // 2 row blocks x 2 steps: 24 KiB
constexpr int kStage = kStageX + 2 * 2 * 3 * kFrag;  // 2 column blocks x 2 steps, 3 digits

// 32 x 32 outputs of one wave as f64 sums, for the rows and columns that the digits do not hold:
// linear_gemm_kernel's wave (the f64 MFMA, operands from L2 into registers two 32-key chunks
// ahead, the same keys a step), with the rows' scales from the workspace. MFMA-bound: 1,024 f64
// products of 64 cycles for 1,024 keys. One element at a time a lane (2-byte loads, a serial
// sum) took 60 ms for a layer's four products of 4,713 rows with one such row in 32, these 1.13,
// linear_gemm_kernel alone 1.09; 13.3, 0.31 and 0.29 at 1,003 rows.
template <int MODE, bool NORM>
struct F64Block {
    struct Chunk {
        float4_t x[2][2], nw[NORM ? 2 : 1];
        half8_t w[2];
    };
    const float* xp[2];
    const float* nwp;
    const half_t* wp[2];
    double scale[2];
    bool col_ok[2];
    double4_t acc[2][2];

    __device__ __forceinline__ void init(const DigitArgs& a, int row_blk, int col_blk, int lane) {
        const DigitLinear& p = a.p;
        const int col = lane & 15, g = lane >> 4;
        nwp = NORM ? p.norm_w + 8 * g : nullptr;
#pragma unroll
        for (int b = 0; b < 2; ++b) {  // past the end: the last row, and the first weight row
            const int row = row_blk * kBlk + 16 * b + col;
            xp[b] = p.x + (int64_t)min(row, p.rows - 1) * p.ldx + 8 * g;
            scale[b] = reinterpret_cast<const double*>(a.ws + a.l.norm_off)[row];
            wp[b] = weight_row(p, col_blk * kBlk + 16 * b + col, col_ok[b]) + 8 * g;
            acc[b][0] = acc[b][1] = double4_t{0.0, 0.0, 0.0, 0.0};
        }
    }
    __device__ __forceinline__ void load(int k0, Chunk& c) const {
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            c.x[b][0] = *reinterpret_cast<const float4_t*>(xp[b] + k0);
            c.x[b][1] = *reinterpret_cast<const float4_t*>(xp[b] + k0 + 4);
            c.w[b] = *reinterpret_cast<const half8_t*>(wp[b] + k0);
            if constexpr (NORM) c.nw[b] = *reinterpret_cast<const float4_t*>(nwp + k0 + 4 * b);
        }
    }
    __device__ __forceinline__ void feed(const Chunk& c) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            double x[2], w[2];
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                float h = c.x[b][i >> 2][i & 3];
                if constexpr (NORM) h = (float)((double)h * scale[b]) * c.nw[i >> 2][i & 3];
                x[b] = (double)h;
                w[b] = (double)(float)c.w[b][i];
            }
#pragma unroll
            for (int j = 0; j < 4; ++j)
                acc[j >> 1][j & 1] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[j >> 1], w[j & 1],
                                                                         acc[j >> 1][j & 1], 0, 0, 0);
        }
    }
    __device__ __forceinline__ void run(int k_in) {  // a multiple of 64
        Chunk c0, c1;
        load(0, c0);
        __builtin_amdgcn_sched_barrier(0);
        load(32, c1);
        __builtin_amdgcn_sched_barrier(0);
        for (int k0 = 0; k0 < k_in; k0 += 64) {  // the last loads are made again, unused
            feed(c0);
            __builtin_amdgcn_sched_barrier(0);
            load(min(k0 + 64, k_in - 64), c0);
            __builtin_amdgcn_sched_barrier(0);
            feed(c1);
            __builtin_amdgcn_sched_barrier(0);
            load(min(k0 + 96, k_in - 32), c1);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    __device__ __forceinline__ void store(const DigitLinear& p, int row_blk, int col_blk, int lane) const {
        const int col = lane & 15, g = lane >> 4;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int row = row_blk * kBlk + 16 * (i >> 2) + g + 4 * (i & 3);
            if (row >= p.rows) continue;
            float* out = p.out + (int64_t)row * p.ldo;
            if constexpr (MODE == kDigitSwiGLU) {
                const float gate = (float)acc[i >> 2][0][i & 3], up = (float)acc[i >> 2][1][i & 3];
                if (col_ok[0]) out[col_blk * 16 + col] = gate / (1.0f + expf(-gate)) * up;
            } else {
#pragma unroll
                for (int b = 0; b < 2; ++b) {
                    const int n = col_blk * kBlk + 16 * b + col;
                    const float y = (float)acc[i >> 2][b][i & 3];
                    if (!col_ok[b]) continue;
                    // out may alias resid: each element is read and written by the same lane
                    out[n] = MODE == kDigitResidual ? p.resid[(int64_t)row * p.ldo + n] + y : y;
                }
            }
        }
    }
};

template <int MODE>
__device__ __forceinline__ void f64_block(const DigitArgs& a, int row_blk, int col_blk, int lane) {
    auto go = [&](auto norm_tag) {
        F64Block<MODE, decltype(norm_tag)::value> f;
        f.init(a, row_blk, col_blk, lane);
        f.run(a.p.k_in);
        f.store(a.p, row_blk, col_blk, lane);
    };
    if (a.p.norm_w) go(std::true_type{});
    else go(std::false_type{});
}

// A 64 x 64 output tile per workgroup of 4 waves, 32 x 32 a wave. MFMA-bound: 15 products of
// 32x32x32 a wave and step (18 with the last activation digit, up to 24 with the fourth weight
// digit) against 9 KiB of LDS reads.
// Stages of 64 keys stream into two LDS buffers with direct-to-LDS loads, the next stage's
// issued between the products; the planes are stored in operand order, so both the copy and
// the reads are linear in the lane and free of bank conflicts. Two workgroups a CU (73.7 KB
// of LDS each): one multiplies while the other waits at its barrier. The weights' fourth
// digit, rare, goes from global memory to registers.
//
// With every SIMD busy on random digits the part runs a 32x32x32 product in 20 ns (13.7 with
// a few CUs busy): 133 to 160 us for the gate/up product of 4,713 rows, traced 205.
// Measured slower: steps of 32 in a ring of 4 (2 workgroups a CU) or 8 buffers, operands
// double-buffered in registers, 32 x 64 outputs a wave (one wave a SIMD, 512 VGPRs), and, for
// grids below the CU count, a second set of 4 waves on every other stage of K.
//
// int8 MFMA 32x32x32: lane l supplies row (column) l & 31 and 16 of the step's 32 keys, the
// half l >> 5 of them (the same keys for both operands), and holds
// D[8 (i >> 2) + 4 (l >> 5) + (i & 3)][l & 31].
template <int MODE>
__global__ __launch_bounds__(kDigitGemmThreads, 2) void digits_gemm_kernel(DigitArgs a) {
    __shared__ __align__(1024) unsigned char s_buf[2][kStage];
    const DigitLinear& p = a.p;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wr = wave >> 1, wc = wave & 1;

    // Workgroup L runs on XCD L % 8; each XCD takes a contiguous piece of the tile list,
    // which walks groups of 8 row tiles column by column: the group's x planes (2.4 MB at
    // K = 768) and a column's w planes stay in the XCD's L2.
    const int L = blockIdx.x;
    const int t = (L & 7) * a.per_xcd + (L >> 3);
    if (t >= a.row_tiles * a.col_tiles) return;  // uniform over the workgroup
    const int group = t / (8 * a.col_tiles);
    const int in_group = min(8, a.row_tiles - 8 * group);
    const int rem = t - group * 8 * a.col_tiles;
    const int ct = rem / in_group;
    const int rt = group * 8 + rem - ct * in_group;

    const int steps = p.k_in / kStep;
    const int n_stage = p.k_in / kStageK;
    const unsigned char* wp = a.ws + a.l.w_off + (int64_t)(2 * ct) * steps * kWBlk;

    // Flags: f64 for the wave's outputs if its row or column block needs it, a fourth weight
    // digit if one is nonzero anywhere in the wave's columns.
    const int* xf = reinterpret_cast<const int*>(a.ws + a.l.xflag_off) + 2 * rt * kRowWgs;
    const int* wf = reinterpret_cast<const int*>(a.ws + a.l.wflag_off) + (int64_t)(2 * ct) * a.l.parts;
    const int parts = (int)a.l.parts;
    const int x_lane = xf[lane & (2 * kRowWgs - 1)];
    int w_lane = 0;  // the second block's flags two bits up
    for (int i = lane; i < 2 * parts; i += 64) w_lane |= wf[i] << (i < parts ? 0 : 2);
    int xflags[2], wflags[2];  // of the tile's row and column blocks
#pragma unroll
    for (int b = 0; b < 2; ++b) {
        const uint64_t lanes = ((1ull << kRowWgs) - 1) << (b * kRowWgs);
        xflags[b] = ((__ballot(x_lane & 1) & lanes) ? 1 : 0) | ((__ballot(x_lane & 2) & lanes) ? 2 : 0);
        wflags[b] = (__ballot(w_lane & (1 << 2 * b)) ? 1 : 0) | (__ballot(w_lane & (2 << 2 * b)) ? 2 : 0);
    }
    const int xflag = wr ? xflags[1] : xflags[0], wflag = wc ? wflags[1] : wflags[0];
    const bool plain = (xflag & 1) != 0 || (wflag & 2) != 0;
    const bool four = (wflag & 1) != 0;
    // every wave's outputs are f64 sums: no digit is needed
    if ((xflags[0] & xflags[1] & 1) != 0 || (wflags[0] & wflags[1] & 2) != 0) {
        f64_block<MODE>(a, 2 * rt + wr, 2 * ct + wc, lane);
        return;
    }

    // One stage: 24 + 12 blocks of 1 KiB. x block (row block b, step q, digit i) goes to LDS
    // slot (b * 2 + q) * 6 + i, w block (b, q, j) to 24 + (b * 2 + q) * 3 + j. Wave w loads
    // (b, q) = (w >> 1, w & 1): 6 + 3 of them, at fixed distances from two running bases.
    const unsigned char* xsrc = a.ws + ((int64_t)(2 * rt + wr) * steps + wc) * kXBlk;
    const unsigned char* wsrc = wp + ((int64_t)wr * steps + wc) * kWBlk;
    const uint32_t lds0 = lds_offset(&s_buf[0][0]);
    const uint32_t voff = (uint32_t)lane * 16;
    auto issue_one = [&](int i, int buf) {  // i = 0 .. 8
        const uint32_t at = lds0 + (uint32_t)(buf * kStage);
        if (i < kXDigits) lds_dma16_base(xsrc + i * kFrag, voff, at + (uint32_t)((wave * 6 + i) * kFrag));
        else lds_dma16_base(wsrc + (i - 6) * kFrag, voff,
                            at + (uint32_t)(kStageX + (wave * 3 + i - 6) * kFrag));
    };

    i32x16_t acc[kGroups];
#pragma unroll
    for (int s = 0; s < kGroups; ++s)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[s][i] = 0;

    struct Frag {
        i32x4_t x[kXDigits], w[3];
    };
    // a step's flags of the last digit as one word
    typedef const __attribute__((address_space(4))) uint32_t* uniform_u32_ptr;
    const uniform_u32_ptr lasts =
        (uniform_u32_ptr)(a.ws + a.l.last_off + (int64_t)(2 * rt + wr) * steps * kRowWgs);
    auto read = [&](int buf, int q, Frag& f) {
        const unsigned char* base = &s_buf[buf][0] + lane * 16;
#pragma unroll
        for (int j = 0; j < 3; ++j)
            f.w[j] = *reinterpret_cast<const i32x4_t*>(base + kStageX + ((wc * 2 + q) * 3 + j) * kFrag);
#pragma unroll
        for (int i = 0; i < kXDigits; ++i)
            f.x[i] = *reinterpret_cast<const i32x4_t*>(base + ((wr * 2 + q) * 6 + i) * kFrag);
    };
    auto loop = [&](auto four_tag) {
        constexpr bool kFour = decltype(four_tag)::value;
        uint32_t last[2] = {lasts[0], lasts[1]};
        for (int st = 0; st < n_stage; ++st) {
            asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            // the stage is in LDS, and every wave has read the other buffer (stage st - 1)
            const int buf = st & 1;
            Frag f[2];
            read(buf, 0, f[0]);
            read(buf, 1, f[1]);
            // The next stage's loads; the last stage re-reads itself into the free buffer.
            const bool more = st + 1 < n_stage;
            xsrc += more ? 2 * kXBlk : 0;
            wsrc += more ? 2 * kWBlk : 0;
            const int ahead = 2 * (more ? st + 1 : st);
            const uint32_t next[2] = {lasts[ahead], lasts[ahead + 1]};
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                i32x4_t w4;
                if constexpr (kFour)
                    w4 = *reinterpret_cast<const i32x4_t*>(
                        wp + ((int64_t)wc * steps + 2 * st + q) * kWBlk + 3 * kFrag + lane * 16);
                auto product = [&](int i, int j, i32x4_t w) {
                    acc[i + j + 1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(f[q].x[i], w, acc[i + j + 1], 0, 0, 0);
                };
                // j outer: consecutive products go to different accumulators
                int n = 0, issued = 0;
#pragma unroll
                for (int j = 0; j < 3; ++j)
#pragma unroll
                    for (int i = 0; i < kXDigits - 1; ++i) {
                        product(i, j, f[q].w[j]);
                        if (!kFour && q == 0 && n * 3 % 5 < 3) {  // 9 of the 15
                            __builtin_amdgcn_sched_barrier(0);
                            issue_one(issued++, buf ^ 1);
                            __builtin_amdgcn_sched_barrier(0);
                        }
                        ++n;
                    }
                if constexpr (kFour) {
#pragma unroll
                    for (int i = 0; i < kXDigits - 1; ++i) product(i, -1, w4);
                }
                if (last[q]) {
#pragma unroll
                    for (int j = 0; j < 3; ++j) product(kXDigits - 1, j, f[q].w[j]);
                    if constexpr (kFour) product(kXDigits - 1, -1, w4);
                }
            }
            last[0] = next[0];
            last[1] = next[1];
            if constexpr (kFour)
#pragma unroll
                for (int i = 0; i < 9; ++i) issue_one(i, buf ^ 1);
        }
    };
#pragma unroll
    for (int i = 0; i < 9; ++i) issue_one(i, 0);
    // The choice is per wave, and the loops pass the same barriers.
    if (plain) {
        // Only its share of the other waves' stages, then the f64 sums. (Taking 64 keys to each
        // stage instead was no faster: the digits of the CU's other workgroup take turns with
        // the f64 products on the matrix unit either way.)
        for (int st = 0; st < n_stage; ++st) {
            asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            const bool more = st + 1 < n_stage;
            xsrc += more ? 2 * kXBlk : 0;
            wsrc += more ? 2 * kWBlk : 0;
#pragma unroll
            for (int i = 0; i < 9; ++i) issue_one(i, (st & 1) ^ 1);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        f64_block<MODE>(a, 2 * rt + wr, 2 * ct + wc, lane);
        return;
    }
    if (four) loop(std::true_type{});
    else loop(std::false_type{});
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no load into LDS outlives the workgroup

    // ---- outputs: column c of the wave's block, rows 8 (i >> 2) + 4 (lane >> 5) + (i & 3)
    const int r0 = (2 * rt + wr) * kBlk + 4 * (lane >> 5);
    const double* scales = reinterpret_cast<const double*>(a.ws + a.l.scale_off);
    const int c = (2 * ct + wc) * kBlk + (lane & 31);
    bool col_ok;
    const half_t* wrow = weight_row(p, c, col_ok);
    const int n = MODE == kDigitSwiGLU ? (c >> 5) * 16 + (c & 15) : c;
    double sums[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        sums[i] = (double)acc[0][i];
#pragma unroll
        for (int s = 1; s < kGroups; ++s) sums[i] = sums[i] * 256.0 + (double)acc[s][i];
    }
    if (xflag & 2) {  // what the rows' digits left out, a row of the block at a time
        const int64_t first = (int64_t)(2 * rt + wr) * kBlk;
        const int count = reinterpret_cast<const int*>(a.ws + a.l.count_off)[first + (lane & 31)];
        const Rest* rests = reinterpret_cast<const Rest*>(a.ws + a.l.rest_off) + first * kRests;
        for (uint32_t left = (uint32_t)__ballot(count > 0); left != 0; left &= left - 1) {
            const int row = __builtin_ctz(left);
            const int n_rest = __builtin_amdgcn_readlane(count, row);
            const Rest mine = rests[row * kRests + (lane & (kRests - 1))];
            double sum = 0.0;
            for (int j0 = 0; j0 < n_rest; j0 += 4) {  // 4 weights a round trip
                float r[4], w[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int at = min(j0 + j, n_rest - 1);
                    const int bits = __builtin_amdgcn_readlane(__builtin_bit_cast(int, mine.r), at);
                    r[j] = j0 + j < n_rest ? __builtin_bit_cast(float, bits) : 0.0f;
                    w[j] = (float)wrow[__builtin_amdgcn_readlane(mine.k, at)];
                }
#pragma unroll
                for (int j = 0; j < 4; ++j) sum += (double)r[j] * (double)(w[j] * 16777216.0f);
            }
#pragma unroll
            for (int i = 0; i < 16; ++i)
                if (8 * (i >> 2) + 4 * (lane >> 5) + (i & 3) == row) sums[i] += sum;
        }
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int row = r0 + 8 * (i >> 2) + (i & 3);
        const float y = (float)(sums[i] * scales[row]);
        const bool ok = row < p.rows && col_ok;
        if constexpr (MODE == kDigitSwiGLU) {
            const float u = __shfl_xor(y, 16);  // lanes 0..15 gate, 16..31 up
            if (ok && !(lane & 16)) p.out[(int64_t)row * p.ldo + n] = y / (1.0f + expf(-y)) * u;
        } else if constexpr (MODE == kDigitResidual) {
            // out may alias resid: each element is read and written by the same lane
            if (ok) p.out[(int64_t)row * p.ldo + n] = p.resid[(int64_t)row * p.ldo + n] + y;
        } else {
            if (ok) p.out[(int64_t)row * p.ldo + n] = y;
        }
    }
}

// Which form a product takes, by what each costs. The lines are fits, in us, to graph replays of
// 18 products at 33 to 8,000 rows: 64 to 50,304 outputs, K of 64 to 16,384, the 120m decoder's
// four among them. W are the weights, 10^9 G the multiply-adds with the rows rounded up to the
// form's tile, out the outputs (gate and up):
//   decode tilings     5 + the longer of 0.0035 K and 52 G (rows to 16), 100 G where every
//                      workgroup normalises its rows again or holds gate and up, up to 16K outputs
//   int8 digits        10, the planes (6 bytes a weight, 10 an activation at 4.5 TB/s), and the
//                      longer of a tile's K, 0.0145 K, and 10 G (rows to 64), and 2.2e-6 out for
//                      the joining of the sums
//   f64 output tiles   3.5 + 0.035 K for each round of workgroups over the CUs + 0.5e-6 out
// What it picks is within 4% of the form each product had by a fixed 128 rows, or faster, and
// within 15% of the best of the three (36% at 33 to 64 rows of 32,000 x 768). Lines without
// the rounding, the planes and the joining, fitted at 768 and 1,024 wide alone, took 125 us for
// 33 rows of 50,304 x 768 (tilings 104, now 80), 172 for 8,000 of 64 x 4,096 (f64 tiles 138, now
// the tilings' 115), 113 for 8,000 of 4,096 x 64 (f64 tiles 100, now those).
struct LinearCost {
    double tiles, digits, gemm;
};
LinearCost linear_cost(int64_t rows, int64_t n_out, int64_t k_in, bool norm, bool swiglu) {
    const double k = (double)k_in, cols = (double)n_out * (swiglu ? 2 : 1);
    const double weights = cols * k, outputs = (double)rows * cols;
    auto g = [&](int64_t tile) { return weights * (double)((rows + tile - 1) / tile * tile) * 1e-9; };
    const bool rows_again = (norm || swiglu) && (swiglu || n_out < kWideOutputs);
    const int64_t cus = device_cu_count(), wg_cols = swiglu ? 64 : 128;
    const int64_t wgs = (n_out + wg_cols - 1) / wg_cols * ((rows + 31) / 32);
    return {5.0 + std::max(0.0035 * k, (rows_again ? 100.0 : 52.0) * g(16)),
            10.0 + 1.33e-6 * weights + 2.2e-6 * (double)rows * k + std::max(0.0145 * k, 10.0 * g(64)) +
                2.2e-6 * outputs,
            3.5 + 0.035 * k * (double)((wgs + cus - 1) / cus) + 0.5e-6 * outputs};
}

// Whether a product takes the digits, given a workspace. Decode-sized batches never do: k_in
// whole stages and within the int32 sums' range; the other bounds keep the grids within 2^31.
bool digit_linear_fits(int64_t rows, int64_t n_out, int64_t k_in, bool norm, bool swiglu) {
    if (k_in <= 0 || k_in % kStageK != 0 || k_in > kMaxK || rows <= 0 || rows > 16 * 65535 ||
        n_out <= 0 || n_out > (1 << 20))
        return false;
    if (const int v = tuning(CRUCIBLE_TUNE_LINEAR_TILE); v > 0) return v == 64;
    if (rows <= kDecodeRows) return false;
    const LinearCost c = linear_cost(rows, n_out, k_in, norm, swiglu);
    return c.digits < c.tiles && c.digits < c.gemm;
}

size_t digit_linear_bytes(int64_t rows, int64_t n_out, int64_t k_in, bool swiglu) {
    return (size_t)make_layout(rows, swiglu ? (n_out + 15) / 16 * 32 : n_out, k_in).bytes;
}

int launch_digit_linear(const DigitLinear& p, int mode, void* workspace, hipStream_t stream,
                        const char* what) {
    const int64_t cols = p.w2 ? (int64_t)(p.n_out + 15) / 16 * 32 : p.n_out;
    DigitArgs a{};
    a.p = p;
    a.ws = static_cast<unsigned char*>(workspace);
    a.l = make_layout(p.rows, cols, p.k_in);
    a.row_wgs = (int)a.l.row_blks * kRowWgs;
    a.row_tiles = (int)a.l.row_blks / 2;
    a.col_tiles = (int)a.l.col_blks / 2;
    a.per_xcd = (int)(((int64_t)a.row_tiles * a.col_tiles + 7) / 8);
    const dim3 digit_grid((unsigned)(a.row_wgs + a.l.col_blks * a.l.parts));
    auto digits = [&](auto norm_tag) {
        constexpr bool kNorm = decltype(norm_tag)::value;
        if (p.k_in <= 1024)
            hipLaunchKernelGGL((digits_kernel<2, kNorm>), digit_grid, dim3(kDigitThreads), 0, stream, a);
        else if (p.k_in <= 2048)
            hipLaunchKernelGGL((digits_kernel<4, kNorm>), digit_grid, dim3(kDigitThreads), 0, stream, a);
        else
            hipLaunchKernelGGL((digits_kernel<0, kNorm>), digit_grid, dim3(kDigitThreads), 0, stream, a);
    };
    if (p.norm_w) digits(std::true_type{});
    else digits(std::false_type{});
    const dim3 grid((unsigned)(8 * a.per_xcd));
    if (mode == kDigitSwiGLU)
        hipLaunchKernelGGL(digits_gemm_kernel<kDigitSwiGLU>, grid, dim3(kDigitGemmThreads), 0, stream, a);
    else if (mode == kDigitResidual)
        hipLaunchKernelGGL(digits_gemm_kernel<kDigitResidual>, grid, dim3(kDigitGemmThreads), 0, stream, a);
    else
        hipLaunchKernelGGL(digits_gemm_kernel<kDigitPlain>, grid, dim3(kDigitGemmThreads), 0, stream, a);
    return fail_launch(what);
}

}  // namespace
}  // namespace crucible
