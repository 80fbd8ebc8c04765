// MFMA attention for head dimensions that are multiples of 32 other than 64.
//
// The reference kernels take any head_dim (kernels.cu:1741-1756, 2100-2276). The kernels of
// attn_decode.hip and attn_prefill.hip are laid out for 64; attend_generic (generic_attend.hpp)
// takes every multiple of 8 with one query row a workgroup and no matrix instructions. The
// routines here share each K/V byte among 16 query columns (the query heads of a GQA group in
// decode, query rows in prefill) on the same 16x16x32 f16 products, operand layouts and
// arithmetic as the 64-wide kernels: f32 sums, P as fp16 hi + lo, an f32 query as fp16
// hi + lo.
//
// A wave handles a pair of pages (32 keys) at a time:
//   S^T[16 keys x 16 columns] = K . Q^T, HD / 32 products a page (twice for an f32 query);
//     lane (col, grp) is left with keys 4 grp .. +3 of each page
//   one online-softmax update in base 2 for its 8 scores
//   O^T[HD x 16] += V^T . P^T, HD / 16 blocks x (hi, lo); the lane's 8 scores are the k range
//     8 grp .. +7 of the step, its V^T operand the two pages' quarters side by side
// The waves' states then merge through LDS in halving rounds. Infinite or NaN values do not
// survive masks (0 times an infinity is NaN) and hi + lo operands; a row that does not come out
// finite goes through attend_generic again, on its own.
#pragma once

#include "common.hpp"

namespace crucible {

inline bool hd_mfma_ok(int64_t hd) { return hd != kHeadDim && hd % 32 == 0 && hd > 0 && hd <= 256; }

// Waves of a workgroup: 8 while a wave's state and one pair fit 256 registers, else 4.
constexpr int hd_waves(int hd) { return hd <= 160 ? 8 : 4; }

typedef const __attribute__((address_space(4))) int32_t* uniform_i32_ptr;

// The online-softmax state of 16 columns: lane (col, grp) holds dims 16 db + 4 grp + r of
// column col, and the column's m (log2 units) and l.
template <int HD>
struct HdState {
    float4_t o[HD / 16];
    float m, l;

    __device__ __forceinline__ void clear() {
#pragma unroll
        for (int d = 0; d < HD / 16; ++d) o[d] = float4_t{0.f, 0.f, 0.f, 0.f};
        m = -INFINITY;
        l = 0.0f;
    }
    template <class Lds>
    __device__ __forceinline__ void read(const Lds& lds, int slot, int c, int grp) {
#pragma unroll
        for (int i = 0; i < HD / 16; ++i)
            o[i] = *reinterpret_cast<const float4_t*>(&lds.o[slot][c][16 * i + 4 * grp]);
        m = lds.m[slot][c];
        l = lds.l[slot][c];
    }
    // Joins another state. Empty states (m = -inf, l = 0, o = 0) have weight 0.
    __device__ __forceinline__ void merge(const HdState& s) {
        const float mx = fmaxf(m, s.m);
        const float at = mx == -INFINITY ? 0.0f : mx;
        const float wa = fast_exp2(m - at), wb = fast_exp2(s.m - at);
        // written as FMAs: which product of a sum the compiler contracts may differ from one
        // kernel to the next, and the forms give the same bits
        l = __builtin_fmaf(s.l, wb, l * wa);
#pragma unroll
        for (int d = 0; d < HD / 16; ++d)
#pragma unroll
            for (int r = 0; r < 4; ++r) o[d][r] = __builtin_fmaf(s.o[d][r], wb, o[d][r] * wa);
        m = mx;
    }
};

// One column block's queries as B operands: chunk kk holds dims 32 kk + 8 grp .. +7 of column
// col. f32 queries are scaled by a power of two that puts their largest value in [256, 512),
// so that neither half of hi + lo leaves fp16's normal range; `scale` undoes it.
template <int HD, bool F32>
struct HdQuery {
    half8_t hi[HD / 32], lo[F32 ? HD / 32 : 1];
    float scale;  // score -> log2 units

    __device__ __forceinline__ void set(float (&x)[HD / 32][8], float scale_log2) {
        scale = scale_log2;
        float up = 1.0f;
        if constexpr (F32) {
            float mx = 0.0f;
#pragma unroll
            for (int k = 0; k < HD / 32; ++k)
#pragma unroll
                for (int i = 0; i < 8; ++i) mx = fmaxf(mx, fabsf(x[k][i]));
            mx = group_max4(mx);
            // up to the largest f32; smaller than 2^-118, both powers of two would not be normal
            const int e = min(max((int)(__builtin_bit_cast(uint32_t, mx) >> 23) - 127, -118), 127);
            up = __builtin_bit_cast(float, (uint32_t)(8 - e + 127) << 23);
            scale *= __builtin_bit_cast(float, (uint32_t)(e - 8 + 127) << 23);
        }
#pragma unroll
        for (int k = 0; k < HD / 32; ++k)
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float v = x[k][i] * up;
                hi[k][i] = (half_t)v;
                if constexpr (F32) lo[k][i] = (half_t)(v - (float)hi[k][i]);
            }
    }
};

// A pair of pages as operands: K rows (key = col of the page), V^T quarters.
template <int HD>
struct HdPair {
    half8_t k[2][HD / 32];
    half4_t v[2][HD / 16];

    // base0, base1: element offsets of the (page, layer) blocks
    __device__ __forceinline__ void load(const half_t* kp, const half_t* vp, int64_t base0,
                                         int64_t base1, int kv_dim, int head_off, int col, int grp) {
        const int ko = col * kv_dim + head_off + 8 * grp;
        const int vo = (head_off + col) * kPageTokens + 4 * grp;
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            const half_t* kb = kp + (p ? base1 : base0) + ko;
#pragma unroll
            for (int i = 0; i < HD / 32; ++i) k[p][i] = *reinterpret_cast<const half8_t*>(kb + 32 * i);
        }
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            const half_t* vb = vp + (p ? base1 : base0) + vo;
#pragma unroll
            for (int i = 0; i < HD / 16; ++i)
                v[p][i] = *reinterpret_cast<const half4_t*>(vb + 16 * kPageTokens * i);
        }
    }
    // Puts keys at or past astart in place from the chunk's own f32 rows, [row][kv_dim] at row
    // `row0` + key - astart, rounded to fp16 as the append stores them (keys past `last` re-read
    // it; they are masked).
    __device__ __forceinline__ void load_rows(const float* kr, const float* vr, int row0, int astart,
                                              int last, int key0, int kv_dim, int head_off, int col,
                                              int grp) {
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            const int kk = key0 + 16 * p + col;
            if (kk >= astart) {
                const float* src = kr + (int64_t)(row0 + min(kk, last) - astart) * kv_dim + head_off + 8 * grp;
#pragma unroll
                for (int i = 0; i < HD / 32; ++i)
#pragma unroll
                    for (int e = 0; e < 8; ++e) k[p][i][e] = (half_t)src[32 * i + e];
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int vk = key0 + 16 * p + 4 * grp + r;
                if (vk < astart) continue;
                const float* src = vr + (int64_t)(row0 + min(vk, last) - astart) * kv_dim + head_off + col;
#pragma unroll
                for (int i = 0; i < HD / 16; ++i) v[p][i][r] = (half_t)src[16 * i];
            }
        }
    }
    // Slots at or past n_keys may hold anything, NaN included, and 0 * NaN is NaN.
    __device__ __forceinline__ void zero_tail(int key0, int n_keys, int grp) {
#pragma unroll
        for (int p = 0; p < 2; ++p)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (key0 + 16 * p + 4 * grp + r >= n_keys)
#pragma unroll
                    for (int i = 0; i < HD / 16; ++i) v[p][i][r] = (half_t)0.0f;
    }
};

// One pair into a column block's state: the column sees keys up to `last` (-1: none), or the
// whole pair (MASK false). s.l is the lane's own sum until hd_merge_waves.
template <int HD, bool F32, bool MASK = true>
__device__ __forceinline__ void hd_attend_pair(HdState<HD>& s, const HdQuery<HD, F32>& q,
                                               const HdPair<HD>& kv, int key0, int last, int grp) {
    float4_t st[2];
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        st[p] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < HD / 32; ++i) {
            st[p] = mfma_16x16x32(kv.k[p][i], q.hi[i], st[p]);
            if constexpr (F32) st[p] = mfma_16x16x32(kv.k[p][i], q.lo[i], st[p]);
        }
    }
    float mx = -INFINITY;
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            if constexpr (MASK) st[p][r] = key0 + 16 * p + 4 * grp + r <= last ? st[p][r] : -INFINITY;
            mx = fmaxf(mx, st[p][r]);
        }
    const float mn = fmaxf(s.m, group_max4(mx) * q.scale);
    const float at = mn == -INFINITY ? 0.0f : mn;
    const float alpha = fast_exp2(s.m - at);
    s.m = mn;
    u32x4_t hw, lw;
    float sum = 0.0f;
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        float pf[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            // rounded as the largest score was, so the difference is at most 0 (an FMA's is not,
            // and past 2^28 its weight leaves fp16's range)
#pragma clang fp contract(off)
            const float t = st[p][r] * q.scale;
            pf[r] = fast_exp2(t - at);
        }
        sum += (pf[0] + pf[1]) + (pf[2] + pf[3]);
        const uint32_t h01 = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(pf[0], pf[1]));
        const uint32_t h23 = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(pf[2], pf[3]));
        uint32_t l01, l23;
        split_lo4(pf, h01, h23, l01, l23);
        hw[2 * p] = h01;
        hw[2 * p + 1] = h23;
        lw[2 * p] = l01;
        lw[2 * p + 1] = l23;
    }
    s.l = __builtin_fmaf(s.l, alpha, sum);
    const half8_t ph = __builtin_bit_cast(half8_t, hw), pl = __builtin_bit_cast(half8_t, lw);
#pragma unroll
    for (int i = 0; i < HD / 16; ++i) {
        const half8_t va = __builtin_shufflevector(kv.v[0][i], kv.v[1][i], 0, 1, 2, 3, 4, 5, 6, 7);
        s.o[i] = mfma_16x16x32(va, ph, s.o[i] * alpha);
        s.o[i] = mfma_16x16x32(va, pl, s.o[i]);
    }
}

// The merge buffer: states of half the waves, padded so that the 16 columns of a block start in
// different banks.
template <int HD, int W, int QB>
struct HdLds {
    alignas(16) float o[W / 2][QB * 16][HD + 4];
    float m[W / 2][QB * 16], l[W / 2][QB * 16];
};

// Merges the waves' states; wave 0 is left with the whole, in a fixed order. Every wave calls
// it; columns at or past n_cols hold nothing and are skipped.
template <int HD, int W, int QB>
__device__ __forceinline__ void hd_merge_waves(HdLds<HD, W, QB>& lds, HdState<HD> (&s)[QB], int wave,
                                               int col, int grp, int n_cols) {
#pragma unroll
    for (int b = 0; b < QB; ++b) s[b].l = group_sum4(s[b].l);
    #pragma unroll
    for (int h = W / 2; h >= 1; h >>= 1) {
        if (wave >= h && wave < 2 * h) {
#pragma unroll
            for (int b = 0; b < QB; ++b) {
                const int c = 16 * b + col;
                if (c >= n_cols) continue;
#pragma unroll
                for (int i = 0; i < HD / 16; ++i)
                    *reinterpret_cast<float4_t*>(&lds.o[wave - h][c][16 * i + 4 * grp]) = s[b].o[i];
                if (grp == 0) {
                    lds.m[wave - h][c] = s[b].m;
                    lds.l[wave - h][c] = s[b].l;
                }
            }
        }
        __syncthreads();
        if (wave < h) {
#pragma unroll
            for (int b = 0; b < QB; ++b) {
                const int c = 16 * b + col;
                if (c >= n_cols) continue;
                HdState<HD> t;
                t.read(lds, wave, c, grp);
                s[b].merge(t);
            }
        }
        __syncthreads();
    }
}

// The columns, as bits, whose merged state holds an infinity or a NaN (0 times it is not 0).
template <int HD>
__device__ __forceinline__ uint32_t hd_not_finite(const HdState<HD>& s, bool mine) {
    float z = s.l * 0.0f;
#pragma unroll
    for (int i = 0; i < HD / 16; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) z = __builtin_fmaf(s.o[i][r], 0.0f, z);
    const uint64_t bad = __ballot(mine && !(z == 0.0f));
    return (uint32_t)(bad | bad >> 16 | bad >> 32 | bad >> 48) & 0xffffu;
}

// A barrier for LDS alone: __syncthreads would also wait for the outputs' stores on their way.
__device__ __forceinline__ void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// The kernel's first argument read from the argument block where it is used, in a branch that
// hardly runs: its fields would otherwise stay in scalar registers through the main loop.
template <class Args>
__device__ __forceinline__ const Args& cold_args() {
    const void* p = (const void*)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return *static_cast<const Args*>(p);
}

// 8 consecutive values of a query row as f32.
template <bool F32>
__device__ __forceinline__ void hd_load8(const void* q, int64_t off, float (&x)[8]) {
    if constexpr (F32) {
        const float4_t* p = reinterpret_cast<const float4_t*>(static_cast<const float*>(q) + off);
        const float4_t a = p[0], b = p[1];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            x[i] = a[i];
            x[4 + i] = b[i];
        }
    } else {
        const half8_t a = *reinterpret_cast<const half8_t*>(static_cast<const half_t*>(q) + off);
#pragma unroll
        for (int i = 0; i < 8; ++i) x[i] = (float)a[i];
    }
}

template <int HD>
__device__ __forceinline__ void hd_store(void* out, int out_f16, int64_t off, const HdState<HD>& s,
                                         int grp) {
    const float inv = 1.0f / s.l;
#pragma unroll
    for (int i = 0; i < HD / 16; ++i) {
        const float4_t v = s.o[i] * inv;
        const int64_t at = off + 16 * i + 4 * grp;
        if (out_f16)
            *reinterpret_cast<half4_t*>(static_cast<half_t*>(out) + at) =
                half4_t{(half_t)v[0], (half_t)v[1], (half_t)v[2], (half_t)v[3]};
        else
            *reinterpret_cast<float4_t*>(static_cast<float*>(out) + at) = v;
    }
}

}  // namespace crucible
