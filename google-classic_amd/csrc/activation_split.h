// activation_split.h -- the activation halves of the exact batched products
// (prefill_exact.hip, few_rows.hip).
#pragma once

#include "common.h"
#include "block_reduce.h"
#include "exact_blocks.h"

#pragma clang fp contract(off)

namespace holo {

// ---- the activation halves: Ah, Al [M][K] f16, block sums Sx [M][K/32], row scales Rs [M] ----
// One workgroup per row.  The row's values y (x; silu(g) * u as
// cuda_silu_mul computes it, cuda_ops.cu:304-314; or the RMS-normed row,
// rms_norm_rows4_k's arithmetic: thread t sums the squares of float4s
// t + 256 j, the same workgroup reduction, x * scale * w, so the normed
// values are the bits the separate norm writes) are scaled by a power of two
// 2^e chosen from the row's largest magnitude a: a * 2^e lies in
// [2^14, 2^15).  The halves then never overflow f16 (|y| up to fp32's range
// is taken) and the low half is a normal f16 for every value above
// a * 2^-17, so x - xh - xl stays within 2^-22 |x| there and within
// a * 2^-40 below.  The product's store multiplies by Rs = 2^-e (exact).  A
// 32-block is the 8 float4 of 8 adjacent lanes (K % 32 == 0); Sx holds the
// block sums of the scaled values (for the Q4_K min term).
// OPS: the halves in the operand order of few_rows.hip instead, and Sx as
// [rows / 16][block][16]; n_zero counters at `zero` are cleared.  Two halves
// cannot hold a row with infinities (an infinity's low half is a NaN, its
// block sum meets the min term's infinity, its neighbours have no common
// scale), nor, in full, one with a 32-block that lies wholly below a * 2^-17
// (where the low half runs out of f16's exponents): such a row's fp32 values go
// to X32 [M][K], and Rs = -1 tells the product to take it from there.  Small
// blocks count only with `range`: the GEMVs, which few rows would take
// otherwise, scale every block by itself, the other tiles do not.
// PART (with OPS): gridDim.y workgroups share a row: each finds the row's
// scale from all of it and splits and stores float4s part * blockIdx.y ..
// of it (part a multiple of 8 and at most NT), which it loads a second time.
// The row's largest |silu(g) u| comes from the hardware's exp2 and reciprocal
// (off by |g| 2^-23 and a few ulp: under 2^-16 down to g = -87; from -87.3 on
// the reciprocal is subnormal and comes out as zero, where silu goes on to
// -88.7); where that could change the power of two, or some g of the row lies
// below -87, it is found again with expf.
namespace {
template <int CTRL>
__device__ __forceinline__ float max_dpp(float v)
{
    return fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, false)));
}
// Maximum over an aligned lane quad, octet, row of 16 and the wave, in every lane of it.
__device__ __forceinline__ float quad_max(float v) { return max_dpp<0x4E>(max_dpp<0xB1>(v)); }
__device__ __forceinline__ float octet_max(float v) { return max_dpp<0x141>(quad_max(v)); }  // half mirror
__device__ __forceinline__ float row_max(float v) { return max_dpp<0x140>(octet_max(v)); }   // mirror
__device__ __forceinline__ float wave_max(float v)
{
    v = row_max(v);
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
    const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

// Two maxima over a workgroup of 4 or 16 waves, in every thread.  Register
// permutes and one barrier: with block_reduce's lane shuffles for both, 16 rows
// of 11008 x 4096 Q4_0 took 15.6 us instead of 14.9.  A second use of the
// scratch needs a barrier before.
template <int NW>
__device__ __forceinline__ float2 block_max2(float a, float b, float2 *scratch)
{
    static_assert(NW == 4 || NW == 16);
    a = wave_max(a);
    b = wave_max(b);
    if ((threadIdx.x & 63) == 0) scratch[threadIdx.x >> 6] = make_float2(a, b);
    __syncthreads();
    const float2 r = scratch[threadIdx.x & (NW - 1)];
    return NW == 4 ? make_float2(quad_max(r.x), quad_max(r.y)) : make_float2(row_max(r.x), row_max(r.y));
}

enum XSplitMode { XS_PLAIN = 0, XS_SWIGLU = 1, XS_NORM = 2 };

template <int NV, int MODE, int NT = 256, bool OPS = false, bool PART = false>
__global__ __launch_bounds__(NT) void xsplit_row_k(uint2 *__restrict__ Ah, uint2 *__restrict__ Al,
                                                    float *__restrict__ Sx, float *__restrict__ Rs,
                                                    const float *__restrict__ X, const float *__restrict__ U,
                                                    const float *__restrict__ NW, int K, float eps, uint32_t *zero,
                                                    int n_zero, int part, bool range, float *X32)
{
    static_assert(OPS || !PART);
    __shared__ float red[16];
    __shared__ float2 red2[16];
    const int n4 = K >> 2;
    const int64_t r4 = (int64_t)blockIdx.x * n4;
    // every load of the row issued first, through buffer resources over the
    // row (and the norm weights): a float4 past K reads zeros, so no load
    // waits behind a branch or behind another's arithmetic
    const __amdgpu_buffer_rsrc_t rx =
        __builtin_amdgcn_make_buffer_rsrc((void *)((const float4 *)X + r4), (short)0, K * 4, kRawBufWord3);
    const __amdgpu_buffer_rsrc_t ru = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(MODE == XS_SWIGLU ? (const float4 *)U + r4 : (const float4 *)X + r4), (short)0, K * 4, kRawBufWord3);
    const __amdgpu_buffer_rsrc_t rw =
        __builtin_amdgcn_make_buffer_rsrc((void *)(MODE == XS_NORM ? NW : X), (short)0, K * 4, kRawBufWord3);
    float4 v[NV], wv[NV];
#pragma unroll
    for (int j = 0; j < NV; j++) {
        const int o = (int)(threadIdx.x + NT * j) * 16;
        v[j] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(rx, o, 0, 0));
        if constexpr (MODE == XS_SWIGLU)
            wv[j] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(ru, o, 0, 0));
        if constexpr (MODE == XS_NORM)
            wv[j] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(rw, o, 0, 0));
    }
    // PART: this thread's own float4 (past its part: none, zeros)
    const int pi = PART ? (int)(blockIdx.y * part + threadIdx.x) : 0;
    const bool mine = (int)threadIdx.x < part && pi < n4;
    float4 pv, pw;
    if constexpr (PART) {
        const int o = mine ? pi * 16 : K * 4;
        pv = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(rx, o, 0, 0));
        if constexpr (MODE == XS_SWIGLU)
            pw = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(ru, o, 0, 0));
        if constexpr (MODE == XS_NORM)
            pw = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(rw, o, 0, 0));
    }
    float ss = 0.f, gmin = 0.f;
#pragma unroll
    for (int j = 0; j < NV; j++) {
        if constexpr (MODE == XS_SWIGLU && PART) {
            gmin = fminf(gmin, fminf(fminf(v[j].x, v[j].y), fminf(v[j].z, v[j].w)));
            auto sg = [](float g) { return g * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(g * -1.44269504f)); };
            v[j] = make_float4(sg(v[j].x) * wv[j].x, sg(v[j].y) * wv[j].y, sg(v[j].z) * wv[j].z, sg(v[j].w) * wv[j].w);
        } else if constexpr (MODE == XS_SWIGLU) {
            const float4 u = wv[j];
            v[j].x = (v[j].x / (1.0f + expf(-v[j].x))) * u.x;
            v[j].y = (v[j].y / (1.0f + expf(-v[j].y))) * u.y;
            v[j].z = (v[j].z / (1.0f + expf(-v[j].z))) * u.z;
            v[j].w = (v[j].w / (1.0f + expf(-v[j].w))) * u.w;
        }
        if constexpr (MODE == XS_NORM)
            ss += v[j].x * v[j].x + v[j].y * v[j].y + v[j].z * v[j].z + v[j].w * v[j].w;
    }
    float scale = 1.f;
    if constexpr (MODE == XS_NORM) {
        ss = block_reduce<false>(ss, red);
        scale = 1.0f / sqrtf(ss / (float)K + eps);
    }
    // the row's largest magnitude, and the least of its blocks' (zero blocks aside)
    float am = 0.f, lo = INFINITY;
    auto magnitude = [&](const float4 x) {
        const float m = fmaxf(fmaxf(fabsf(x.x), fabsf(x.y)), fmaxf(fabsf(x.z), fabsf(x.w)));
        am = fmaxf(am, m);
        if (OPS && range) {
            const float b = octet_max(m);
            lo = b > 0.f ? fminf(lo, b) : lo;
        }
    };
    auto reduce = [&]() {
        if constexpr (OPS) {
            const float2 r = block_max2<NT / 64>(am, -lo, red2);
            am = r.x;
            lo = -r.y;
        } else {
            am = block_reduce<true>(am, red);
        }
    };
#pragma unroll
    for (int j = 0; j < NV; j++) {
        if constexpr (MODE == XS_NORM) {
            const float4 w4 = wv[j];
            v[j] = make_float4(v[j].x * scale * w4.x, v[j].y * scale * w4.y, v[j].z * scale * w4.z,
                               v[j].w * scale * w4.w);
        }
        magnitude(v[j]);
    }
    if (MODE == XS_SWIGLU && PART && gmin < -87.0f) am = INFINITY;
    reduce();
    if constexpr (MODE == XS_SWIGLU && PART) {
        // within 2^-15 of a power of two, tiny, not finite or a g below -87
        if (((__float_as_uint(am) + 256u) & 0x7FFFFFu) < 512u || am < 1e-30f) {
            am = 0.f;
            lo = INFINITY;
            for (int j = 0; j < NV; j++) {
                const int o = (int)(threadIdx.x + NT * j) * 16;
                const float4 g = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(rx, o, 0, 0));
                const float4 u = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(ru, o, 0, 0));
                magnitude(make_float4((g.x / (1.0f + expf(-g.x))) * u.x, (g.y / (1.0f + expf(-g.y))) * u.y,
                                      (g.z / (1.0f + expf(-g.z))) * u.z, (g.w / (1.0f + expf(-g.w))) * u.w));
            }
            __syncthreads();
            reduce();
        }
    }
    const bool raw = OPS && (am == INFINITY || lo < am * 0x1p-17f);
    // 2^e with a * 2^e in [2^14, 2^15); e = 0 for a zero or non-finite row
    int e = 0;
    if (am > 0.f && am <= 3.4028235e38f) {
        int ea;
        (void)frexpf(am, &ea);  // am = f * 2^ea, f in [0.5, 1)
        e = 15 - ea;
    }
    if (threadIdx.x == 0 && (!PART || blockIdx.y == 0)) Rs[blockIdx.x] = raw ? -1.0f : ldexpf(1.0f, -e);
    if (OPS && blockIdx.x == 0 && (!PART || blockIdx.y == 0))
        for (int j = threadIdx.x; j < n_zero; j += NT) zero[j] = 0;
    if constexpr (PART) {
        if constexpr (MODE == XS_SWIGLU) {
            pv.x = (pv.x / (1.0f + expf(-pv.x))) * pw.x;
            pv.y = (pv.y / (1.0f + expf(-pv.y))) * pw.y;
            pv.z = (pv.z / (1.0f + expf(-pv.z))) * pw.z;
            pv.w = (pv.w / (1.0f + expf(-pv.w))) * pw.w;
        }
        if constexpr (MODE == XS_NORM)
            pv = make_float4(pv.x * scale * pw.x, pv.y * scale * pw.y, pv.z * scale * pw.z, pv.w * scale * pw.w);
    }
#pragma unroll
    for (int j = 0; j < (PART ? 1 : NV); j++) {
        const int i = PART ? pi : (int)threadIdx.x + NT * j;
        const float4 x = PART ? pv : v[j];
        if (!PART && NT * j >= n4) break;  // uniform: no lane of this or a later j is live
        const float y[4] = {ldexpf(x.x, e), ldexpf(x.y, e), ldexpf(x.z, e), ldexpf(x.w, e)};
        _Float16 h[4], l[4];
#pragma unroll
        for (int q = 0; q < 4; q++) {
            h[q] = (_Float16)y[q];
            l[q] = (_Float16)(y[q] - (float)h[q]);
        }
        // the block's sum over its 8 lanes (octets are wholly live or dead)
        float s = (y[0] + y[1]) + (y[2] + y[3]);
        s += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(s), 0xB1, 0xF, 0xF, false));  // [1,0,3,2]
        s += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(s), 0x4E, 0xF, 0xF, false));  // [2,3,0,1]
        s += __shfl_xor(s, 4, 64);
        if constexpr (OPS) {
            // float4 i is block i / 8, weights 4 (i % 8) .. of it: operand lane
            // row + 16 (i % 4), half (i % 8) / 4 of its 16 bytes, order 0, 2, 1, 3.
            // Lanes i and i + 4 trade halves: one stores the high operand's 16
            // bytes, the other the low one's.
            const bool up = (i >> 2) & 1;
            const uint32_t h0 = __builtin_bit_cast(uint32_t, h2{h[0], h[2]}), h1 = __builtin_bit_cast(uint32_t, h2{h[1], h[3]});
            const uint32_t l0 = __builtin_bit_cast(uint32_t, h2{l[0], l[2]}), l1 = __builtin_bit_cast(uint32_t, h2{l[1], l[3]});
            const uint32_t t0 = (uint32_t)__shfl_xor((int)(up ? h0 : l0), 4, 64), t1 = (uint32_t)__shfl_xor((int)(up ? h1 : l1), 4, 64);
            if (PART ? mine : i < n4) {
                const int64_t b = (int64_t)(blockIdx.x >> 4) * (n4 >> 3) + (i >> 3);
                const int m = blockIdx.x & 15;
                if (raw) ((float4 *)X32)[r4 + i] = x;
                ((uint4 *)Ah)[b * 128 + m + 16 * (i & 3) + (up ? 64 : 0)] = up ? make_uint4(t0, t1, l0, l1) : make_uint4(h0, h1, t0, t1);
                if (Sx && (i & 7) == 0) Sx[b * 16 + m] = s;
            }
        } else if (i < n4) {
            Ah[r4 + i] = make_uint2(__builtin_bit_cast(uint32_t, h2{h[0], h[1]}), __builtin_bit_cast(uint32_t, h2{h[2], h[3]}));
            Al[r4 + i] = make_uint2(__builtin_bit_cast(uint32_t, h2{l[0], l[1]}), __builtin_bit_cast(uint32_t, h2{l[2], l[3]}));
            if (Sx && (i & 7) == 0) Sx[r4 / 8 + (i >> 3)] = s;
        }
    }
}

}  // namespace

}  // namespace holo
