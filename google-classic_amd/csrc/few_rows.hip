// few_rows.hip -- the exact batched product for a few activation rows (a
// short prompt): Y[M][N] = X[M][K] . W[N][K]^T for 3 to kFrMaxRows rows, where
// one GEMV per row streams and unpacks the weights M times, and the 64 x 256
// tiles of prefill_exact.hip leave most of the chip idle.
//
// The reference runs a prompt one token at a time (src/ai/llm.c:1049, matmul_q
// llm.c:770-926).  The arithmetic here is prefill_exact.hip's: activations as
// two f16 halves of a row scaled by a power of two, the blocks' integers exact
// in f16, per 32-block C = sum_k (xh + xl) * w on the f16 matrix cores, then
// acc = fmaf(scale, C, acc) in fp32.  Rows that the halves do not hold
// (infinities; under 64 rows also blocks far below the row's largest value) are
// left as fp32 by the split and multiplied so at the end.
//
// Workgroup: 8 waves and a tile of 16 MT rows by 16 CT columns; each wave
// multiplies the whole tile over its own eighth of K (of the workgroup's part
// of K) and the waves' sums meet in LDS at the end, in wave order.  The main
// loop has no barrier: a wave stages its own weights and reads the activation
// operands, which the split kernel leaves in operand order, from L2.
//
// v_mfma_f32_16x16x32_f16 (wave64): lane (c, g) = (l % 16, l / 16) supplies
// eight k of row (A) or column (B) c; any k, as long as A and B agree.  Lane
// group g takes k = 4g .. 4g + 3 and 16 + 4g .. of a 32-block: one dword of a
// Q4_0 / Q4_K block's nibbles, and of each 16-weight group of Q6_K the four
// that v_mfma_f32_16x16x16_f16 wants.  D: lane (c, g) holds rows 4g .. 4g + 3
// of column c, so a block's scale is one value per lane.
//
// Weights: a unit is 256 weights of each of the tile's columns.  They are
// loaded row by row in 16-byte pieces (a lane reading its own block's window
// straight from memory takes 53 cycles of the CU's address unit per load, a
// run of pieces 16 to 20), put into the wave's LDS stage, and read back as
// block windows: lane (c, g) reads block g of each four blocks, and a 4 x 4
// transpose over the lane groups (v_permlane32_swap, v_permlane16_swap) hands
// every group its dword of all four blocks.
//
// What bounds it (16 x 11008 x 4096 Q4_0, 230 workgroups of 16 x 48): the CU's
// address unit, 61% of a CU's time busy (TA_TA_BUSY over SQ_BUSY_CU_CYCLES),
// mostly with activation operands (4 bytes per value, read once per workgroup),
// beside vector instructions (44%) and products (a quarter), which two waves a
// SIMD do not overlap.  Measured with the split launch, three matrices in turn,
// us, one GEMV per row -> this kernel (Q4_0, 16 rows): 4096 x 4096 67.6 -> 10.8,
// 11008 x 4096 118.9 -> 15.1, 4096 x 11008 118.6 -> 19.9; 64 rows, 64 x 256 tiles
// -> this kernel: 38.8 -> 16.1, 39.9 -> 25.2, 72.9 -> 29.8.
#include "common.h"
#include "quant_blocks.h"
#include "activation_split.h"
#include "exact_blocks.h"
#include "stream_scratch.h"

#include <hip/hip_ext.h>
#include <algorithm>
#include <limits.h>

#include <type_traits>

#pragma clang fp contract(off)

namespace holo {

namespace {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef _Float16 v4h __attribute__((ext_vector_type(4)));
typedef uint32_t v2u __attribute__((ext_vector_type(2)));

struct FrArgs {
    float *Y[kExactMats];
    const uint8_t *W[kExactMats];
    int n[kExactMats];      // columns of each matrix
    int t_end[kExactMats];  // prefix sums of their column tiles; unused entries INT_MAX
    const uint8_t *A;       // activation halves in operand order
    const float *Sx;        // [M/16][nb][16] block sums (Q4_K)
    const float *Rs;        // [M] row scales; -1: the row is in X32 instead
    const float *X32;       // [M][32 nb] fp32 values of such rows
    const float *R;         // one matrix only: Y = R + product (may alias Y)
    float *part;
    uint32_t *cnt;
    int M, nb;
    int items, nrt, ks;     // column tiles x K parts, row tiles, K parts
};

constexpr int kFrWaves = 8;
// Two rows: two GEMVs take 9.3 us at 4096 x 4096, the split and the product
// 11; three rows 13.7 against 11.4.
constexpr int kFrMinRows = 3;
// From 64 rows the estimates choose between this and the 64 x 256 tiles (us
// there against here: 256 x 4096 x 4096 44.6 / 33.1, 192 x 11008 x 4096 74.8 /
// 63.7, 512 x 1024 x 4096 44.3 / 26.3, 256 x 11008 x 4096 72.1 / 77.9), and
// the tiles run where they fill every CU twice (512 x 11008 x 4096 122 / 150, 916
// x 4082 x 2336 Q8_0 72 / 121; the line is a coarse one: 512 x 4096 x 4096, 65.4
// / 58.8, falls on the wrong side of it) or this would take more than three
// rounds of workgroups (764 x 14319 x 1792 Q6_K, eleven rounds: 129 / 202: the
// weights leave the caches between the row tiles), and above this many rows.
constexpr int kFrMaxRows = 1024;
constexpr int64_t kFrMaxParts = 16 << 20;  // bytes of the K parts of a launch
constexpr int kFrMaxCounters = 4096;
constexpr uint32_t kFrOut = 0x80000000u;  // a buffer offset past any range: reads zeros
constexpr int kFrDevScope = 16;

// One step (four 32-weight blocks) of a lane's column, as loaded.
template <int WF>
struct FrRaw;
template <>
struct FrRaw<EW_Q4_0> {
    v4u w;
    uint32_t e;
};
template <>
struct FrRaw<EW_Q8_0> {
    v4u w, v;
    uint32_t e;
};
template <>
struct FrRaw<EW_Q4_K> {
    v4u hd, q;
};
template <>
struct FrRaw<EW_Q6_K> {
    v4u l, m;
    uint32_t le, me;
};
template <>
struct FrRaw<EW_F16> {
    v2u s[8];
};

// A step's operands: block i of the step, this lane's eight weights.
template <int WF>
struct FrOps;
template <>
struct FrOps<EW_Q4_0> {
    uint32_t t[4];
    float sc[4];
};
template <>
struct FrOps<EW_Q8_0> {
    uint32_t t[4], u[4];
    float sc[4];
};
template <>
struct FrOps<EW_Q4_K> {
    uint32_t t[4];
    float sc[4];
    float mneg;
};
template <>
struct FrOps<EW_Q6_K> {
    uint32_t t[4], h[2];
    uint32_t s0, s1;
    float d;
};
template <>
struct FrOps<EW_F16> {
    v2u s[8];
};

__device__ __forceinline__ void swap32(uint32_t &a, uint32_t &b)
{
    const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = r[0];
    b = r[1];
}
__device__ __forceinline__ void swap16(uint32_t &a, uint32_t &b)
{
    const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    a = r[0];
    b = r[1];
}

// Transposes four registers over the four 16-lane groups: register i of
// group g becomes register g of group i.
__device__ __forceinline__ void transpose4(uint32_t (&r)[4])
{
    swap32(r[0], r[2]);
    swap32(r[1], r[3]);
    swap16(r[0], r[1]);
    swap16(r[2], r[3]);
}

// out[i] = x of lane group i, in every group.
__device__ __forceinline__ void spread4(uint32_t x, uint32_t (&out)[4])
{
    uint32_t a = x, b = x;
    swap32(a, b);
    out[0] = out[1] = a;
    out[2] = out[3] = b;
    swap16(out[0], out[1]);
    swap16(out[2], out[3]);
}

__device__ __forceinline__ v4u ld128(__amdgpu_buffer_rsrc_t r, uint32_t vo, uint32_t so)
{
    return __builtin_bit_cast(v4u, __builtin_amdgcn_raw_buffer_load_b128(r, (int)vo, (int)so, 0));
}
__device__ __forceinline__ uint32_t ld32(__amdgpu_buffer_rsrc_t r, uint32_t vo, uint32_t so)
{
    return __builtin_bit_cast(uint32_t, __builtin_amdgcn_raw_buffer_load_b32(r, (int)vo, (int)so, 0));
}
__device__ __forceinline__ v2u ld64(__amdgpu_buffer_rsrc_t r, uint32_t vo, uint32_t so)
{
    return __builtin_bit_cast(v2u, __builtin_amdgcn_raw_buffer_load_b64(r, (int)vo, (int)so, 0));
}

// Eight nibbles of x as f16 (nibble + off): pairs (bytes 0, 2) and (1, 3),
// low nibbles then high.  A nibble in the low mantissa bits of 1024 is 1024 +
// n, four bits further up 1024 + 16 n: one packed add, or one packed fused
// multiply-add by 1/16, leaves n + off exactly.
__device__ __forceinline__ v4u nibbles_02(uint32_t x, _Float16 off)
{
    const uint32_t m = 0x000F000Fu, b = 0x64006400u, y = x >> 8;
    const _Float16 bl = (_Float16)-1024.0f + off, bh = (_Float16)-64.0f + off;
    const h2 vl = {bl, bl}, vh = {bh, bh}, s = {(_Float16)0.0625f, (_Float16)0.0625f};
    auto low = [&](uint32_t q) { return __builtin_bit_cast(uint32_t, __builtin_bit_cast(h2, (q & m) | b) + vl); };
    auto high = [&](uint32_t q) {
        return __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(__builtin_bit_cast(h2, (q & (m << 4)) | b), s, vh));
    };
    return v4u{low(x), low(y), high(x), high(y)};
}
// f16 (byte + bias - 1024) of bytes (0, 2) and (1, 3) of x.
__device__ __forceinline__ void bytes_f16(uint32_t x, _Float16 bias, uint32_t &p02, uint32_t &p13)
{
    p02 = f16_pair(x, 0x04020400u, bias);
    p13 = f16_pair(x, 0x04030401u, bias);
}

// What a unit (256 weights of a row) looks like in LDS: bytes loaded per row
// in 16-byte pieces, and the row stride (its dwords mod 64 spread 16 rows
// over the banks).
template <int WF>
struct FrUnit {
    static constexpr int BYTES = WF == EW_Q8_0 ? 272 : WF == EW_Q6_K ? 210 : 144;
    static constexpr int NP = WF == EW_Q8_0 ? 17 : WF == EW_Q6_K ? 14 : 9;
    static constexpr int STRIDE = WF == EW_Q8_0 ? 272 : WF == EW_Q6_K ? 240 : 144;
    static constexpr int RI = 64 / NP;  // whole rows per load instruction
    static constexpr int loads(int rows) { return (rows + RI - 1) / RI; }
    static constexpr int stage(int rows) { return loads(rows) * RI * STRIDE; }
};

// One step of a lane's column out of the wave's stage (row: the column's row
// in it; e: the unit's step).
template <int WF>
__device__ __forceinline__ FrRaw<WF> fr_stage(const uint8_t *row, uint32_t g, int e)
{
    FrRaw<WF> x;
    typedef const u32x4 *p4;
    typedef const uint32_t *p1;
    if constexpr (WF == EW_Q4_0) {
        const uint8_t *p = row + ((72u * e + 18u * g) & ~3u);
        x.w = *(p4)p;
        x.e = *(p1)(p + 16);
    } else if constexpr (WF == EW_Q8_0) {
        const uint8_t *p = row + ((136u * e + 34u * g) & ~3u);
        x.w = *(p4)p;
        x.v = *(p4)(p + 16);
        x.e = *(p1)(p + 32);
    } else if constexpr (WF == EW_Q4_K) {
        x.hd = *(const v4u *)row;
        x.q = *(const v4u *)(row + 16 + 64 * e + 16 * g);
    } else if constexpr (WF == EW_Q6_K) {
        const uint8_t *pl = row + 64 * e + 16 * g;
        const uint8_t *pm = row + (g < 2 ? 128u + 32u * e + 16u * g : 160u + 16u * g);
        x.l = *(const v4u *)pl;
        x.le = *(p1)(pl + 16);
        x.m = *(const v4u *)pm;
        x.me = *(p1)(pm + 16);
    }
    return x;
}

// One step (blocks 4 s ..) straight from memory: row_o + so the row's byte offset.
template <int WF>
__device__ __forceinline__ FrRaw<WF> fr_fetch(__amdgpu_buffer_rsrc_t r, uint32_t row_o, uint32_t so, uint32_t g, int s)
{
    FrRaw<WF> x;
    if constexpr (WF == EW_Q4_0) {
        const uint32_t vo = (row_o + 18u * g) & ~3u;  // a step is 72 bytes
        x.w = ld128(r, vo, so + 72u * s);
        x.e = ld32(r, vo + 16, so + 72u * s);
    } else if constexpr (WF == EW_Q8_0) {
        const uint32_t vo = (row_o + 34u * g) & ~3u;  // 136
        x.w = ld128(r, vo, so + 136u * s);
        x.v = ld128(r, vo + 16, so + 136u * s);
        x.e = ld32(r, vo + 32, so + 136u * s);
    } else if constexpr (WF == EW_F16) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            x.s[2 * i] = ld64(r, row_o + 8u * g, so + 64u * (uint32_t)(4 * s + i));
            x.s[2 * i + 1] = ld64(r, row_o + 8u * g + 32, so + 64u * (uint32_t)(4 * s + i));
        }
    }
    return x;
}

// ph: the byte phase (0 or 2) of the lane's window within its dwords.
// Blocks past nb get a zero scale (F16: zero weights).
template <int WF>
__device__ __forceinline__ FrOps<WF> fr_ops(const FrRaw<WF> &x, uint32_t ph, uint32_t g, int s, int nb)
{
    FrOps<WF> o;
    uint32_t sb[4];
    if constexpr (WF == EW_Q4_0) {
        const uint32_t sel = realign_sel(ph);
#pragma unroll
        for (int i = 0; i < 4; i++) o.t[i] = perm(i < 3 ? x.w[i + 1] : x.e, x.w[i], sel);
        transpose4(o.t);
        const float d = 4 * s + (int)g < nb ? half_bits_to_float(x.w[0] >> (8 * ph)) : 0.f;
        spread4(__float_as_uint(d), sb);
    } else if constexpr (WF == EW_Q8_0) {
        const uint32_t sel = realign_sel(ph);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            o.t[i] = perm(i < 3 ? x.w[i + 1] : x.v[0], x.w[i], sel);
            o.u[i] = perm(i < 3 ? x.v[i + 1] : x.e, x.v[i], sel);
        }
        transpose4(o.t);
        transpose4(o.u);
        const float d = 4 * s + (int)g < nb ? half_bits_to_float(x.w[0] >> (8 * ph)) : 0.f;
        spread4(__float_as_uint(d), sb);
    } else if constexpr (WF == EW_Q4_K) {
#pragma unroll
        for (int i = 0; i < 4; i++) o.t[i] = x.q[i];
        transpose4(o.t);
        uint32_t sc, mn;
        q4_k_scale_min(x.hd.y, x.hd.z, x.hd.w, 4u * (uint32_t)(s & 1) + g, sc, mn);
        spread4(__float_as_uint(half_bits_to_float(x.hd.x) * (float)sc), sb);
        o.mneg = -(half_bits_to_float(x.hd.x >> 16) * (float)mn);
    } else if constexpr (WF == EW_Q6_K) {
        uint32_t m[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            o.t[i] = __builtin_amdgcn_alignbyte(i < 3 ? x.l[i + 1] : x.le, x.l[i], ph);
            m[i] = __builtin_amdgcn_alignbyte(i < 3 ? x.m[i + 1] : x.me, x.m[i], ph);
        }
        transpose4(o.t);
        // groups 0 and 1 hold the high bits, 2 the scales, 3 starts with d
        spread4(m[0], sb);
        o.d = half_bits_to_float(sb[3]);
        const uint32_t s0 = s & 1 ? m[2] : m[0], s1 = s & 1 ? m[3] : m[1];
        spread4(s0, sb);
        o.s0 = sb[2];
        spread4(s1, sb);
        o.s1 = sb[2];
        transpose4(m);
        o.h[0] = m[0];
        o.h[1] = m[1];
    } else {
#pragma unroll
        for (int i = 0; i < 8; i++) o.s[i] = 4 * s + i / 2 < nb ? x.s[i] : v2u{0u, 0u};
    }
    if constexpr (WF == EW_Q4_0 || WF == EW_Q8_0 || WF == EW_Q4_K)
#pragma unroll
        for (int i = 0; i < 4; i++) o.sc[i] = __uint_as_float(sb[i]);
    return o;
}

// The B operand of block i of the step: lane group g's weights 4g .. 4g + 3
// and 16 + 4g .. of the block, each four in the order 0, 2, 1, 3.
template <int WF>
__device__ __forceinline__ v4u fr_operand(const FrOps<WF> &o, int i)
{
    v4u w;
    if constexpr (WF == EW_Q4_0 || WF == EW_Q4_K) {
        w = nibbles_02(o.t[i], WF == EW_Q4_0 ? (_Float16)-8.0f : (_Float16)0.0f);
    } else if constexpr (WF == EW_Q8_0) {
        uint32_t a, b, c, d;
        bytes_f16(o.t[i] ^ 0x80808080u, (_Float16)-1152.0f, a, b);
        bytes_f16(o.u[i] ^ 0x80808080u, (_Float16)-1152.0f, c, d);
        w = v4u{a, b, c, d};
    } else if constexpr (WF == EW_Q6_K) {
        const int r = 2 * (i & 1);
        uint32_t a, b, c, d;
        bytes_f16(((o.t[r] >> (4 * (i >> 1))) & 0x0F0F0F0Fu) | (((o.h[0] >> (2 * i)) & 0x03030303u) << 4),
                  (_Float16)-1056.0f, a, b);  // 1024 + q - 1056 = q - 32
        bytes_f16(((o.t[r + 1] >> (4 * (i >> 1))) & 0x0F0F0F0Fu) | (((o.h[1] >> (2 * i)) & 0x03030303u) << 4),
                  (_Float16)-1056.0f, c, d);
        w = v4u{a, b, c, d};
    } else {
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const v2u p = o.s[2 * i + h];
            w[2 * h] = perm(p.y, p.x, 0x05040100u);
            w[2 * h + 1] = perm(p.y, p.x, 0x07060302u);
        }
    }
    return w;
}

// Eight f16 weights with infinities (and NaNs) replaced by the largest finite
// values, for the low half: a weight's infinity has the high half's product for
// its sign, and a low half of zero or of the other sign would make it a NaN.
// As integers: positive values in signed order, negative ones in unsigned
// (16 x 11008 x 4096 33.9 -> 34.1 us; float minima 35.2).
__device__ __forceinline__ v4u finite_f16(v4u w)
{
    typedef short s2 __attribute__((ext_vector_type(2)));
    typedef unsigned short us2 __attribute__((ext_vector_type(2)));
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const uint32_t x = w[i];
        const s2 p = __builtin_elementwise_min(__builtin_bit_cast(s2, x), s2{0x7BFF, 0x7BFF});
        w[i] = __builtin_bit_cast(uint32_t, __builtin_elementwise_min(__builtin_bit_cast(us2, p), us2{0xFBFF, 0xFBFF}));
    }
    return w;
}

// Weights 4i .. 4i + 3 of block b of a row, dequantised.
template <int WF>
__device__ __forceinline__ float4 fr_weights(const uint8_t *row, int b, int i)
{
    auto four = [](const uint8_t *p) {  // at a 2-byte-aligned address
        return (uint32_t)((const uint16_t *)p)[0] | (uint32_t)((const uint16_t *)p)[1] << 16;
    };
    uint32_t q;
    float d, off, mn = 0.f;
    if constexpr (WF == EW_Q4_0) {
        const uint8_t *p = row + 18 * (int64_t)b;
        d = half_bits_to_float(*(const uint16_t *)p);
        q = (four(p + 2 + 4 * (i & 3)) >> (i & 4)) & 0x0F0F0F0Fu;
        off = 8.f;
    } else if constexpr (WF == EW_Q8_0) {
        const uint8_t *p = row + 34 * (int64_t)b;
        d = half_bits_to_float(*(const uint16_t *)p);
        q = four(p + 2 + 4 * i) ^ 0x80808080u;
        off = 128.f;
    } else if constexpr (WF == EW_Q4_K) {
        const uint8_t *p = row + 144 * (int64_t)(b >> 3);
        const v4u h = *(const v4u *)p;
        uint32_t sc, m;
        q4_k_scale_min(h.y, h.z, h.w, (uint32_t)b & 7u, sc, m);
        d = half_bits_to_float(h.x) * (float)sc;
        mn = half_bits_to_float(h.x >> 16) * (float)m;
        q = (*(const uint32_t *)(p + 16 + 16 * (b & 7) + 4 * (i & 3)) >> (i & 4)) & 0x0F0F0F0Fu;
        off = 0.f;
    } else if constexpr (WF == EW_Q6_K) {
        const uint8_t *p = row + 210 * (int64_t)(b >> 3);
        const int h = (b >> 2) & 1, j = b & 3;
        d = half_bits_to_float(*(const uint16_t *)(p + 208)) * (float)(int8_t)p[192 + 8 * h + 2 * j + (i >> 2)];
        q = ((four(p + 64 * h + 32 * (j & 1) + 4 * i) >> (4 * (j >> 1))) & 0x0F0F0F0Fu) |
            ((four(p + 128 + 32 * h + 4 * i) >> (2 * j)) & 0x03030303u) << 4;
        off = 32.f;
    } else {
        const v2u w = *(const v2u *)(row + 64 * (int64_t)b + 8 * i);
        return make_float4(half_bits_to_float(w.x), half_bits_to_float(w.x >> 16), half_bits_to_float(w.y),
                           half_bits_to_float(w.y >> 16));
    }
    return make_float4(d * ((float)(q & 255u) - off) - mn, d * ((float)((q >> 8) & 255u) - off) - mn,
                       d * ((float)((q >> 16) & 255u) - off) - mn, d * ((float)(q >> 24) - off) - mn);
}

// fp32 activation rows (those of the four from x on that `rows` has a bit for)
// times a weight row, by a wave: consecutive lanes take consecutive weights,
// every lane gets the sums.
template <int WF>
__device__ __forceinline__ float4 fr_dot4(const uint8_t *row, const float *x, uint32_t rows, int nb, int lane)
{
    const float4 *x4 = (const float4 *)x;
    const int n4 = 8 * nb;
    float s[4] = {0.f, 0.f, 0.f, 0.f};
    for (int k0 = lane; k0 < n4; k0 += 256) {
        float4 w[4], v[4][4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int k = min(k0 + 64 * u, n4 - 1);
            w[u] = fr_weights<WF>(row, k >> 3, k & 7);
#pragma unroll
            for (int r = 0; r < 4; r++)
                if ((rows >> r) & 1u) v[u][r] = x4[(int64_t)r * n4 + k];
        }
#pragma unroll
        for (int u = 0; u < 4; u++)
            if (k0 + 64 * u < n4)
#pragma unroll
                for (int r = 0; r < 4; r++)
                    if ((rows >> r) & 1u)
                        s[r] = fmaf(w[u].w, v[u][r].w, fmaf(w[u].z, v[u][r].z, fmaf(w[u].y, v[u][r].y, fmaf(w[u].x, v[u][r].x, s[r]))));
    }
    return make_float4(wave_reduce_sum(s[0]), wave_reduce_sum(s[1]), wave_reduce_sum(s[2]), wave_reduce_sum(s[3]));
}

__device__ __forceinline__ v4f mfma_k32(v4u a, v4u b, v4f c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, a), __builtin_bit_cast(v8h, b), c, 0, 0, 0);
}
__device__ __forceinline__ v4f mfma_k16(uint32_t a0, uint32_t a1, uint32_t b0, uint32_t b1, v4f c)
{
    return __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(v4h, v2u{a0, a1}),
                                                 __builtin_bit_cast(v4h, v2u{b0, b1}), c, 0, 0, 0);
}

template <int WF, int MT, int CT, bool ST>
__global__ __launch_bounds__(64 * kFrWaves, 1) void gemm_few_k(FrArgs a)
{
    using U = FrUnit<WF>;
    constexpr int T = MT * CT;
    constexpr int GB = MT == 1 ? 4 : MT == 2 ? 2 : 1;  // blocks of activation operands loaded at a time
    constexpr int NG = 4 / GB;
    constexpr bool MIN = WF == EW_Q4_K;  // a min term per block
    constexpr int NI = ST ? U::loads(16 * CT) : 1;  // 16-byte loads per lane and unit
    extern __shared__ __align__(16) uint8_t lds[];
    float4 *red = (float4 *)lds;  // [waves][T][64], after the loop
    __shared__ uint32_t last;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    uint8_t *stage = lds + wave * U::stage(16 * CT);
    const uint32_t g = (uint32_t)lane >> 4, c = (uint32_t)lane & 15u;
    // item = (column tile, K part); the row tiles of one item sit on one XCD
    const int bx = blockIdx.x, q8 = bx >> 3;
    const int item = (q8 / a.nrt) * 8 + (bx & 7), rg = q8 % a.nrt;
    if (item >= a.items) return;
    const int ct0 = item / a.ks, kz = item - ct0 * a.ks;
    const int sel = (ct0 >= a.t_end[0]) + (ct0 >= a.t_end[1]);
    const uint8_t *Wm = sel == 2 ? a.W[2] : sel == 1 ? a.W[1] : a.W[0];
    float *Ym = sel == 2 ? a.Y[2] : sel == 1 ? a.Y[1] : a.Y[0];
    const int Nm = sel == 2 ? a.n[2] : sel == 1 ? a.n[1] : a.n[0];
    const int nl = (ct0 - (sel == 2 ? a.t_end[1] : sel == 1 ? a.t_end[0] : 0)) * 16 * CT, nb = a.nb;
    const uint32_t rowb = WF == EW_Q4_K   ? (uint32_t)(nb >> 3) * 144u
                          : WF == EW_Q6_K ? (uint32_t)(nb >> 3) * 210u
                                          : (uint32_t)nb * (WF == EW_Q4_0 ? 18u : WF == EW_Q8_0 ? 34u : 64u);
    const uint32_t mis = WF == EW_Q6_K ? (uint32_t)((uintptr_t)Wm & 2u) : 0u;
    const uint32_t wbytes = ((uint32_t)Nm * rowb + mis + 3u) & ~3u;
    const int nu = (nb + 7) >> 3;
    const int slices = a.ks * kFrWaves, sl = kz * kFrWaves + wave;
    const int u0 = (int)((int64_t)sl * nu / slices), u1 = (int)((int64_t)(sl + 1) * nu / slices);

    // staged: load i of a unit takes RI whole rows, lane l piece l % NP of row
    // RI i + l / NP (the last lanes repeat the one before them); direct: lane
    // (c, g) the windows of row c.  Rows past the matrix read zeros.
    const int pl = min(lane, U::RI * U::NP - 1), pr = pl / U::NP, pc = pl - pr * U::NP;
    const uint32_t row0 = (uint32_t)(nl + (ST ? pr : (int)c)) * rowb + mis;
    const uint32_t wo = row0 + (ST ? 16u * (uint32_t)pc : 0u);
    uint32_t put = (uint32_t)(pr * U::STRIDE + 16 * pc);  // in the stage
    const uint8_t *const get = stage + c * U::STRIDE;
    // byte phase of the lane's windows (Q6_K: of its column's row, the unit's comes on top)
    const uint32_t phase = WF == EW_Q6_K ? ((uint32_t)(nl + (int)c) * rowb + mis) & 2u
                                         : ((ST ? 0u : row0) + (WF == EW_Q8_0 ? 34u : 18u) * g) & 2u;
    const int rt0 = rg * MT;  // first 16-row tile
    const uint32_t tile_b = (uint32_t)nb * 2048u;
    // rows past M hold whatever the buffer held: their sums are not stored
    const uint32_t va = 16u * (uint32_t)lane, vs = 4u * (16u * g + c);
    const int ntm = (a.M + 15) >> 4;
    const uint32_t abytes = (uint32_t)ntm * tile_b;
    v4u wr[NI];
    FrRaw<WF> raw[2][ST ? 1 : CT];
    auto wrsrc = [&](int u) {
        return __builtin_amdgcn_make_buffer_rsrc((void *)(Wm - mis), (short)0, u < u1 ? (int)wbytes : 0, kRawBufWord3);
    };
    auto fetch_unit = [&](int u) {
        const __amdgpu_buffer_rsrc_t r = wrsrc(u);
        if constexpr (WF == EW_Q6_K) {
            // a row's unit starts 0 or 2 bytes into a dword
            const uint32_t so = (210u * (uint32_t)u) & ~3u, kp = (2u * (uint32_t)u) & 2u;
#pragma unroll
            for (int i = 0; i < NI; i++)
                wr[i] = ld128(r, (wo & ~3u) + ((wo & kp) << 1), so + (uint32_t)(U::RI * i) * rowb);
        } else {
#pragma unroll
            for (int i = 0; i < NI; i++) wr[i] = ld128(r, wo, (uint32_t)u * (uint32_t)U::BYTES + (uint32_t)(U::RI * i) * rowb);
        }
    };
    auto stash_unit = [&]() {
        // what one lane stores others read: with an offset that the compiler does
        // not know it cannot move a read past these stores, nor the next ones past
        // a read (wave_lds_fence, which holds back the loads of the next unit too,
        // makes 16 x 11008 x 4096 take 16.0 us instead of 14.9)
        asm("" : "+v"(put));
#pragma unroll
        for (int i = 0; i < NI; i++) *(v4u *)(stage + put + U::RI * i * U::STRIDE) = wr[i];
    };
    auto fetch_raw = [&](int u, int e) {
        const __amdgpu_buffer_rsrc_t r = wrsrc(u);
#pragma unroll
        for (int j = 0; j < CT; j++) raw[e][j] = fr_fetch<WF>(r, wo, (uint32_t)(16 * j) * rowb, g, 2 * u + e);
    };
    // activation operands of blocks b .. b + GB - 1 (clamped to the row's last block)
    auto load_a = [&](v4u(&x)[GB][MT][2], int b) {
        const __amdgpu_buffer_rsrc_t r =
            __builtin_amdgcn_make_buffer_rsrc((void *)a.A, (short)0, b < 8 * u1 ? (int)abytes : 0, kRawBufWord3);
#pragma unroll
        for (int i = 0; i < GB; i++) {
            const uint32_t so = (uint32_t)rt0 * tile_b + (uint32_t)min(b + i, nb - 1) * 2048u;
#pragma unroll
            for (int m = 0; m < MT; m++) {
                x[i][m][0] = ld128(r, va, so + (uint32_t)m * tile_b);
                x[i][m][1] = ld128(r, va + 1024u, so + (uint32_t)m * tile_b);
            }
        }
    };
    const __amdgpu_buffer_rsrc_t rsx = __builtin_amdgcn_make_buffer_rsrc(
        (void *)a.Sx, (short)0, MIN ? (int)((uint32_t)ntm * (uint32_t)nb * 64u) : 0, kRawBufWord3);
    auto load_sx = [&](float(&x)[MT], int s) {
        if constexpr (MIN)
#pragma unroll
            for (int m = 0; m < MT; m++) x[m] = __uint_as_float(ld32(rsx, vs, (uint32_t)(rt0 + m) * (uint32_t)nb * 64u + (uint32_t)s * 256u));
    };
    v4f acc[MT][CT];
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int j = 0; j < CT; j++) acc[m][j] = v4f{0.f, 0.f, 0.f, 0.f};
    v4u av[2][GB][MT][2];
    float sx[2][MT];

    const float row_scale = a.Rs[min(rt0 * 16 + lane, a.M - 1)];  // here, so that its wait is over at the end
    load_a(av[0], 8 * u0);
    load_sx(sx[0], 2 * u0);
    if constexpr (ST) {
        fetch_unit(u0);
    } else {
        fetch_raw(u0, 0);
        fetch_raw(u0, 1);
    }
    for (int u = u0; u < u1; u++) {
#pragma unroll
        for (int e = 0; e < 2; e++) {
            const int s = 2 * u + e;
            FrOps<WF> o[CT];
#pragma unroll
            for (int gi = 0; gi < NG; gi++) {
                const int cur = (e * NG + gi) & 1;
                load_a(av[cur ^ 1], 4 * s + GB * (gi + 1));
                if (gi == 0) {
                    load_sx(sx[e ^ 1], s + 1);
                    if constexpr (ST) {
                        if (e == 0) {
                            stash_unit();
                            fetch_unit(u + 1);
                        }
                    }
#pragma unroll
                    for (int j = 0; j < CT; j++) {
                        const uint32_t ph = WF == EW_Q6_K ? (phase ^ (2u * (uint32_t)u)) & 2u : phase;
                        if constexpr (ST)
                            o[j] = fr_ops<WF>(fr_stage<WF>(get + 16 * j * U::STRIDE, g, e), ph, g, s, nb);
                        else
                            o[j] = fr_ops<WF>(raw[e][j], ph, g, s, nb);
                    }
                    if constexpr (!ST) fetch_raw(u + 1, e);
                }
#pragma unroll
                for (int i = 0; i < GB; i++) {
                    const int b = gi * GB + i;
#pragma unroll
                    for (int j = 0; j < CT; j++) {
                        const v4u w = fr_operand<WF>(o[j], b);
                        v4u wl = w;
                        if constexpr (WF == EW_F16) wl = finite_f16(w);
#pragma unroll
                        for (int m = 0; m < MT; m++) {
                            const v4u ah = av[cur][i][m][0], al = av[cur][i][m][1];
                            const v4f zero = {0.f, 0.f, 0.f, 0.f};
                            if constexpr (WF == EW_F16) {
                                // a block's two products summed first: all in one chain of products on
                                // acc, 16 x 4096 x 14336 was off by 3.9e-7 (2-norm), a GEMV a row is by
                                // 2.8e-7, this by 1.3e-7
                                acc[m][j] += mfma_k32(ah, w, zero) + mfma_k32(al, wl, zero);
                            } else if constexpr (WF == EW_Q6_K) {
                                const uint32_t sc = ((b & 2) ? o[j].s1 : o[j].s0) >> (16 * (b & 1));
                                const float sc0 = o[j].d * (float)(int8_t)(sc & 0xFFu);
                                const float sc1 = o[j].d * (float)(int8_t)((sc >> 8) & 0xFFu);
                                v4f d = mfma_k16(al[0], al[1], w[0], w[1], mfma_k16(ah[0], ah[1], w[0], w[1], zero));
#pragma unroll
                                for (int r = 0; r < 4; r++) acc[m][j][r] = __builtin_fmaf(sc0, d[r], acc[m][j][r]);
                                d = mfma_k16(al[2], al[3], w[2], w[3], mfma_k16(ah[2], ah[3], w[2], w[3], zero));
#pragma unroll
                                for (int r = 0; r < 4; r++) acc[m][j][r] = __builtin_fmaf(sc1, d[r], acc[m][j][r]);
                            } else {
                                const v4f d = mfma_k32(al, w, mfma_k32(ah, w, zero));
#pragma unroll
                                for (int r = 0; r < 4; r++)
                                    acc[m][j][r] = __builtin_fmaf(o[j].sc[b], d[r], acc[m][j][r]);
                            }
                        }
                        // this block's products are folded in here, and the next operands not
                        // built before: left alone, the compiler keeps a step's products in
                        // registers until its end
                        if constexpr (MT * CT >= 4) {
#pragma unroll
                            for (int m = 0; m < MT; m++) asm volatile("" : "+v"(acc[m][j]));
                            __builtin_amdgcn_sched_barrier(0);
                        }
                    }
                }
            }
            if constexpr (MIN) {
                // the step's four blocks: A[m][b] = sum of x over block b, B[b][n] = -dmin m
#pragma unroll
                for (int m = 0; m < MT; m++)
#pragma unroll
                    for (int j = 0; j < CT; j++)
                        acc[m][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(sx[e][m], o[j].mneg, acc[m][j], 0, 0, 0);
            }
        }
    }
    // the workgroup's rows whose fp32 values were left: bit i, row i
    const uint64_t whole = __ballot(lane < 16 * MT && rt0 * 16 + lane < a.M && row_scale < 0.f);
    if constexpr (ST) __syncthreads();  // the sums' buffer lies over the stages

    // the waves' sums, in wave order
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int j = 0; j < CT; j++)
            red[(wave * T + m * CT + j) * 64 + lane] = __builtin_bit_cast(float4, acc[m][j]);
    __syncthreads();
    constexpr int TW = (T + kFrWaves - 1) / kFrWaves;  // tiles a wave finishes
    v4f v[TW];
#pragma unroll
    for (int i = 0; i < TW; i++) {
        const int t = wave + kFrWaves * i;
        if (t < T) {
            v[i] = __builtin_bit_cast(v4f, red[t * 64 + lane]);
#pragma unroll
            for (int w = 1; w < kFrWaves; w++) v[i] += __builtin_bit_cast(v4f, red[(w * T + t) * 64 + lane]);
        }
    }
    if (a.ks > 1) {
        const int grp = ct0 * a.nrt + rg;
        const __amdgpu_buffer_rsrc_t rp = __builtin_amdgcn_make_buffer_rsrc(
            (void *)a.part, (short)0, (int)((uint32_t)(a.items * a.nrt) * (uint32_t)T * 1024u), kRawBufWord3);
        auto word = [&](int z, int t) {
            return (uint32_t)((grp * a.ks + z) * T + t) * 1024u + 16u * (uint32_t)lane;
        };
#pragma unroll
        for (int i = 0; i < TW; i++) {
            const int t = wave + kFrWaves * i;
            if (t < T)
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4u, v[i]), rp, (int)word(kz, t), 0,
                                                       kFrDevScope);
        }
        __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the stores have completed (device scope)
        __syncthreads();
        if (tid == 0) {
            const uint32_t old = __hip_atomic_fetch_add(a.cnt + grp, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            last = old == (uint32_t)(a.ks - 1);
        }
        __syncthreads();
        if (!last) return;
        if (tid == 0) __hip_atomic_store(a.cnt + grp, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
        for (int i = 0; i < TW; i++) {
            const int t = wave + kFrWaves * i;
            if (t >= T) continue;
            v4f sum = {0.f, 0.f, 0.f, 0.f};
            for (int z0 = 0; z0 < a.ks; z0 += 4) {
                v4u pv[4];
#pragma unroll
                for (int z = 0; z < 4; z++)
                    pv[z] = __builtin_bit_cast(v4u, __builtin_amdgcn_raw_buffer_load_b128(
                                                        rp, z0 + z < a.ks ? (int)word(z0 + z, t) : (int)kFrOut, 0,
                                                        kFrDevScope));
#pragma unroll
                for (int z = 0; z < 4; z++) sum += __builtin_bit_cast(v4f, pv[z]);
            }
            v[i] = sum;
        }
    }
#pragma unroll
    for (int i = 0; i < TW; i++) {
        const int t = wave + kFrWaves * i;
        if (t >= T) continue;
        const int m0 = (rt0 + t / CT) * 16 + 4 * (int)g, n = nl + 16 * (t % CT) + (int)c;
        float rs[4], rv[4];
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int m = min(m0 + r, a.M - 1);
            rs[r] = a.Rs[m];
            rv[r] = a.R ? a.R[(int64_t)m * Nm + min(n, Nm - 1)] : 0.f;
        }
#pragma unroll
        for (int r = 0; r < 4; r++)
            if (m0 + r < a.M && n < Nm && !(rs[r] < 0.f)) {
                const float y = v[i][r] * rs[r];  // a power of two: exact
                Ym[(int64_t)(m0 + r) * Nm + n] = a.R ? rv[r] + y : y;
            }
    }
    // rows that the halves do not hold: fp32 products, each wave columns of its
    // own, four rows at a time (16 x 11008 x 4096 Q4_0 with 0, 1 and 16 such rows
    // 14.2, 38.6 and 139 us; a GEMV per row 114; the values read back from operand
    // order, in 16-byte pieces, 105 and 370)
    for (int q = 0; whole != 0 && q < 4 * MT; q++) {
        const uint32_t rows = (uint32_t)(whole >> (4 * q)) & 15u;
        if (rows == 0) continue;
        for (int c16 = wave; c16 < 16 * CT && nl + c16 < Nm; c16 += kFrWaves) {
            const int m = rt0 * 16 + 4 * q;
            const float4 y = fr_dot4<WF>(Wm + (int64_t)(nl + c16) * rowb, a.X32 + (int64_t)m * 32 * nb, rows, nb, lane);
            const int64_t at = (int64_t)(m + lane) * Nm + nl + c16;
            if (lane < 4 && (rows >> lane) & 1u) {
                const float v1 = lane == 0 ? y.x : lane == 1 ? y.y : lane == 2 ? y.z : y.w;
                Ym[at] = a.R ? a.R[at] + v1 : v1;
            }
        }
    }
}

// ---- host side ---------------------------------------------------------------------

// The tile of a launch: MT 16-row and CT 16-column tiles per workgroup, the K
// units dealt to the waves of KS workgroups.
struct FrPlan {
    int mt, ct, ks, nct, nrt, rounds;
    float us;  // the estimate
};

// Column tiles of a workgroup before its registers spill (four of F16: 128 to
// 216 bytes a lane; three of 64 rows, 92 bytes, still the fastest at 48 x 11008
// x 4096: 50.6 us, two 56.4).
constexpr int few_max_ct(int kind, int mt) { return kind == EW_F16 || (kind == EW_Q8_0 && mt == 4) ? 3 : 4; }

// Picks the plan with the least estimated time, fitted to a sweep of mt, ct
// and ks over 30 shapes of all types, 16 to 400 rows, out 500 to 14336, in
// 1024 to 14336 (the picks there are within 3% of the best plan).  In us: per
// unit of a workgroup's longest wave 0.75 per row tile (every wave reads its
// own activations), 0.73 per column tile (its loads and unpacking) and 0.32
// per product tile; a round of workgroups over the CUs 0.75, a second part of
// K its exchange, 3.2; and at least the activation operands of all workgroups
// out of L2, 22.5 TB/s.  Above 32 rows 64-row tiles: more, narrower row tiles
// read the weights again (64 x 11008 x 4096: 25.2 against 30.8).  At 16 rows
// of 11008 x 4096: 48 columns and one round 15.1, 32 columns 17.4, 64 columns
// 17.9, 16 columns 19.2.
FrPlan few_plan(int kind, const int *N, int nmat, int M, int nb)
{
    FrPlan best = {};
    const int nu = (nb + 7) / 8;
    // F16: 3.6 times Q4_0's bytes, in 8-byte pieces (192 x 4096 x 11008 132 us, Q4_0 66)
    const float type = kind == EW_Q8_0 ? 1.15f : kind == EW_Q6_K ? 1.39f : kind == EW_Q4_K ? 1.09f : kind == EW_F16 ? 2.f : 1.f;
    for (int mt = 1; mt <= 4; mt *= 2) {
        if (mt > 1 && 16 * mt >= 2 * M) break;
        if (mt < 4 && M > 32) continue;
        for (int ct = 1; ct <= few_max_ct(kind, mt); ct++) {
            int nct = 0;
            for (int i = 0; i < nmat; i++) nct += (N[i] + 16 * ct - 1) / (16 * ct);
            const int nrt = (M + 16 * mt - 1) / (16 * mt);
            for (int ks = 1; ks <= 4; ks++) {
                if (ks > 1 && ((int64_t)nct * nrt * ks * mt * ct * 1024 > kFrMaxParts || nct * nrt > kFrMaxCounters ||
                               nu < kFrWaves * ks))
                    break;
                const int units = (nu + kFrWaves * ks - 1) / (kFrWaves * ks);
                const int rounds = (nct * nrt * ks + num_cus() - 1) / num_cus();
                float us = (float)rounds * (0.75f + type * (float)units * (0.73f * ct + 0.75f * mt + 0.32f * ct * mt)) +
                           (ks > 1 ? 3.2f : 0.f);
                us = std::max(us, (float)((int64_t)nct * ((M + 15) / 16) * nb * 2048) * (1.f / 22.5e6f));
                if (best.mt == 0 || us < best.us) best = {mt, ct, ks, nct, nrt, rounds, us};
            }
        }
    }
    return best;
}

template <int WF, int MT, int CT, bool ST>
void launch_few(const FrArgs &a)
{
    constexpr size_t RED = (size_t)kFrWaves * MT * CT * 1024;
    constexpr size_t STG = ST ? (size_t)kFrWaves * FrUnit<WF>::stage(16 * CT) : 0;
    constexpr size_t LDS = RED > STG ? RED : STG;
    auto kern = gemm_few_k<WF, MT, CT, ST>;
    static const hipError_t attr =
        hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)LDS);
    if (attr != hipSuccess) {
        HOLO_CHECK(attr);
        return;
    }
    const int grid = (a.items + 7) / 8 * 8 * a.nrt;
    launch_timed(kern, dim3((unsigned)grid), dim3(64 * kFrWaves), LDS, a);
    HOLO_LAUNCH_CHECK();
}

template <int WF, int MT, int CT>
void launch_few_st(const FrArgs &a)
{
    if constexpr (WF == EW_F16) launch_few<WF, MT, CT, false>(a);
    else if constexpr (WF == EW_Q4_K || WF == EW_Q6_K) launch_few<WF, MT, CT, true>(a);
    else if (a.nb % 8 == 0) launch_few<WF, MT, CT, true>(a);
    else launch_few<WF, MT, CT, false>(a);
}
template <int WF, int MT>
void launch_few_ct(const FrArgs &a, int ct)
{
    constexpr int M = few_max_ct(WF, MT);
    if (ct == 1) launch_few_st<WF, MT, 1>(a);
    else if (ct == 2) launch_few_st<WF, MT, 2>(a);
    else if (ct == 3) launch_few_st<WF, MT, M < 3 ? M : 3>(a);
    else launch_few_st<WF, MT, M < 4 ? M : 4>(a);
}
template <int WF>
void launch_few_mt(const FrArgs &a, const FrPlan &p)
{
    if (p.mt == 1) launch_few_ct<WF, 1>(a, p.ct);
    else if (p.mt == 2) launch_few_ct<WF, 2>(a, p.ct);
    else launch_few_ct<WF, 4>(a, p.ct);
}

int few_kind(int type)
{
    switch (type) {
    case HOLO_TYPE_Q4_0: return EW_Q4_0;
    case HOLO_TYPE_Q8_0: return EW_Q8_0;
    case HOLO_TYPE_Q4_K: return EW_Q4_K;
    case HOLO_TYPE_Q6_K: return EW_Q6_K;
    case HOLO_TYPE_F16: return EW_F16;
    default: return -1;
    }
}

}  // namespace

bool few_rows_take(int M) { return M >= kFrMinRows && gemv_default_mode(); }

namespace {

// What a call runs: one launch per weight kind, over that kind's matrices in
// order, and the scratch they share (the launches run one after the other).
struct FrLaunch {
    FrPlan p;
    int kind, n, mat[kExactMats];
};
struct FrChoice {
    FrLaunch l[kExactMats];
    int nl, counters;
    size_t parts;
    bool need_sx;
};

// Whether the few-row tiles take a call, and their plan.  prepared[i]: a
// repacked copy of matrix i is registered.
bool few_choose(const int *types, const int *N, const bool *prepared, int nmat, int M, int K, FrChoice &c)
{
    if (M > kFrMaxRows) return false;
    const int nb = K / 32;
    int kinds[kExactMats];
    c.nl = c.counters = 0;
    c.parts = 0;
    c.need_sx = false;
    for (int i = 0; i < nmat; i++) {
        kinds[i] = few_kind(types[i]);
        if (kinds[i] < 0 || N[i] <= 0) return false;
        // a GEMV per row: its sums of a short row round less (K = 512: 8.5e-8
        // normwise, here 9.2e-8; 1024: 1.0e-7 and 9.6e-8)
        if (kinds[i] == EW_F16 && M < 64 && nb < 32) return false;
        c.need_sx = c.need_sx || kinds[i] == EW_Q4_K;
        // 32-bit byte offsets into a matrix
        const int64_t rowb = kinds[i] == EW_Q4_K   ? (int64_t)(nb / 8) * 144
                             : kinds[i] == EW_Q6_K ? (int64_t)(nb / 8) * 210
                                                   : (int64_t)nb * (kinds[i] == EW_Q4_0 ? 18 : kinds[i] == EW_Q8_0 ? 34 : 64);
        if ((N[i] + 128) * rowb >= (1LL << 31)) return false;
    }
    bool many = false;
    float here = 7.6f, tiled = 0.f;  // estimates, us (7.6: the split and two launches)
    bool done[kExactMats] = {false, false, false};
    for (int i = 0; i < nmat; i++) {
        if (done[i]) continue;
        FrLaunch &l = c.l[c.nl++];
        l.kind = kinds[i];
        l.n = 0;
        int n[kExactMats], columns = 0;
        bool copies = true;
        for (int j = i; j < nmat; j++) {
            if (done[j] || kinds[j] != kinds[i]) continue;
            done[j] = true;
            columns += N[j];
            copies = copies && prepared[j];
            n[l.n] = N[j];
            l.mat[l.n++] = j;
        }
        l.p = few_plan(kinds[i], n, l.n, M, nb);
        here += l.p.us;
        many = many || l.p.rounds > 3;
        bool full;
        tiled += exact_tiles_us(types[i], columns, M, nb, copies, &full);
        many = many || full;
        if (l.p.ks > 1) {
            c.parts = std::max(c.parts, (size_t)l.p.nct * l.p.nrt * l.p.ks * l.p.mt * l.p.ct * 1024);
            c.counters = std::max(c.counters, l.p.nct * l.p.nrt);
        }
    }
    // From 64 rows on, the other tiling where it is estimated 6% better (both
    // sides measured on 70 shapes: the taken one is the faster or within 5% for
    // all that are not `full`): 192 x 11008 x 4096 Q4_0 here 63.7 us, there 74.8;
    // 231 x 6825 x 5632 Q6_K 92.6 and 88.1; 1015 x 890 x 4864 Q8_0 70.8 and 58.4.
    return M < 64 || !(many || tiled <= 0.94f * here);
}

}  // namespace

bool few_rows_product(float *const *Y, const void *const *W, const int *types, const int *N, int nmat, const float *X,
                      const float *U, const float *R, int M, int K, const float *NW, float eps)
{
    FrChoice c;
    bool prepared[kExactMats] = {false, false, false};
    for (int i = 0; i < nmat; i++) {
        if (!Y[i]) return false;
        prepared[i] = M >= 64 && types[i] == HOLO_TYPE_Q6_K && q6_prepared(W[i], N[i], K);
    }
    if (!few_choose(types, N, prepared, nmat, M, K, c)) return false;
    const int nb = K / 32, counters = c.counters;
    const size_t parts = c.parts;
    const int ntm = (M + 15) / 16;
    auto up = [](size_t b) { return (b + 255) & ~(size_t)255; };
    const size_t ob = up((size_t)ntm * nb * 2048), sb = c.need_sx ? up((size_t)ntm * nb * 64) : 0, rb = up((size_t)M * 4),
                 cb = up((size_t)counters * 4);
    const size_t xb = up((size_t)M * K * 4);
    const size_t total = ob + sb + rb + cb + xb + parts;
    const StreamScratch scratch(total);
    uint8_t *ws = (uint8_t *)scratch.get();
    if (!ws) return false;
    uint8_t *A = ws;
    float *Sx = c.need_sx ? (float *)(ws + ob) : nullptr, *Rs = (float *)(ws + ob + sb);
    uint32_t *cnt = (uint32_t *)(ws + ob + sb + rb);
    float *X32 = (float *)(ws + ob + sb + rb + cb);
    // Few rows leave most CUs idle: four workgroups a row (each of at most
    // `most` float4s) while they fit the CUs.  23 rows, alone -> four -> eight:
    // SwiGLU 11008 wide 8.6 -> 6.6 -> 7.5 us, the norm 4096 wide 5.0 -> 4.6 ->
    // 4.5, plain 4.9 -> 4.4 -> 4.3.
    int shares = 1, part = 0;
    auto share = [&](int most) {
        const int n4 = K >> 2, need = (n4 + most - 1) / most;
        shares = std::max(need, std::min(4, num_cus() / M));
        if (shares * M > num_cus()) shares = 1;
        part = ((n4 + shares - 1) / shares + 7) & ~7;
        return shares > 1;
    };
    auto split = [&](auto kern, int nt) {
        hipLaunchKernelGGL(kern, dim3(M, shares), dim3(nt), 0, stream(), (uint2 *)A, (uint2 *)nullptr, Sx, Rs, X, U, NW, K,
                           eps, cnt, counters, part, M < 64, X32);
    };
    const bool small = K <= 4096;
    // the normed form keeps rms_norm_rows4_k's 256 threads and summation order
    if (NW && share(256))
        small ? split(xsplit_row_k<4, XS_NORM, 256, true, true>, 256) : split(xsplit_row_k<16, XS_NORM, 256, true, true>, 256);
    else if (NW) small ? split(xsplit_row_k<4, XS_NORM, 256, true>, 256) : split(xsplit_row_k<16, XS_NORM, 256, true>, 256);
    else if (U && share(1024))
        small ? split(xsplit_row_k<1, XS_SWIGLU, 1024, true, true>, 1024) : split(xsplit_row_k<4, XS_SWIGLU, 1024, true, true>, 1024);
    else if (U) small ? split(xsplit_row_k<1, XS_SWIGLU, 1024, true>, 1024) : split(xsplit_row_k<4, XS_SWIGLU, 1024, true>, 1024);
    else if (share(1024))
        small ? split(xsplit_row_k<1, XS_PLAIN, 1024, true, true>, 1024) : split(xsplit_row_k<4, XS_PLAIN, 1024, true, true>, 1024);
    else small ? split(xsplit_row_k<1, XS_PLAIN, 1024, true>, 1024) : split(xsplit_row_k<4, XS_PLAIN, 1024, true>, 1024);
    HOLO_LAUNCH_CHECK();
    for (int i = 0; i < c.nl; i++) {
        const FrLaunch &l = c.l[i];
        const FrPlan &p = l.p;
        FrArgs a = {};
        int tiles = 0;
        for (int j = 0; j < kExactMats; j++) {
            if (j < l.n) {
                a.Y[j] = Y[l.mat[j]];
                a.W[j] = (const uint8_t *)W[l.mat[j]];
                a.n[j] = N[l.mat[j]];
                tiles += (a.n[j] + 16 * p.ct - 1) / (16 * p.ct);
            }
            a.t_end[j] = j < l.n ? tiles : INT_MAX;
        }
        a.A = A;
        a.Sx = Sx;
        a.Rs = Rs;
        a.R = nmat == 1 ? R : nullptr;
        a.X32 = X32;
        a.part = (float *)(ws + ob + sb + rb + cb + xb);
        a.cnt = cnt;
        a.M = M;
        a.nb = nb;
        a.items = p.nct * p.ks;
        a.nrt = p.nrt;
        a.ks = p.ks;
        switch (l.kind) {
        case EW_Q4_0: launch_few_mt<EW_Q4_0>(a, p); break;
        case EW_Q8_0: launch_few_mt<EW_Q8_0>(a, p); break;
        case EW_Q4_K: launch_few_mt<EW_Q4_K>(a, p); break;
        case EW_Q6_K: launch_few_mt<EW_Q6_K>(a, p); break;
        default: launch_few_mt<EW_F16>(a, p); break;
        }
    }
    return true;
}

}  // namespace holo

extern "C" int holo_few_rows_plan(int type, int M, int N, int K, int prepared, int *plan)
{
    holo::FrChoice c;
    const bool copy = prepared != 0;
    if (!plan || M < holo::kFrMinRows || !holo::exact_ok(type, K, nullptr) || !holo::few_choose(&type, &N, &copy, 1, M, K, c)) return 0;
    const int kind = c.l[0].kind;
    plan[0] = c.l[0].p.mt;
    plan[1] = c.l[0].p.ct;
    plan[2] = c.l[0].p.ks;
    plan[3] = kind == holo::EW_Q4_K || kind == holo::EW_Q6_K || (kind != holo::EW_F16 && K % 256 == 0);
    return 1;
}
