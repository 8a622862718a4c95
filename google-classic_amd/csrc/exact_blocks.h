// exact_blocks.h -- what the exact batched products (prefill_exact.hip,
// few_rows.hip) share: the weight kinds of a launch, the vector types, and
// the integers of a block as f16.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace holo {

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));
typedef uint32_t v3u __attribute__((ext_vector_type(3)));

// Weight source of one launch (EW_Q6R: Q6_K repacked for the second tiling).
enum ExactW { EW_Q4_0 = 0, EW_Q8_0 = 1, EW_Q4_K = 2, EW_P16 = 3, EW_F16 = 4, EW_Q6_K = 5, EW_Q6R = 6 };

constexpr int kExactMats = 3;

// ---- integers of a block in f16 ----------------------------------------------------
// v_perm pairs a byte with 0x64, giving the f16 value 1024 + byte; one
// packed f16 add removes the bias, exactly.

__device__ __forceinline__ uint32_t f16_pair(uint32_t bytes, uint32_t sel, _Float16 bias)
{
    const h2 b2 = {bias, bias};
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, bytes, sel)) + b2);
}

// Eight nibbles of x (four bytes): lo[0..1] = low nibbles (k = 4j..4j+3 of the
// block), hi[0..1] = high nibbles (k = 16+4j..), each as f16 (nibble + off).
__device__ __forceinline__ void nibbles_f16(uint32_t x, _Float16 off, uint32_t lo[2], uint32_t hi[2])
{
    const uint32_t t0 = x & 0x0F0F0F0Fu, t1 = (x >> 4) & 0x0F0F0F0Fu;
    const _Float16 bias = (_Float16)(-1024.0f) + off;
    lo[0] = f16_pair(t0, 0x04010400u, bias);
    lo[1] = f16_pair(t0, 0x04030402u, bias);
    hi[0] = f16_pair(t1, 0x04010400u, bias);
    hi[1] = f16_pair(t1, 0x04030402u, bias);
}

// Four signed bytes as f16: byte ^ 0x80 is q + 128 in 0..255.
__device__ __forceinline__ void int8s_f16(uint32_t x, uint32_t out[2])
{
    const uint32_t t = x ^ 0x80808080u;
    out[0] = f16_pair(t, 0x04010400u, (_Float16)-1152.0f);
    out[1] = f16_pair(t, 0x04030402u, (_Float16)-1152.0f);
}

}  // namespace holo
