// Device helpers of the 16-bit matrix-core prefill kernels (kernels_prefill.hip,
// kernels_prefill_wide.hip): LDS DMA, matrix products, packing and the online
// softmax's maxima. HIP device code only.
#pragma once

#include "ckv_internal.h"

namespace ckv {
namespace {

constexpr float log2e = 1.4426950408889634f;

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef short i16x4_t __attribute__((ext_vector_type(4)));

// One 16-byte LDS DMA per lane: lane l's 16 bytes at `src` land at LDS byte
// address lds + 16 * l. Written out rather than through the compiler builtin,
// which makes the compiler wait for every outstanding DMA before any later
// LDS read; here completion is awaited explicitly (vmcnt) before the barrier
// that publishes the data. M0 (the LDS base) is saved and restored around
// the load, with the wait state its write needs before the load reads it.
__device__ __forceinline__ void dma16(const void* src, uint32_t lds)
{
    uint32_t saved;
    asm volatile("s_mov_b32 %0, m0\n\t"
                 "s_mov_b32 m0, %2\n\t"
                 "s_nop 0\n\t"
                 "global_load_lds_dwordx4 %1, off\n\t"
                 "s_mov_b32 m0, %0"
                 : "=&s"(saved)
                 : "v"(src), "s"(__builtin_amdgcn_readfirstlane(lds)));
}

// The same with a scalar 64-bit base and a per-lane 32-bit byte offset: no
// vector address arithmetic.
__device__ __forceinline__ void dma16_s(const void* base, uint32_t voff, uint32_t lds)
{
    uint32_t saved;
    asm volatile("s_mov_b32 %0, m0\n\t"
                 "s_mov_b32 m0, %3\n\t"
                 "s_nop 0\n\t"
                 "global_load_lds_dwordx4 %1, %2\n\t"
                 "s_mov_b32 m0, %0"
                 : "=&s"(saved)
                 : "v"(voff), "s"(base), "s"(__builtin_amdgcn_readfirstlane(lds)));
}

// vmcnt wait (the other counters left alone) that lets `outstanding` of this
// wave's newest DMA loads (a K and a V load per region it stages per block)
// stay in flight.
__device__ __forceinline__ void wait_dma(uint32_t outstanding)
{
    if (outstanding >= 8)
        __builtin_amdgcn_s_waitcnt(0x0F78); // vmcnt(8)
    else if (outstanding >= 4)
        __builtin_amdgcn_s_waitcnt(0x0F74); // vmcnt(4)
    else if (outstanding >= 2)
        __builtin_amdgcn_s_waitcnt(0x0F72); // vmcnt(2)
    else
        __builtin_amdgcn_s_waitcnt(0x0F70); // vmcnt(0)
}

__device__ __forceinline__ const uint8_t* uniform_ptr(const uint8_t* ptr)
{
    const uint64_t v = (uint64_t)(uintptr_t)ptr;
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return (const uint8_t*)(uintptr_t)(((uint64_t)hi << 32) | lo);
}

// LDS row of physical key `key` in a block (an involution: bits 2 and 3 swapped).
__device__ __forceinline__ uint32_t key_row(uint32_t key)
{
    return (key & ~12u) | ((key & 4u) << 1) | ((key & 8u) >> 1);
}

template <bool F16>
__device__ __forceinline__ f32x16_t mfma(uint4 a, uint4 b, f32x16_t c)
{
    if constexpr (F16)
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, a),
                                                      __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                       __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}

// Two floats to a packed 16-bit pair, round to nearest even.
template <bool F16>
__device__ __forceinline__ uint32_t pack2(float lo, float hi)
{
    const f32x2_t v = { lo, hi };
    if constexpr (F16)
        return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, f16x2_t));
    else
        return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t));
}

template <bool F16>
__device__ __forceinline__ float half_value(uint16_t bits)
{
    if constexpr (F16)
        return static_cast<float>(__builtin_bit_cast(_Float16, bits));
    else
        return __builtin_bit_cast(float, static_cast<uint32_t>(bits) << 16);
}

// 1 / (1 + e^-g) in float (src/metal/kernels/tensor_ops.metal:108-124 with sigmoid_only)
__device__ __forceinline__ float sigmoid(float g)
{
    return 1.0f / (1.0f + __builtin_amdgcn_exp2f(-g * log2e));
}

// Growth of the running maximum (log2 units) that forces a rescale. Below it
// the probabilities keep using the older, smaller maximum and may reach
// 2^rescale_log2 (exact in fp32 and in the 16-bit P operand's exponent
// range); the final division by the denominator, accumulated with the same
// maximum, removes the offset exactly. Skipping the rescale of 64 fp32
// accumulators per block matters because on random data some lane of a
// 32-query block sees a new maximum in most key blocks.
constexpr float rescale_log2 = 8.0f;

// Maxima by v_maximum3_f32 (IEEE 754-2019 maximum: a NaN propagates, so the
// scores the matrix core writes need no quieting first, which fmaxf's maxNum
// would make the compiler insert).
__device__ __forceinline__ float max2(float a, float b)
{
    return __builtin_elementwise_maximum(a, b);
}

// The maximum of the 16 scores a lane holds, as a tree of three-input maxima
// (depth 3 instead of a chain of 8). Both lanes of a query compare their own
// maximum with the query's rescale threshold; only a rescale needs the pair's.
__device__ __forceinline__ float lane_max(const f32x16_t& s)
{
    const float a = max2(max2(s[0], s[1]), s[2]), b = max2(max2(s[3], s[4]), s[5]);
    const float d = max2(max2(s[6], s[7]), s[8]), e = max2(max2(s[9], s[10]), s[11]);
    const float f = max2(max2(s[12], s[13]), s[14]);
    return max2(max2(max2(a, b), d), max2(max2(e, f), s[15]));
}

// The maximum of a lane's value and its partner lane's (lane l ^ 32, the same
// query's other 16 keys). The partner is read with v_permlane32_swap, which
// exchanges the two 32-lane halves inside the VALU: of its two results, lanes
// 0-31 find the upper half's value in the second and lanes 32-63 the lower
// half's in the first, while the other result holds the lane's own value, so
// the maximum of all three is the pair's. A ds_bpermute would put an LDS
// round trip on the chain from the scores to the next block's exponentials.
__device__ __forceinline__ float pair_max(float mx)
{
    const uint32_t bits = __builtin_bit_cast(uint32_t, mx);
    const auto sw = __builtin_amdgcn_permlane32_swap(bits, bits, false, false);
    return max2(max2(mx, __builtin_bit_cast(float, (uint32_t)sw[0])),
                __builtin_bit_cast(float, (uint32_t)sw[1]));
}

} // namespace
} // namespace ckv
