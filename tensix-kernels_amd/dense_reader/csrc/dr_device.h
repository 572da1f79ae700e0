// dr_device.h: what the library's device sources share: the packed layout's constants, a launch's segment as the kernels
// see it, bf16 conversions, the MFMA, the column scales and the GLU's activation.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "dense_reader.h"
#include "moe.h"

// No contraction of a multiply and an add into an FMA unless the code asks for one: the compiler would otherwise
// decide per kernel instantiation, and a weight would round differently in a block list than alone.
#pragma clang fp contract(off)

namespace drk {

constexpr int KALIGN = 256;  // K padding: one exponent group; a multiple of every format's k-block

constexpr int TILE = 32;    // output columns of a 32 x 32 tile

__host__ __device__ constexpr int kblk(int fmt) {
    return fmt == DR_BFP8 ? 64 : (fmt == DR_BFP4 || fmt == DR_INT4 || fmt == DR_BFP4_KB) ? 128 : 32;
}

__device__ __forceinline__ float bf16_to_f32(uint32_t b) { return __uint_as_float(b << 16); }

// fp32 -> bf16 bits, round to nearest even; a NaN becomes the quiet NaN 0x7FC0
__device__ __forceinline__ uint32_t f32_to_bf16(float f) {
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7FFFFFFFu) > 0x7F800000u) return 0x7FC0u;
    return (u + 0x7FFFu + ((u >> 16) & 1u)) >> 16;
}

struct SegDev {
    const uint8_t* codes;
    const uint8_t* exps;
    const uint8_t* codes_up;
    const uint8_t* exps_up;
    const void* scale;
    const void* scale_up;
    const uint16_t* gscale;  // DR_INT4: the group scales [panel][k-block][4][16] bf16
    int fmt, n, n_pad, glu, scale_f32, col0;
    int n_out, tiles, tile_begin;
    unsigned pstride;  // bytes of codes a panel
};

__device__ __forceinline__ float load_scale(const void* s, int f32, int col) {
    if (s == nullptr) return 1.f;
    return f32 ? reinterpret_cast<const float*>(s)[col] : bf16_to_f32(reinterpret_cast<const uint16_t*>(s)[col]);
}

// the dense GLU's activation: silu(g) = g * sigmoid(g); gelu_tanh(g) = g * sigmoid(1.5957691216 g + 0.0713548162 g^3)
// (dense_ops.h:46-59)
__device__ __forceinline__ float act_glu(float g, int act) {
    const float z = act == DR_ACT_GELU_TANH ? g * (1.5957691216f + 0.0713548162f * (g * g)) : g;
    return g / (1.f + __expf(-z));
}

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;

// two fp32 values with at most 8 significant bits as one bf16 pair (truncation is exact)
__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
    return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u);
}

__device__ __forceinline__ f32x4 mfma(uint4 a, uint4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

}  // namespace drk
