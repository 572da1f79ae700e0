// dense_gemm.h: the matmul of many rows (dense_gemm.hip), as dr_matmul launches it.
#pragma once

#include "dr_device.h"

namespace drk {

constexpr int GEMM_W = 4;  // wavefronts a workgroup, side by side over the columns
constexpr int F32_MT4_K = 4096;

struct GemmArgs {
    const uint16_t* x;
    int m, k, k_pad, ldx;
    void* y;
    int ldy, y_f32;
    const uint16_t* res;
    int ldr, res_mode;
    int act;
    int vec4;    // y's rows take 4 columns in one store (aligned)
    int tiles;   // 32-column output tiles
    int tm, tn;  // row tiles, column tiles
    SegDev seg;
};

// mt: row tiles of 32 a workgroup (2, 4, 6 or 8; for a float32 y 2, or 4 of block-float up to K = F32_MT4_K); ks: the wavefronts split K (mt 2)
hipError_t launch_gemm(const GemmArgs& g, int mt, bool ks, hipStream_t st);

// LDS bytes a workgroup: four stages of x, 64 k of its rows each (ks: one for each wavefront)
constexpr int gemm_lds(int mt, bool ks) { return 4 * 32 * mt * 128 * (ks ? GEMM_W : 1); }

}  // namespace drk
