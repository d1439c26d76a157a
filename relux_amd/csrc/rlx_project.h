// Device helpers shared by the projection kernels (rlx_project.hip: decode
// sizes; rlx_project_gemm.hip: prefill sizes).
#pragma once
#include "rlx_common.h"

namespace rlx {

// Output layouts (features in packed order, each part a multiple of 16):
//   kProjGQA: q (H heads x D, RoPE)    -> q_out [rows][H][D]
//             k (KVH x D, RoPE)        -> K pages (k-step-major)
//             v (KVH x D)              -> dim-major V pages
//   kProjMLA: q_c (H x D)              -> q_out  [rows][H][D]
//             q_r (H x d_r, RoPE)      -> q_out2 [rows][H][d_r]
//             c^KV (d_c)               -> latent rows [0, d_c)
//             k^R (d_r, RoPE)          -> latent rows [d_c, d_c + d_r)
//   kProjOut:  out (N = features)      -> q_out [rows][N] (+ q_out2, the
//                                         residual, in the same dtype)
constexpr int kProjGQA = 0;
constexpr int kProjMLA = 1;
constexpr int kProjOut = 2;

// Part of packed feature n: output part, feature within it, features per
// RoPE head and rotated dims per head (0, 0: no RoPE).
template <int MODEL>
__device__ __forceinline__ void proj_part(const ProjDims &pd, int n, int &part, int &nn, int &hw, int &tw) {
    part = 0;
    nn = n;
    hw = tw = 0;
    if constexpr (MODEL == kProjGQA) {
        const int NQ = pd.H * pd.DW, NK = pd.KVH * pd.DW;
        part = n < NQ ? 0 : (n < NQ + NK ? 1 : 2);
        nn = n - (part == 0 ? 0 : (part == 1 ? NQ : NQ + NK));
        hw = part < 2 ? pd.DW : 0;  // (features past D: zero weights, no rotation)
        tw = part < 2 ? pd.D : 0;
    } else if constexpr (MODEL == kProjMLA) {
        const int NQC = pd.H * pd.DW, NQR = pd.H * pd.DRP;
        part = n < NQC ? 0 : (n < NQC + NQR ? 1 : (n < NQC + NQR + pd.DCP ? 2 : 3));
        nn = n - (part == 0 ? 0 : (part == 1 ? NQC : (part == 2 ? NQC + NQR : NQC + NQR + pd.DCP)));
        hw = (part == 1 || part == 3) ? pd.DRP : 0;
        tw = hw ? pd.DR : 0;
    }
}

// Activations as MFMA A operands: bf16 pairs {hi, lo} of two f32 values
// (lo = bf16(x - hi), zero where hi is not finite).
__device__ __forceinline__ u32x2 proj_split2(float a, float b) {
    const uint16_t ha = bf16_rne(a), hb = bf16_rne(b);
    const float ra = bf16_f32(ha), rb = bf16_f32(hb);
    const uint16_t la = (fabsf(ra) < INFINITY) ? bf16_rne(a - ra) : (uint16_t)0;
    const uint16_t lb = (fabsf(rb) < INFINITY) ? bf16_rne(b - rb) : (uint16_t)0;
    return u32x2{(uint32_t)ha | ((uint32_t)hb << 16), (uint32_t)la | ((uint32_t)lb << 16)};
}

}  // namespace rlx
