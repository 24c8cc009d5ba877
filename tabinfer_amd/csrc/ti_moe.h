// ti_moe.h — shared by the int3 expert kernels (k_moe.hip, k_moe_gemm.hip).
#pragma once
#include "ti_internal.h"
#include <type_traits>

// Place of a group's element in the f16 activation rows of k_moe_gemm: slice j = element % 4 holds j, j+16,
// j+8, j+24, j+4, j+20, j+12, j+28, as the weights' words leave q3_nibs and q3_f16.
__device__ __forceinline__ constexpr int moe_slot(int el) {
    const int r = el >> 2;
    return (el & 3) * 8 + (((r & 1) << 2) | (r & 2) | (r >> 2));
}

// A group's (q3 + 4) codes from its bit planes. Elements 4t + r (r = 0..3, t = 0..7) take plane bit
// positions 4t + r; gathering plane b's bits of one r beside each other gives X_r with element
// 4t + r's code in nibble t (for r >= 2 shifted down by 2 first, so that nothing leaves the word).
__device__ __forceinline__ void q3_nibs(uint32_t b0, uint32_t b1, uint32_t b2, uint32_t (&x)[4]) {
    constexpr uint32_t M = 0x11111111u;
    x[0] = (b0 & M) | ((b1 & M) << 1) | ((b2 & M) << 2);
    x[1] = ((b0 & (M << 1)) | ((b1 & (M << 1)) << 1) | ((b2 & (M << 1)) << 2)) >> 1;
    x[2] = ((b0 & (M << 2)) >> 2) | ((b1 & (M << 2)) >> 1) | (b2 & (M << 2));
    x[3] = (((b0 & (M << 3)) >> 2) | ((b1 & (M << 3)) >> 1) | (b2 & (M << 3))) >> 1;
}
// As bytes: q[c] byte i = element 8i + c: nibbles h, h+2, h+4, h+6 of X_r are q[4h + r]. 36 VALU
// operations per 32 codes.
__device__ __forceinline__ void q3_cols(uint32_t b0, uint32_t b1, uint32_t b2, uint32_t (&q)[8]) {
    uint32_t x[4];
    q3_nibs(b0, b1, b2, x);
#pragma unroll
    for (int r = 0; r < 4; r++) {
        q[r] = x[r] & 0x07070707u;
        q[r + 4] = (x[r] >> 4) & 0x07070707u;
    }
}

int ti_moe_gemm_launch(ti_ctx* c, const uint16_t* xh, const float* xs, const uint32_t* p3, const uint16_t* s3,
                       const int32_t* ridx, float* y, int P, int N, int K, int src_div, int nE);
int ti_moe_gateup_launch(ti_ctx* c, const uint16_t* xh, const float* xs, const uint32_t* w1p, const uint16_t* w1s,
                         const uint32_t* w3p, const uint16_t* w3s, const int32_t* ridx, float* gate, float* up, float* act,
                         uint16_t* yh, float* ys, int P, int I, int H, int src_div, int nE);
