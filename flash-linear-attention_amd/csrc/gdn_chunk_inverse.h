// The inverse of a 64 x 64 unit lower triangular matrix by one wave, in fp32, transposed: shared by the chunk-parallel kernels of the
// forward (gdn_chunk_prepare.hip) and of the backward pass (gdn_chunk_bwd_prepare.h).
//
// Everything is kept TRANSPOSED: U = L^T is strictly upper triangular, T = X^T = (I + U)^-1.  A tile in accumulator layout (lane
// (c16, g): rows 4g..4g+3, column c16) serves directly as the RIGHT factor of a product on the fp32 matrix cores (step e contracts over
// the indices {4g + e}), the left factor comes from LDS by rows, and the result is again in accumulator layout.
//   * Diagonal 16x16 blocks: lane group g inverts block g by substitution, one row of X per lane (all 64 lanes busy).
//   * Merges: T(lo,hi) = -(T(lo,lo) U(lo,hi)) T(hi,hi) on 16-tiles, then on 32-blocks with the zero tiles left out: the gated
//     tiles U are right factors and never leave the registers, only the products T U pass through LDS.
#pragma once
#include "gdn_chunk_common.h"

namespace gdn {

// LDS per wave: seven 16x16 fp32 tiles that serve as left factors.  The caller leaves the diagonal blocks of L, by rows ([4][16 i][16 j]),
// in the first 1024 floats; the room behind them is free until the call.
constexpr int TP = 20;                                       // pitch (floats) of a 16x16 fp32 tile in LDS
constexpr int PW_FLOATS = 7 * 16 * TP;                       // 2240 floats per wave

// U[a][b], a < b: rows of tile a, columns of tile b.  X[a][b], a <= b: the same places of T.
__device__ __forceinline__ void inverse_transposed(float* tiles, const f32x4 (&U)[4][4], f32x4 (&X)[4][4], int c16, int g) {
    // left factors: the transposed diagonal blocks T(0,0) .. T(3,3) and the intermediate products V = T U
    constexpr int I_T00 = 0, I_T11 = 1, I_T22 = 2, I_T33 = 3, I_V01 = 4, I_V23 = 5, I_T01 = I_V01;
    constexpr int I_V02 = I_T22, I_V03 = I_T33, I_V12 = I_V23, I_V13 = 6;      // (T(2,2), T(3,3), V(2,3) are in registers by then)
    const float* sLd = tiles;
    auto tile = [&](int i) { return tiles + i * 16 * TP; };
    auto lds_sync = [] { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); };   // (LDS operations of a wave execute in order)
    // ---- diagonal blocks: X (I + L) = I by rows, from the right.  Lane c16 of group g owns row c16 of block g; as soon as
    // x_i is known it is folded into the pending sums of all earlier columns (a dependent chain of 16 short steps) ----
    {
        const float* ld = sLd + g * 256;
        float x[16], acc[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[i] = 0.f;
#pragma unroll
        for (int i = 15; i >= 0; --i) {
            x[i] = ((i == c16) ? 1.f : 0.f) - acc[i];
            float row[16];
#pragma unroll
            for (int q4 = 0; q4 < (i + 3) / 4; ++q4) *(f32x4*)(row + 4 * q4) = *(const f32x4*)(ld + i * 16 + 4 * q4);
#pragma unroll
            for (int j = 0; j < i; ++j) acc[j] += row[j] * x[i];
        }
        // T(g,g) = X_gg^T as a left factor: [row j][column c16]
        float* tt = tile(I_T00 + g);             // (group g: block g)
#pragma unroll
        for (int j = 0; j < 16; ++j) tt[j * TP + c16] = x[j];
    }
    lds_sync();
    auto acc_layout = [&](int i) {               // a tile of LDS in accumulator layout
        const float* t = tile(i);
        return f32x4{t[(4 * g) * TP + c16], t[(4 * g + 1) * TP + c16], t[(4 * g + 2) * TP + c16], t[(4 * g + 3) * TP + c16]};
    };
    // acc + A B: A a tile of LDS by rows, B in accumulator layout
    auto mul = [&](int ia, f32x4 B, f32x4 acc) {
        const f32x4 a = *(const f32x4*)(tile(ia) + c16 * TP + 4 * g);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], B[e], acc, 0, 0, 0);
        return acc;
    };
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    auto put = [&](int i, f32x4 v) {             // a tile in accumulator layout to LDS, by rows
#pragma unroll
        for (int r = 0; r < 4; ++r) tile(i)[(4 * g + r) * TP + c16] = v[r];
    };
    const f32x4 T00 = acc_layout(I_T00), T11 = acc_layout(I_T11), T22 = acc_layout(I_T22), T33 = acc_layout(I_T33);
    // ---- merge 16 -> 32: T(lo,hi) = -(T(lo,lo) U(lo,hi)) T(hi,hi) ----
    put(I_V01, mul(I_T00, U[0][1], zero));
    put(I_V23, mul(I_T22, U[2][3], zero));
    lds_sync();
    const f32x4 T01 = -mul(I_V01, T11, zero);
    const f32x4 T23 = -mul(I_V23, T33, zero);
    put(I_T01, T01);
    lds_sync();
    // ---- merge 32 -> 64: V = T[0:32][0:32] U[0:32][32:64], T[0:32][32:64] = -V T[32:64][32:64] (zero tiles left out) ----
    put(I_V02, mul(I_T00, U[0][2], mul(I_T01, U[1][2], zero)));
    put(I_V03, mul(I_T00, U[0][3], mul(I_T01, U[1][3], zero)));
    put(I_V12, mul(I_T11, U[1][2], zero));
    put(I_V13, mul(I_T11, U[1][3], zero));
    lds_sync();
    const f32x4 T02 = -mul(I_V02, T22, zero), T03 = -mul(I_V03, T33, mul(I_V02, T23, zero));
    const f32x4 T12 = -mul(I_V12, T22, zero), T13 = -mul(I_V13, T33, mul(I_V12, T23, zero));
    X[0][0] = T00; X[0][1] = T01; X[0][2] = T02; X[0][3] = T03; X[1][1] = T11; X[1][2] = T12; X[1][3] = T13;
    X[2][2] = T22; X[2][3] = T23; X[3][3] = T33;
}

}  // namespace gdn
