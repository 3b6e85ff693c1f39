// Device functions of the lane-private transforms (lanes.hip, staged.hip): a lane is one (operator column, orbital j),
// a 4x4x1 FP32 MFMA applies four rows of a real matrix, one step at a time, to a value of every lane.
#pragma once
#include "common.hpp"

namespace ephip {

constexpr int LP_STEPS = 8;

// One 4x4x1 MFMA a step: rows of the step's block of `m`, the lane's own x.
template <int S>
__device__ __forceinline__ void lp_step(f32x4 &yr, f32x4 &yi, float m, float xr, float xi) {
    yr = __builtin_amdgcn_mfma_f32_4x4x1f32(m, xr, yr, 4, S, 0);
    yi = __builtin_amdgcn_mfma_f32_4x4x1f32(m, xi, yi, 4, S, 0);
}

template <int N, int S = 0>
__device__ __forceinline__ void lp_steps(f32x4 &yr, f32x4 &yi, float m, const float (&xr)[N], const float (&xi)[N]) {
    if constexpr (S < N) {
        lp_step<S>(yr, yi, m, xr[S], xi[S]);
        lp_steps<N, S + 1>(yr, yi, m, xr, xi);
    }
}
template <int N>
__device__ __forceinline__ void lp_apply(f32x4 &yr, f32x4 &yi, float m, const float (&xr)[N], const float (&xi)[N]) {
    yr = yi = f32x4{0.f, 0.f, 0.f, 0.f};
    lp_steps<N>(yr, yi, m, xr, xi);
}

// B[0 .. N) along an axis to (B[h], S_1 .., -D.im / D.re ..), the order of the table's (1, cos_1 .., sin_1 ..)
template <int N>
__device__ __forceinline__ void lp_fold(float (&xr)[N], float (&xi)[N], const float (&br)[N], const float (&bi)[N]) {
    constexpr int H = N / 2;
    xr[0] = br[H];
    xi[0] = bi[H];
#pragma unroll
    for (int p = 1; p <= H; p++) {
        xr[p] = br[H + p] + br[H - p];
        xi[p] = bi[H + p] + bi[H - p];
        xr[H + p] = bi[H - p] - bi[H + p];
        xi[H + p] = br[H + p] - br[H - p];
    }
}

__device__ __forceinline__ float lp_sum16(float x, float y) {  // rows: x01, y01, x23, y23
    const auto s = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(y), false, false);
    return __uint_as_float(s[0]) + __uint_as_float(s[1]);
}
__device__ __forceinline__ float lp_sum32(float x, float y) {  // lower half x, upper half y
    const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(y), false, false);
    return __uint_as_float(s[0]) + __uint_as_float(s[1]);
}
template <int CTRL>
__device__ __forceinline__ float lp_dpp(float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xf, 0xf, true));
}

// Sum over the lanes of one column: row r of the result holds v[r], columns in its first 64 / JL lanes.
template <int JL>
__device__ __forceinline__ float lp_reduce(const float (&v)[4]) {
    float s = lp_sum32(lp_sum16(v[0], v[1]), lp_sum16(v[2], v[3]));
    if constexpr (JL >= 8) s += lp_dpp<0x128>(s);   // row_ror:8
    if constexpr (JL >= 16) s += lp_dpp<0x124>(s);  // row_ror:4
    return s;
}

// v[r] = U_k of unit r, held by lane r of each quad, times (gr[r] + i gi[r])
template <int R>
__device__ __forceinline__ void lp_times(float &tr, float &ti, float ur, float ui, float gr, float gi) {
    constexpr int Q = R | R << 2 | R << 4 | R << 6;  // quad_perm: lane R of the quad to all four
    tr = lp_dpp<Q>(ur) * gr;
    tr = fmaf(-lp_dpp<Q>(ui), gi, tr);
    ti = lp_dpp<Q>(ur) * gi;
    ti = fmaf(lp_dpp<Q>(ui), gr, ti);
}

}  // namespace ephip
