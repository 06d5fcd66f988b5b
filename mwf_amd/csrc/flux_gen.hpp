// GENERATED by gen_galerkin.py -- do not edit.
// Flux (conservative) form of the wall-normal Galerkin products: the real
// rows of the z pass at one point, from the base values v[KK] of the
// perturbation and the laminar profile (lu, lw) sin(beta y), which adds lu to
// u_1 and lw to w_1.  The constants of the profile's own products (lu lu, lu
// lw, lw lw) are left out: they touch the (0,0) mode of uw, ww - uu and vv - uu
// only, which nothing reads.  See gen_galerkin.py for the derivation.
#pragma once

template <int K0> struct FluxRows;

template <> struct FluxRows<4> {
  template <int ROW, typename R>
  __host__ __device__ static __forceinline__ R row(const R* v, R lu, R lw) {
    const R u1 = v[1] + lu, w1 = v[8] + lw;
    if constexpr (ROW == 0) { return (v[0] * v[7]) + (R)(1.0/2.0) * (v[1] * w1 + lu * v[8]) + (R)(1.0/2.0) * (v[2] * v[9]) + (R)(1.0/2.0) * (v[3] * v[10]); }  // uw_0
    else if constexpr (ROW == 1) { return (R)-1.0 * (v[0] * v[0]) + (R)(-1.0/2.0) * (v[1] * (u1 + lu)) + (R)(-1.0/2.0) * (v[2] * v[2]) + (R)(-1.0/2.0) * (v[3] * v[3]) + (v[7] * v[7]) + (R)(1.0/2.0) * (v[8] * (w1 + lw)) + (R)(1.0/2.0) * (v[9] * v[9]) + (R)(1.0/2.0) * (v[10] * v[10]); }  // ww_0 - uu_0
    else if constexpr (ROW == 2) { return (v[0] * v[4]) + (R)(1.0/2.0) * (u1 * v[5]) + (R)(1.0/2.0) * (v[2] * v[4]) + (R)(1.0/2.0) * (v[2] * v[6]) + (R)(1.0/2.0) * (v[3] * v[5]); }  // uv_1
    else if constexpr (ROW == 3) { return (v[0] * w1) + (u1 * v[7]) + (R)(-1.0/2.0) * (u1 * v[9]) + (R)(-1.0/2.0) * (v[2] * w1) + (R)(1.0/2.0) * (v[2] * v[10]) + (R)(1.0/2.0) * (v[3] * v[9]); }  // uw_1
    else if constexpr (ROW == 4) { return (R)-2.0 * (v[0] * u1) + (u1 * v[2]) + (R)-1.0 * (v[2] * v[3]) + (v[4] * v[5]) + (R)-1.0 * (v[5] * v[6]); }  // vv_1 - uu_1
    else if constexpr (ROW == 5) { return (v[4] * v[7]) + (R)(1.0/2.0) * (v[4] * v[9]) + (R)(1.0/2.0) * (v[5] * w1) + (R)(1.0/2.0) * (v[5] * v[10]) + (R)(1.0/2.0) * (v[6] * v[9]); }  // vw_1
    else if constexpr (ROW == 6) { return (v[4] * v[5]) + (R)-1.0 * (v[5] * v[6]) + (R)-2.0 * (v[7] * w1) + (w1 * v[9]) + (R)-1.0 * (v[9] * v[10]); }  // vv_1 - ww_1
    else if constexpr (ROW == 7) { return (v[0] * v[5]) + (R)(1.0/2.0) * (u1 * v[4]) + (R)(-1.0/2.0) * (u1 * v[6]) + (R)(1.0/2.0) * (v[3] * v[4]); }  // uv_2
    else if constexpr (ROW == 8) { return (v[0] * v[9]) + (R)(-1.0/2.0) * (v[1] * w1 + lu * v[8]) + (R)(1.0/2.0) * (u1 * v[10]) + (v[2] * v[7]) + (R)(1.0/2.0) * (v[3] * w1); }  // uw_2
    else if constexpr (ROW == 9) { return (R)-2.0 * (v[0] * v[2]) + (R)(1.0/2.0) * (v[1] * (u1 + lu)) + (R)-1.0 * (u1 * v[3]) + (R)(1.0/2.0) * (v[4] * v[4]) + (v[4] * v[6]); }  // vv_2 - uu_2
    else if constexpr (ROW == 10) { return (R)(1.0/2.0) * (v[4] * w1) + (R)(1.0/2.0) * (v[4] * v[10]) + (v[5] * v[7]) + (R)(-1.0/2.0) * (v[6] * w1); }  // vw_2
    else if constexpr (ROW == 11) { return (R)(1.0/2.0) * (v[4] * v[4]) + (v[4] * v[6]) + (R)-2.0 * (v[7] * v[9]) + (R)(1.0/2.0) * (v[8] * (w1 + lw)) + (R)-1.0 * (w1 * v[10]); }  // vv_2 - ww_2
    else if constexpr (ROW == 12) { return (v[0] * v[6]) + (R)(-1.0/2.0) * (u1 * v[5]) + (R)(1.0/2.0) * (v[2] * v[4]); }  // uv_3
    else if constexpr (ROW == 13) { return (v[0] * v[10]) + (R)(1.0/2.0) * (u1 * v[9]) + (R)(1.0/2.0) * (v[2] * w1) + (v[3] * v[7]); }  // uw_3
    else if constexpr (ROW == 14) { return (R)-2.0 * (v[0] * v[3]) + (R)-1.0 * (u1 * v[2]) + (v[4] * v[5]); }  // vv_3 - uu_3
    else if constexpr (ROW == 15) { return (R)(1.0/2.0) * (v[4] * v[9]) + (R)(-1.0/2.0) * (v[5] * w1) + (v[6] * v[7]); }  // vw_3
    else if constexpr (ROW == 16) { return (v[4] * v[5]) + (R)-2.0 * (v[7] * v[10]) + (R)-1.0 * (w1 * v[9]); }  // vv_3 - ww_3
    else { return (R)0; }
  }
};

template <> struct FluxRows<6> {
  template <int ROW, typename R>
  __host__ __device__ static __forceinline__ R row(const R* v, R lu, R lw) {
    const R u1 = v[1] + lu, w1 = v[12] + lw;
    if constexpr (ROW == 0) { return (v[0] * v[11]) + (R)(1.0/2.0) * (v[1] * w1 + lu * v[12]) + (R)(1.0/2.0) * (v[2] * v[13]) + (R)(1.0/2.0) * (v[3] * v[14]) + (R)(1.0/2.0) * (v[4] * v[15]) + (R)(1.0/2.0) * (v[5] * v[16]); }  // uw_0
    else if constexpr (ROW == 1) { return (R)-1.0 * (v[0] * v[0]) + (R)(-1.0/2.0) * (v[1] * (u1 + lu)) + (R)(-1.0/2.0) * (v[2] * v[2]) + (R)(-1.0/2.0) * (v[3] * v[3]) + (R)(-1.0/2.0) * (v[4] * v[4]) + (R)(-1.0/2.0) * (v[5] * v[5]) + (v[11] * v[11]) + (R)(1.0/2.0) * (v[12] * (w1 + lw)) + (R)(1.0/2.0) * (v[13] * v[13]) + (R)(1.0/2.0) * (v[14] * v[14]) + (R)(1.0/2.0) * (v[15] * v[15]) + (R)(1.0/2.0) * (v[16] * v[16]); }  // ww_0 - uu_0
    else if constexpr (ROW == 2) { return (v[0] * v[6]) + (R)(1.0/2.0) * (u1 * v[7]) + (R)(1.0/2.0) * (v[2] * v[6]) + (R)(1.0/2.0) * (v[2] * v[8]) + (R)(1.0/2.0) * (v[3] * v[7]) + (R)(1.0/2.0) * (v[3] * v[9]) + (R)(1.0/2.0) * (v[4] * v[8]) + (R)(1.0/2.0) * (v[4] * v[10]) + (R)(1.0/2.0) * (v[5] * v[9]); }  // uv_1
    else if constexpr (ROW == 3) { return (v[0] * w1) + (u1 * v[11]) + (R)(-1.0/2.0) * (u1 * v[13]) + (R)(-1.0/2.0) * (v[2] * w1) + (R)(1.0/2.0) * (v[2] * v[14]) + (R)(1.0/2.0) * (v[3] * v[13]) + (R)(-1.0/2.0) * (v[3] * v[15]) + (R)(-1.0/2.0) * (v[4] * v[14]) + (R)(1.0/2.0) * (v[4] * v[16]) + (R)(1.0/2.0) * (v[5] * v[15]); }  // uw_1
    else if constexpr (ROW == 4) { return (R)-2.0 * (v[0] * u1) + (u1 * v[2]) + (R)-1.0 * (v[2] * v[3]) + (v[3] * v[4]) + (R)-1.0 * (v[4] * v[5]) + (v[6] * v[7]) + (R)-1.0 * (v[7] * v[8]) + (v[8] * v[9]) + (R)-1.0 * (v[9] * v[10]); }  // vv_1 - uu_1
    else if constexpr (ROW == 5) { return (v[6] * v[11]) + (R)(1.0/2.0) * (v[6] * v[13]) + (R)(1.0/2.0) * (v[7] * w1) + (R)(1.0/2.0) * (v[7] * v[14]) + (R)(1.0/2.0) * (v[8] * v[13]) + (R)(1.0/2.0) * (v[8] * v[15]) + (R)(1.0/2.0) * (v[9] * v[14]) + (R)(1.0/2.0) * (v[9] * v[16]) + (R)(1.0/2.0) * (v[10] * v[15]); }  // vw_1
    else if constexpr (ROW == 6) { return (v[6] * v[7]) + (R)-1.0 * (v[7] * v[8]) + (v[8] * v[9]) + (R)-1.0 * (v[9] * v[10]) + (R)-2.0 * (v[11] * w1) + (w1 * v[13]) + (R)-1.0 * (v[13] * v[14]) + (v[14] * v[15]) + (R)-1.0 * (v[15] * v[16]); }  // vv_1 - ww_1
    else if constexpr (ROW == 7) { return (v[0] * v[7]) + (R)(1.0/2.0) * (u1 * v[6]) + (R)(-1.0/2.0) * (u1 * v[8]) + (R)(1.0/2.0) * (v[2] * v[9]) + (R)(1.0/2.0) * (v[3] * v[6]) + (R)(-1.0/2.0) * (v[3] * v[10]) + (R)(-1.0/2.0) * (v[4] * v[7]) + (R)(1.0/2.0) * (v[5] * v[8]); }  // uv_2
    else if constexpr (ROW == 8) { return (v[0] * v[13]) + (R)(-1.0/2.0) * (v[1] * w1 + lu * v[12]) + (R)(1.0/2.0) * (u1 * v[14]) + (v[2] * v[11]) + (R)(1.0/2.0) * (v[2] * v[15]) + (R)(1.0/2.0) * (v[3] * w1) + (R)(1.0/2.0) * (v[3] * v[16]) + (R)(1.0/2.0) * (v[4] * v[13]) + (R)(1.0/2.0) * (v[5] * v[14]); }  // uw_2
    else if constexpr (ROW == 9) { return (R)-2.0 * (v[0] * v[2]) + (R)(1.0/2.0) * (v[1] * (u1 + lu)) + (R)-1.0 * (u1 * v[3]) + (R)-1.0 * (v[2] * v[4]) + (R)-1.0 * (v[3] * v[5]) + (R)(1.0/2.0) * (v[6] * v[6]) + (v[6] * v[8]) + (v[7] * v[9]) + (v[8] * v[10]); }  // vv_2 - uu_2
    else if constexpr (ROW == 10) { return (R)(1.0/2.0) * (v[6] * w1) + (R)(1.0/2.0) * (v[6] * v[14]) + (v[7] * v[11]) + (R)(-1.0/2.0) * (v[7] * v[15]) + (R)(-1.0/2.0) * (v[8] * w1) + (R)(1.0/2.0) * (v[8] * v[16]) + (R)(1.0/2.0) * (v[9] * v[13]) + (R)(-1.0/2.0) * (v[10] * v[14]); }  // vw_2
    else if constexpr (ROW == 11) { return (R)(1.0/2.0) * (v[6] * v[6]) + (v[6] * v[8]) + (v[7] * v[9]) + (v[8] * v[10]) + (R)-2.0 * (v[11] * v[13]) + (R)(1.0/2.0) * (v[12] * (w1 + lw)) + (R)-1.0 * (w1 * v[14]) + (R)-1.0 * (v[13] * v[15]) + (R)-1.0 * (v[14] * v[16]); }  // vv_2 - ww_2
    else if constexpr (ROW == 12) { return (v[0] * v[8]) + (R)(-1.0/2.0) * (u1 * v[7]) + (R)(1.0/2.0) * (u1 * v[9]) + (R)(1.0/2.0) * (v[2] * v[6]) + (R)(1.0/2.0) * (v[2] * v[10]) + (R)(1.0/2.0) * (v[4] * v[6]) + (R)(1.0/2.0) * (v[5] * v[7]); }  // uv_3
    else if constexpr (ROW == 13) { return (v[0] * v[14]) + (R)(1.0/2.0) * (u1 * v[13]) + (R)(-1.0/2.0) * (u1 * v[15]) + (R)(1.0/2.0) * (v[2] * w1) + (R)(1.0/2.0) * (v[2] * v[16]) + (v[3] * v[11]) + (R)(-1.0/2.0) * (v[4] * w1) + (R)(1.0/2.0) * (v[5] * v[13]); }  // uw_3
    else if constexpr (ROW == 14) { return (R)-2.0 * (v[0] * v[3]) + (R)-1.0 * (u1 * v[2]) + (u1 * v[4]) + (R)-1.0 * (v[2] * v[5]) + (v[6] * v[7]) + (v[6] * v[9]) + (R)-1.0 * (v[7] * v[10]); }  // vv_3 - uu_3
    else if constexpr (ROW == 15) { return (R)(1.0/2.0) * (v[6] * v[13]) + (R)(1.0/2.0) * (v[6] * v[15]) + (R)(-1.0/2.0) * (v[7] * w1) + (R)(1.0/2.0) * (v[7] * v[16]) + (v[8] * v[11]) + (R)(1.0/2.0) * (v[9] * w1) + (R)(1.0/2.0) * (v[10] * v[13]); }  // vw_3
    else if constexpr (ROW == 16) { return (v[6] * v[7]) + (v[6] * v[9]) + (R)-1.0 * (v[7] * v[10]) + (R)-2.0 * (v[11] * v[14]) + (R)-1.0 * (w1 * v[13]) + (w1 * v[15]) + (R)-1.0 * (v[13] * v[16]); }  // vv_3 - ww_3
    else if constexpr (ROW == 17) { return (v[0] * v[9]) + (R)(1.0/2.0) * (u1 * v[8]) + (R)(-1.0/2.0) * (u1 * v[10]) + (R)(1.0/2.0) * (v[2] * v[7]) + (R)(1.0/2.0) * (v[3] * v[6]) + (R)(1.0/2.0) * (v[5] * v[6]); }  // uv_4
    else if constexpr (ROW == 18) { return (v[0] * v[15]) + (R)(-1.0/2.0) * (u1 * v[14]) + (R)(1.0/2.0) * (u1 * v[16]) + (R)(1.0/2.0) * (v[2] * v[13]) + (R)(-1.0/2.0) * (v[3] * w1) + (v[4] * v[11]) + (R)(1.0/2.0) * (v[5] * w1); }  // uw_4
    else if constexpr (ROW == 19) { return (R)-2.0 * (v[0] * v[4]) + (u1 * v[3]) + (R)-1.0 * (u1 * v[5]) + (R)(-1.0/2.0) * (v[2] * v[2]) + (v[6] * v[8]) + (v[6] * v[10]) + (R)(-1.0/2.0) * (v[7] * v[7]); }  // vv_4 - uu_4
    else if constexpr (ROW == 20) { return (R)(1.0/2.0) * (v[6] * v[14]) + (R)(1.0/2.0) * (v[6] * v[16]) + (R)(1.0/2.0) * (v[7] * v[13]) + (R)(1.0/2.0) * (v[8] * w1) + (v[9] * v[11]) + (R)(-1.0/2.0) * (v[10] * w1); }  // vw_4
    else if constexpr (ROW == 21) { return (v[6] * v[8]) + (v[6] * v[10]) + (R)(-1.0/2.0) * (v[7] * v[7]) + (R)-2.0 * (v[11] * v[15]) + (w1 * v[14]) + (R)-1.0 * (w1 * v[16]) + (R)(-1.0/2.0) * (v[13] * v[13]); }  // vv_4 - ww_4
    else if constexpr (ROW == 22) { return (v[0] * v[10]) + (R)(-1.0/2.0) * (u1 * v[9]) + (R)(1.0/2.0) * (v[2] * v[8]) + (R)(-1.0/2.0) * (v[3] * v[7]) + (R)(1.0/2.0) * (v[4] * v[6]); }  // uv_5
    else if constexpr (ROW == 23) { return (v[0] * v[16]) + (R)(1.0/2.0) * (u1 * v[15]) + (R)(1.0/2.0) * (v[2] * v[14]) + (R)(1.0/2.0) * (v[3] * v[13]) + (R)(1.0/2.0) * (v[4] * w1) + (v[5] * v[11]); }  // uw_5
    else if constexpr (ROW == 24) { return (R)-2.0 * (v[0] * v[5]) + (R)-1.0 * (u1 * v[4]) + (R)-1.0 * (v[2] * v[3]) + (v[6] * v[9]) + (v[7] * v[8]); }  // vv_5 - uu_5
    else if constexpr (ROW == 25) { return (R)(1.0/2.0) * (v[6] * v[15]) + (R)(-1.0/2.0) * (v[7] * v[14]) + (R)(1.0/2.0) * (v[8] * v[13]) + (R)(-1.0/2.0) * (v[9] * w1) + (v[10] * v[11]); }  // vw_5
    else if constexpr (ROW == 26) { return (v[6] * v[9]) + (v[7] * v[8]) + (R)-2.0 * (v[11] * v[16]) + (R)-1.0 * (w1 * v[15]) + (R)-1.0 * (v[13] * v[14]); }  // vv_5 - ww_5
    else { return (R)0; }
  }
};

