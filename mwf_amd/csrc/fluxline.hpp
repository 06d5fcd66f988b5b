// fluxline.hpp -- the lines in which the nonlinear term of the flux form crosses
// from the z to the x kernels, and the weights with which psi and phi take them.
// Plain arithmetic, host and device (zflux.hpp has the rows).
//
// With a = alpha m, g = gamma n, ak = ak1(k), psi and phi of a wall-normal index
// k >= 1 are polynomials in a whose coefficients are four lines: uw, uv and two of
//
//   A = ak (vv - uu) - i g vw,         B = ak g (vv - ww) + i (ak^2 - g^2) vw
//   C = ak (ww - uu) - i (ak^2 / g) vw,  D = B / g = ak (vv - ww) + i (ak^2 / g - g) vw
//
//   psi = (a^2 - g^2) uw + i g ak uv + (a g / ak) A - (a / ak) B        = ... + (a g / ak) C
//   phi = i a (ak^2 - a^2 - g^2) uv - 2 ak a g uw + a^2 A + g B         = ... + a^2 C + (a^2 + g^2) D
//
// A line is rounded to the precision of the transforms before its weight is
// applied, so no weighted part of a line may be large and cancel.  Of A, B the
// parts a (g^2 / ak) vw cancel in psi, of C, D the parts a^2 (ak^2 / g) vw in phi:
// harmless where |g| <= |ak| and where |g| > |ak| respectively, g / ak and ak / g times
// the result's own rounding elsewhere.  So the pair is chosen per n: C, D
// where |g| > |ak| (far), else A, B.  The first line has the same weights in both.
// With A and B throughout, the nonlinear term of a full spectrum with alpha
// MM = gamma NN = 4096 was off by 9.3e-6 in FP32 and 2.1e-14 in FP64 (MM = NN = 32),
// with the rule by 1.9e-7 and 4.9e-16, and at every box tried it is closer in FP32 than the
// form with a line per velocity component (alpha MM = gamma NN = 512, evaluated on
// the CPU: 1.6e-7 and 2.4e-7; 8: 1.7e-7 and 3.3e-7).  It costs the z kernels up to
// 1.5 % (FP64 M6 NN = 512, 211 -> 214 us), a step at most 1 % but for short launches of
// FP64 rows of 512 (M4 MM = 128, 87.6 -> 90.6 us), and the one-buffer FP64 form, which no
// rule picks, the registers it has not got (M4 MM = NN = 512, k_zc 152 -> 191 us).
// For k = 0: uw and B = g (ww - uu), psi = (a^2 - g^2) uw + a B.
#pragma once

// Lines of k >= 1: uw, B or D, uv, A or C; of k = 0: uw and B.
enum { DEV_UW, DEV_F, DEV_UV, DEV_E };
__host__ __device__ constexpr int dev_line(int k) { return k == 0 ? 0 : 4 * k - 2; }
__host__ __device__ constexpr int dev_lines(int K0) { return 4 * K0 - 2; }
// with the vw and ww shares of A or C on a line of its own, dev_lines + k - 1 (FP64
// rows of 1024 points; Geo::NLL tells the x kernels)
__host__ __device__ constexpr int dev_lines_split(int K0) { return 5 * K0 - 3; }

// the z kernels and the x kernels decide alike: g = gamma * n and ak = ak1_of(k)
// are the same products in both
__host__ __device__ inline bool dev_far(double g, double ak)
{
    return ak != 0.0 && __builtin_fabs(g) > __builtin_fabs(ak);
}

// Multipliers of the rows at one n: line DEV_E is ak vvuu - i e vw, less ak vvww
// where far, line DEV_F is f vvww + i h vw.  Formed in FP64 and rounded once; rg is
// 1 / g, used where far only.
template <typename R> struct DevMul {
    R ak, e, f, h;
    bool far;
};
template <typename R> __host__ __device__ inline DevMul<R> dev_mul(double g, double rg, double ak)
{
    const bool far = dev_far(g, ak);
    const double q = ak * ak, e = far ? q * rg : g;
    return DevMul<R>{(R)ak, (R)e, (R)(far ? ak : ak * g), (R)(far ? e - g : q - g * g), far};
}

// weights cp, cq of line li (for DEV_UV of i uv) in psi_k and phi_k; rak is 1 / ak,
// -1 for k = 0
__host__ __device__ inline void dev_weights(int li, double a, double g, double ak, double rak, double& cp, double& cq)
{
#pragma clang fp contract(off)
    const double a2 = a * a, g2 = g * g;
    if (li == DEV_UW) {
        cp = a2 - g2;
        cq = -2.0 * ak * (a * g);
    } else if (li == DEV_F) {
        const bool far = dev_far(g, ak);
        cp = far ? 0.0 : -(a * rak);
        cq = far ? a2 + g2 : g;
    } else if (li == DEV_UV) {
        cp = g * ak;
        cq = a * (ak * ak - (a2 + g2));
    } else {
        cp = a * g * rak;
        cq = a2;
    }
}
