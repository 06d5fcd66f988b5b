// xall.hpp -- the fused x kernel of the flux form with all lines of a block
// transformed at once, for tiles of few columns.
//
// k_xstep takes the lines of its tile (2048/MM columns) one after another: the
// longest contiguous pieces, but a chain of up to seven transforms with three
// barriers each, and few blocks where MM NN is small.  Here a block takes XA/MM
// columns (XA = 128, 256 or 512 values a line) and holds its four NL lines, and
// then its three U lines, in LDS together: one load, one transform stage and
// one unfold for all of them, five barriers in all, and four to sixteen times
// as many blocks.  The loads of the state and the history start with those of
// the lines.  Arithmetic and order per value are k_xstep's, so a member steps
// the same whichever kernel its launch takes (xtile_log).
#pragma once
#include "kernels.hpp"

template <int LOGXA> constexpr int xa_threads() { return 3 << (LOGXA - 1); }
template <typename R, int LOGMM, int LOGXA> constexpr size_t xa_lds_bytes()
{
    constexpr size_t MM = (size_t)1 << LOGMM;
    return (((size_t)12 << LOGXA) + ptw_size<(1 << LOGMM), 1, 7>()) * sizeof(cplx_t<R>) + (2 * MM + 1) * sizeof(double2);
}

template <typename R, int LOGMM, int LOGXA, bool INV_ONLY>
__global__ __launch_bounds__(xa_threads<LOGXA>()) void k_xall(Batch bt, const cplx_t<R>* __restrict__ NL,
                                                              double2* __restrict__ c, cplx_t<R>* __restrict__ onl,
                                                              cplx_t<R>* __restrict__ U,
                                                              const cplx_t<R>* __restrict__ twMM,
                                                              const double2* __restrict__ twP, int nst)
{
    using CT = cplx_t<R>;
    constexpr int MM = 1 << LOGMM, XA = 1 << LOGXA;
    constexpr int T = xa_threads<LOGXA>();
    constexpr int LOGNT = LOGXA - LOGMM, NT = 1 << LOGNT; // columns
    constexpr int G = group_lanes<MM>(), PL = MM / G;
    static_assert(LOGMM <= 9 && LOGNT >= 0 && 12 * NT * G == T, "one lane group per sequence");
    extern __shared__ unsigned char smem_raw[];
    CT* reg = reinterpret_cast<CT*>(smem_raw); // [line][t][b] sequences of MM, swizzled
    CT* twMl = reg + 12 * XA;                  // pass twiddles of the MM-point transforms (seven-entry)
    double2* twPl = reinterpret_cast<double2*>(twMl + ptw_size<MM, 1, 7>()); // exp(2 pi i j/P), j <= 2 MM

    const Geo g = bt.geo[blockIdx.z];
    NL += blockIdx.z * bt.nl_stride;
    c += blockIdx.z * bt.c_stride;
    onl += blockIdx.z * bt.c_stride;
    U += blockIdx.z * bt.u_stride;
    const int n0 = xcd_tile(blockIdx.x, gridDim.x) << LOGNT;
    const int k = blockIdx.y;
    const int tid = threadIdx.x;
    const double ak1 = ak1_of(k, g.beta), rak = k == 0 ? -1.0 : 1.0 / ak1;
    const double ak2 = ak2_of(k, g.beta);
    const int nlin = k == 0 ? 2 : 4; // NL lines

    // item (t, r) of a thread, and its slots of the state (psi, phi at m = r, r - MM)
    const bool item = tid < XA;
    const int t = tid >> LOGMM, r = tid & (MM - 1), n = n0 + t;
    const size_t cpsi = ((size_t)n * g.K + k) * g.ldM, cphi = ((size_t)n * g.K + (g.K0 - 1 + k)) * g.ldM;
    double2 psi[2] = {}, phi[2] = {};

    // transposes between a line ([x][t], element i = tid + T q, x = 3a + b) and
    // its sequences: two elements per thread and line, a MM/2 apart
    const int t0 = tid & (NT - 1), x0 = tid >> LOGNT, a0 = x0 / 3, b0 = x0 - 3 * a0;
    CT* const rb = reg + (t0 * 3 + b0) * MM;
    const int pa = pidx(a0) ^ xsw<R>(t0, b0);
    // this thread's sequence (line, t, b) and lane
    const int s = tid / G, gl = tid % G;
    CT* const sq = reg + s * MM;
    const int sxo = xsw<R>((s / 3) & (NT - 1), s % 3);
    const int pg = pidx(gl) ^ sxo;
    auto transform = [&](auto sign, int nl) {
        if (s < 3 * NT * nl) {
            CT v[PL];
            static_for<0, PL>([&](auto qi) { v[qi] = swz<decltype(qi)::value * G>(sq, pg); });
            group_fft<CT, LOGMM, decltype(sign)::value, true, 7>(v, sq, gl, twMl, sxo);
            static_for<0, PL>([&](auto qi) { swz<decltype(qi)::value * G>(sq, pg) = v[qi]; });
        }
        __syncthreads();
    };

    double2 cv[2][2];
    CT ov[2][2];
    auto state_at = [&](int h) { return h == 0 ? r : MM - 1 + r; };
    if constexpr (INV_ONLY) {
        if (item) {
#pragma unroll
            for (int h = 0; h < 2; h++) {
                if (h == 1 && r == 0) continue;
                psi[h] = c[cpsi + state_at(h)];
                if (k > 0) phi[h] = c[cphi + state_at(h)];
            }
        }
        ptw_fill<CT, LOGMM, 1, 7>(twMl, twMM, tid, T);
        for (int i = tid; i <= 2 * MM; i += T) twPl[i] = twP[i];
        __syncthreads();
    } else {
        CT lv[4][2];
        const CT* pan = nl_panel(g, NL, n0, dev_line(k)) + ((size_t)x0 << g.lgNS) + t0;
        const size_t lstep = (size_t)g.P << g.lgNS, xstep = (size_t)(3 * MM / 2) << g.lgNS;
#pragma unroll
        for (int l = 0; l < 4; l++)
            if (l < nlin) {
                lv[l][0] = pan[l * lstep];
                lv[l][1] = pan[l * lstep + xstep];
            }
        if (nlin == 4 && g.NLL > dev_lines(g.K0)) { // its vw and ww shares have a line of their own
            const CT* pe = pan + (ptrdiff_t)(dev_lines(g.K0) + k - 1 - dev_line(k)) * lstep;
            lv[DEV_E][0] = cadd(lv[DEV_E][0], pe[0]);
            lv[DEV_E][1] = cadd(lv[DEV_E][1], pe[xstep]);
        }
        if (item) {
#pragma unroll
            for (int h = 0; h < 2; h++) {
                if (h == 1 && r == 0) continue;
                cv[h][0] = c[cpsi + state_at(h)];
                if (!nst) ov[h][0] = onl[cpsi + state_at(h)];
                if (k > 0) {
                    cv[h][1] = c[cphi + state_at(h)];
                    if (!nst) ov[h][1] = onl[cphi + state_at(h)];
                }
            }
        }
        ptw_fill<CT, LOGMM, 1, 7>(twMl, twMM, tid, T);
        for (int i = tid; i <= 2 * MM; i += T) twPl[i] = twP[i];
#pragma unroll
        for (int l = 0; l < 4; l++)
            if (l < nlin) {
                CT* rl = rb + l * 3 * XA;
                rl[pa] = lv[l][0];
                swz<MM / 2>(rl, pa) = lv[l][1];
            }
        __syncthreads();
        transform(std::integral_constant<int, -1>{}, nlin);

        // ---------------- psi, phi of the nonlinear term, update ----------------
        if (item) {
#pragma unroll
            for (int l = 0; l < 4; l++) {
                if (l >= nlin) continue;
                const CT* bt3 = reg + (l * NT + t) * 3 * MM;
                double2 Xp, Xn;
                xunfold(bt3[pidx(r) ^ xsw<R>(t, 0)], bt3[MM + (pidx(r) ^ xsw<R>(t, 1))],
                        bt3[2 * MM + (pidx(r) ^ xsw<R>(t, 2))], twPl, r, MM, Xp, Xn);
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    if (h == 1 && r == 0) continue;
                    const int mi = state_at(h);
                    double am1, am2, an1, an2;
                    xwave(g, mi, am1, am2);
                    zwave(g, n, an1, an2);
                    dev_term(l, mi == 0 && n == 0, h == 0 ? Xp : Xn, am1, an1, ak1, rak, psi[h], phi[h]);
                }
            }
            const double dt = g.dt;
#pragma unroll
            for (int h = 0; h < 2; h++) {
                if (h == 1 && r == 0) continue;
                const int mi = state_at(h);
                double am1, am2, an1, an2;
                xwave(g, mi, am1, am2);
                zwave(g, n, an1, an2);
                const bool mean = (mi == 0 && n == 0);
#pragma unroll
                for (int which = 0; which < 2; which++) {
                    if (which == 1 && k == 0) continue;
                    const size_t idx = (which == 0 ? cpsi : cphi) + mi;
                    double2 nl = which == 0 ? psi[h] : phi[h];
                    nl = double2{nl.x * dev_scale(g), nl.y * dev_scale(g)};
                    double lhs, rhs;
                    lhsrhs_k(g, k, which, mean, am2, an2, ak2, lhs, rhs);
                    const double2 old = nst ? nl : hist_wide(ov[h][which]);
                    double2 cn = ab2_update(cv[h][which], nl, old, lhs, rhs, dt);
                    if (mean && which == 0 && k == 0) cn.x = 0.0;
                    c[idx] = cn;
                    hist_store(onl + idx, nl, true);
                    if (which == 0) psi[h] = cn;
                    else phi[h] = cn;
                }
            }
        }
        __syncthreads();
    }

    // ---------------- inverse x transform of the new state: u, v, w ----------------
    if (item) {
        double2 f[2][3];
#pragma unroll
        for (int h = 0; h < 2; h++) {
            f[h][0] = f[h][1] = f[h][2] = double2{0.0, 0.0};
            if (h == 1 && r == 0) continue;
            mpt2spec_k(g, k, state_at(h), n, psi[h], phi[h], false, f[h][0], f[h][1], f[h][2]);
        }
#pragma unroll
        for (int l = 0; l < 3; l++) {
            CT* bt3 = reg + (l * NT + t) * 3 * MM;
            const double2 X0 = f[0][l], X1 = f[1][l], y0 = xfold_0(X0, X1);
            bt3[pidx(r) ^ xsw<R>(t, 0)] = CT{(R)y0.x, (R)y0.y};
#pragma unroll
            for (int b = 1; b < 3; b++) {
                const double2 y = xfold_b(X0, X1, twPl[r * b], twPl[(MM - r) * b]); // w2 conj: exp(2 pi i (r-MM) b / P)
                bt3[b * MM + (pidx(r) ^ xsw<R>(t, b))] = CT{(R)y.x, (R)y.y};
            }
        }
    }
    __syncthreads();
    transform(std::integral_constant<int, +1>{}, 3);
    const bool wide = NT * (int)sizeof(CT) >= 64;
#pragma unroll
    for (int l = 0; l < 3; l++) {
        if (k == 0 && l == 1) continue;
        // spec slot of u_k, v_k, w_k: k, K0-1+k, 2K0-1+k
        const int line = l == 0 ? k : (l == 1 ? g.K0 - 1 + k : 2 * g.K0 - 1 + k);
        CT* ub = U + ((size_t)x0 * g.UL + line) * g.NN + n0 + t0;
        CT* rl = rb + l * 3 * XA;
        st_piece(ub, rl[pa], wide);
        st_piece(ub + (size_t)(3 * MM / 2) * g.UL * g.NN, swz<MM / 2>(rl, pa), wide);
    }
}

// The fused x kernel of a launch of nblk full k_xstep blocks (2048/MM columns
// each): log2 of the values of a line in a tile, 11 and 10 for k_xstep (whole and
// half tiles), 6 to 9 for k_xall.  us per launch on the MI355X, FP64 M4 unless said:
//   nblk   8 (MM = NN = 64):    k_xstep 50, k_xall 64..512 12, 12, 14, 20
//         32 (256, 64):         53; 256, 512 23, 28
//         48 (M6 128, 128):     58; 128..512 32, 33, 28
//         64 (512, 64):         61; 512 38;  (256, 128): half tiles 43, k_xall 31
//         96 (M6 256, 128; 512, 64; 128, 256): half tiles 44, 50, 44, k_xall 53, 67, 46
//            (FP32: 38, 39, 36 and 38, 42, 32)
//        128 (256, 256; 128, 512; 512, 128): whole 57, 63, 64, half 45, 45, 52; (FP32
//            48, 48, 49 and 39, 36, 40); k_xall 512 (256, 256) 60
//        192 (M6 256, 256):     whole 62, half 84
//        512 (512, 512):        whole 147, half 201, k_xall 271
//        2048 (256 members of 64, 64): a step 899, with k_xall 512 1067
// Up to one block per CU smaller tiles win, beyond it the longer pieces do.
// Below, k_xall takes the largest tile that still gives about 160 blocks.
template <typename R, int LOGMM> inline int xtile_log(int nblk, int NN)
{
    if (LOGMM > 9 || nblk > 128) return LOG_XTILE;
    if (LOGMM >= 6 && NN >= (1 << 10) >> LOGMM && (nblk > 96 || (nblk > 64 && LOGMM >= (sizeof(R) == 8 ? 7 : 9)))) return 10;
    if (nblk >= 128) return LOG_XTILE;
    int lx = 9;
    while (lx > 6 && lx > LOGMM && (nblk << (LOG_XTILE - lx)) < 160) lx--;
    while (lx > LOGMM && (1 << (lx - LOGMM)) > NN) lx--; // whole tiles
    return lx;
}
