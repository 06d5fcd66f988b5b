// zbatch.hpp -- the flux-form z pass (zflux.hpp has its algebra) with every
// sequence of an x-row in one batch, for short rows.
//
// k_zc keeps three points per thread and takes its sequences a few at a time,
// which suits rows long enough to fill a block's LDS: at NN = 32..128 a launch
// is then a handful of blocks, each a chain of eight or nine batches.  Here a
// block of K0 NN threads (at most 1024) takes one x-row and does each stage of
// the pass once: fold of all base lines, their inverse transforms, one point
// per thread for the products, the forward transforms of all rows, and one
// (k, n) per thread for the lines, with six block barriers in all.
//
// Sequences: inverse (pair p of base lines, phase b) at 3 p + b.  Forward: k = 0
// (uw, ww - uu) at b; k >= 1 from 3 + 8 (k-1): (uv, uw) at b, (vv - uu, vv - ww) at 3
// + b, and vw alone with its phases 0 and 1 as the real and imaginary part of
// one sequence (6) and phase 2 in the next (7), so that every k >= 1 is laid
// out alike.
#pragma once
#include "zflux.hpp"

template <int K0, int LOGNN> constexpr int zs_threads() { return (K0 << LOGNN) < 1024 ? (K0 << LOGNN) : 1024; }
template <int K0> constexpr int zs_iseq() { return 3 * ((3 * K0 - 1 + 1) / 2); }
template <int K0> constexpr int zs_fseq() { return 3 + 8 * (K0 - 1); }
template <typename R> constexpr int zs_ls()
{
     return sizeof(R) == 4 ? 4 : 0; // padded or XOR-swizzled (lslot)
}

template <typename R, int K0, int LOGNN> constexpr size_t zs_lds_bytes()
{
    constexpr int NN = 1 << LOGNN;
    return sizeof(cplx_t<R>) * ((size_t)zs_fseq<K0>() * lspan<NN, zs_ls<R>()>() + ptw_size<NN, 1, 7>() + (size_t)NN);
}
// Rows of up to 256 points whose batch fits LDS.  There k_zs is faster than both
// forms of k_zc (us per launch, FP64 M4, one buffer / two buffers / k_zs): NN = 32
// (96 rows) 32 / 26 / 9, NN = 64 (192 rows) 27 / 24 / 10, 256 (768 rows) 51 / 51 /
// 42; M6 128 (384 rows) 45 / 40 / 27; a step of 256 members with NN = 64, 1018
// (two buffers) -> 899; FP32 M6 256 41 / 41 / 40.
template <typename R, int K0, int LOGNN> constexpr bool zs_fits()
{
    return LOGNN <= 8 && zs_lds_bytes<R, K0, LOGNN>() <= 160 * 1024;
}

template <typename R, int K0, int LOGNN>
__global__ __launch_bounds__((zs_threads<K0, LOGNN>())) void k_zs(Batch bt, const cplx_t<R>* __restrict__ U,
                                                               cplx_t<R>* __restrict__ NL,
                                                               const cplx_t<R>* __restrict__ twNN,
                                                               const cplx_t<R>* __restrict__ twQ)
{
    using CT = cplx_t<R>;
    using FR = FluxRows<K0>;
    const Geo g = bt.geo[blockIdx.z];
    U += blockIdx.z * bt.u_stride;
    NL += blockIdx.z * bt.nl_stride;
    constexpr int KK = 3 * K0 - 1;
    constexpr int NN = 1 << LOGNN, H = NN / 2;
    constexpr int T = zs_threads<K0, LOGNN>();
    constexpr int NPI = (KK + 1) / 2;            // pairs of base lines
    constexpr int ISEQ = zs_iseq<K0>(), FSEQ = zs_fseq<K0>();
    constexpr int LS = zs_ls<R>(), LPZ = lspan<NN, LS>();
    constexpr int G = group_lanes<NN>(), PL = NN / G;
    static_assert(ISEQ <= FSEQ, "one buffer");
    extern __shared__ unsigned char smem_raw[];
    CT* buf = reinterpret_cast<CT*>(smem_raw);   // [FSEQ][LPZ]
    CT* twNl = buf + FSEQ * LPZ;                 // [ptw_size<NN, 1, 7>()] pass twiddles
    CT* twQl = twNl + ptw_size<NN, 1, 7>();      // [NN]: w^k, k < NN (twq2 extends them)
    const int tid = threadIdx.x;
    const int x = xcd_tile(blockIdx.x, gridDim.x);
    const bool wide = g.NTs * (int)sizeof(CT) >= 64;

    // ---- fold of the base lines (c2r): task (pair fp, index fr) ----
    constexpr int FTASK = NPI * H, FT = (FTASK + T - 1) / T;
    CT pf[FT][4];
    const CT* u0 = U + ((size_t)(x * KK) << LOGNN);
#pragma unroll
    for (int f = 0; f < FT; f++) {
        const int tau = tid + T * f;
        const int fp = tau / H, fr = tau % H, r2 = fr == 0 ? H : NN - fr;
        const CT z{(R)0, (R)0};
        pf[f][0] = pf[f][1] = pf[f][2] = pf[f][3] = z;
        if (tau < FTASK) {
            const CT* up = u0 + 2 * fp * NN;
            pf[f][0] = up[fr];
            pf[f][1] = up[r2];
            if (2 * fp + 1 < KK) {
                pf[f][2] = up[NN + fr];
                pf[f][3] = up[NN + r2];
            }
        }
    }
    ptw_fill<CT, LOGNN, 1, 7>(twNl, twNN, tid, T);
    for (int i = tid; i < NN; i += T) twQl[i] = twQ[i];
    __syncthreads();
#pragma unroll
    for (int f = 0; f < FT; f++) {
        const int tau = tid + T * f;
        const int fp = tau / H, fr = tau % H, fm = fr == 0 ? H : NN - fr;
        if (tau >= FTASK) continue;
        CT* seq = buf + fp * 3 * LPZ;
        const CT one{(R)1, (R)0};
        zfold_bw<R, LS>(seq, 0, fr, NN, pf[f][0], pf[f][1], pf[f][2], pf[f][3], one, one);
        zfold_bw<R, LS>(seq + LPZ, 1, fr, NN, pf[f][0], pf[f][1], pf[f][2], pf[f][3], twQl[fr], twQl[fm]);
        zfold_bw<R, LS>(seq + 2 * LPZ, 2, fr, NN, pf[f][0], pf[f][1], pf[f][2], pf[f][3], twq2<R>(twQl, NN, 2 * fr),
                        twq2<R>(twQl, NN, 2 * fm));
    }
    __syncthreads();
    // transforms of the first S sequences in place, one lane group each
    auto transform = [&](auto sign, auto nseq) {
        constexpr int S = decltype(nseq)::value;
        const int gl = tid % G;
#pragma unroll
        for (int s0 = 0; s0 < S; s0 += T / G) {
            const int s = s0 + tid / G;
            if (s < S) {
                CT* sq = buf + s * LPZ;
                CT v[PL];
                const int pg = lslot<LS>(gl);
                static_for<0, PL>([&](auto qi) { v[qi] = lsw<decltype(qi)::value * G, LS>(sq, pg); });
                group_fft<CT, LOGNN, decltype(sign)::value, true, 7, 1, 0, LS>(v, sq, gl, twNl);
                static_for<0, PL>([&](auto qi) { lsw<decltype(qi)::value * G, LS>(sq, pg) = v[qi]; });
            }
        }
        __syncthreads();
    };
    transform(std::integral_constant<int, +1>{}, std::integral_constant<int, ISEQ>{});

    // ---- products: task (phase b, r) is the point z = 3 r + b ----
    constexpr int PT = (3 * NN + T - 1) / T;
    static_assert(PT == 1, "one point per thread");
    const R lu = (R)g.cth, lw = (R)g.sth;        // laminar u_1, w_1
    const int b = tid / NN, r = tid & (NN - 1);
    const int pr = lslot<LS>(r);
    R v[KK];
    if (b < 3) {
        static_for<0, NPI>([&](auto pi) {
            constexpr int p = decltype(pi)::value;
            const CT zv = buf[(3 * p + b) * LPZ + pr];
            v[2 * p] = zv.x;
            if constexpr (2 * p + 1 < KK) v[2 * p + 1] = zv.y;
        });
    }
    __syncthreads();
    if (b < 3) {
        buf[b * LPZ + pr] = CT{FR::template row<0>(v, lu, lw), FR::template row<1>(v, lu, lw)};
        static_for<1, K0>([&](auto kc) {
            constexpr int k = decltype(kc)::value, r0 = 2 + 5 * (k - 1);
            CT* sk = buf + (3 + 8 * (k - 1)) * LPZ + pr;
            sk[b * LPZ] = CT{FR::template row<r0 + Dev<K0>::UV>(v, lu, lw), FR::template row<r0 + Dev<K0>::UW>(v, lu, lw)};
            sk[(3 + b) * LPZ] = CT{FR::template row<r0 + Dev<K0>::VVUU>(v, lu, lw),
                                   FR::template row<r0 + Dev<K0>::VVWW>(v, lu, lw)};
            const R vw = FR::template row<r0 + Dev<K0>::VW>(v, lu, lw);
            if (b == 2) sk[7 * LPZ] = CT{vw, (R)0};
            else if (b == 1) sk[6 * LPZ].y = vw;
            else sk[6 * LPZ].x = vw;
        });
    }
    __syncthreads();
    transform(std::integral_constant<int, -1>{}, std::integral_constant<int, FSEQ>{});

    // ---- lines: task (k, n) ----
    constexpr int LT = (K0 * NN + T - 1) / T;
#pragma unroll
    for (int f = 0; f < LT; f++) {
        const int tau = tid + T * f;
        const int k = tau >> LOGNN, n = tau & (NN - 1), nm = (NN - n) & (NN - 1);
        if (k >= K0) continue;
        const int pn = lslot<LS>(n), pm = lslot<LS>(nm);
        const CT w1 = cconj(twQl[n]), w2 = cconj(twq2<R>(twQl, NN, 2 * n));
        // twice the transforms of the two real sequences of complex sequence s
        auto split = [&](const CT* s, CT& F1, CT& F2) {
            const CT zn = s[pn], zm = s[pm];
            F1 = CT{zn.x + zm.x, zn.y - zm.y};
            F2 = CT{zn.y + zm.y, zm.x - zn.x};
        };
        // rows X1, X2 of the pair whose phases are the sequences s, s + 1, s + 2
        auto pair = [&](const CT* s, CT& X1, CT& X2) {
            CT a, c;
            split(s, X1, X2);
            split(s + LPZ, a, c);
            X1 = cadd(X1, cmul(a, w1));
            X2 = cadd(X2, cmul(c, w1));
            split(s + 2 * LPZ, a, c);
            X1 = cadd(X1, cmul(a, w2));
            X2 = cadd(X2, cmul(c, w2));
        };
        CT* nlr = NL + ((((size_t)(n >> g.lgNS) * dev_lines(K0) + dev_line(k)) * g.P + x) << g.lgNS) + (n & (g.NTs - 1));
        const size_t nls = (size_t)g.P << g.lgNS;
        const double gn = g.gamma * n;
        CT uw;
        if (k == 0) {
            CT d;
            pair(buf, uw, d);
            st_piece(nlr + DEV_UW * nls, uw, wide);
            st_piece(nlr + DEV_F * nls, cscale(d, (R)gn), wide);
            continue;
        }
        const CT* sk = buf + (3 + 8 * (k - 1)) * LPZ;
        CT uv, vvuu, vvww, vw, a, c;
        pair(sk, uv, uw);
        st_piece(nlr + DEV_UW * nls, uw, wide);
        st_piece(nlr + DEV_UV * nls, uv, wide);
        pair(sk + 3 * LPZ, vvuu, vvww);
        split(sk + 6 * LPZ, vw, a);
        vw = cadd(vw, cmul(a, w1));
        split(sk + 7 * LPZ, a, c);
        vw = cadd(vw, cmul(a, w2));
        const DevMul<R> m = dev_mul<R>(gn, 1.0 / gn, ak1_of(k, g.beta));
        if (m.far) vvuu = csub(vvuu, vvww); // ww - uu
        st_piece(nlr + DEV_F * nls, CT{m.f * vvww.x - m.h * vw.y, m.f * vvww.y + m.h * vw.x}, wide);
        st_piece(nlr + DEV_E * nls, CT{m.ak * vvuu.x + m.e * vw.y, m.ak * vvuu.y - m.e * vw.x}, wide);
    }
}
