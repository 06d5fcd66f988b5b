// zflux.hpp -- the z pass of the flux (conservative) form of the nonlinear
// term.
//
// For the divergence-free Galerkin field, (u.grad)u = div(u u), and the
// wall-normal derivative moves onto the bases exactly (gen_galerkin.py has
// the derivation).  The z pass then needs only the KK base lines of U (u_k,
// v_k, w_k; no x- or z-derivatives).  The step needs the nonlinear term only as
// its psi and phi parts (var_spec2mpt), and of the six projected products
// uu, uw, ww, uv, vw, vv of a wall-normal index k these take the trace-free
// part alone (the trace is a pressure gradient): five real rows per k >= 1 (uv,
// uw, vv - uu, vw, vv - ww; two for k = 0) are transformed forward, and four lines
// per k >= 1 (two for k = 0; fluxline.hpp has them and their algebra) cross to the
// x kernel, which applies the powers of a and the scale 1/(2 PQ) (Dev below, and
// dev_term in kernels.hpp): M4 17 rows and 14 lines, M6 27 and 22.  The form with
// one line to be differentiated in x and one for the rest per spec slot has 21 rows
// and 22 lines (33 and 34), so 36 % of NL's bytes and of the forward x transforms
// are saved: at M4 1024^2 k_zc 157 -> 141 us and k_xstep 192 -> 149 us in FP64, 79
// -> 72 and 121 -> 101 us in FP32 (134, 148, 69 and 101 us with the later changes
// noted below and in kernels.hpp and the line pair chosen per n).
//
// Block: T = max(512, NN) threads, XB = T/NN x-rows; thread (xl, r) owns the
// points z = 3r + b, b = 0..2, of row xl, and the output index n = r of that
// row in every line, so a line whose rows straddle two batches is summed in
// the thread's registers.  Sequences of ZP pairs per batch; lane group g of
// G = min(64, NN/8) lanes transforms sequence g of the batch in place with
// wave-local exchanges only (group_fft), so the radix passes need no block
// barrier: a batch has one barrier between its fold and its transforms and
// one between the transforms and the unfold (NN = 1024 and the FP64 one-
// buffer form, whose registers do not hold a lane group's values, keep
// block-wide Stockham passes).  With two buffers (PP) batches
// alternate between them and need no third barrier; one buffer (at or under
// 80 KB, so that two blocks can share a CU) adds a barrier after the unfold.
#pragma once
#include "kernels.hpp"
#include "flux_gen.hpp"

// Rows and lines of the z pass.  Row r (value: FluxRows in flux_gen.hpp): 0, 1
// are uw_0, ww_0 - uu_0; 2 + 5 (k-1) + t, t = 0..4, are uv, uw, vv - uu, vw, vv -
// ww of k >= 1, transformed two per complex sequence in the order of order().
// Lines of k start at dev_line(k).
//
// U holds the perturbation; the laminar profile enters where the rows are
// formed, without its own products, whose constants only the unused (0,0) modes
// would see.  With the profile in U the rounding of its unit-size constant
// spread over every mode: the FP32 nonlinear term is 1.5 to 6 times closer to
// the FP64 one this way (rms velocity 0.3 to 0.05).
//
// PART 0 is the whole pass.  PART 1, 2, 3 take the rows that need two of the
// three components only (u w: uw and ww_0 - uu_0; u v: uv, vv - uu; v w: vw,
// vv - ww), for rows so long that one block's registers do not hold all the base
// values of its points; the vw and ww shares of line DEV_E then go to a line of their
// own, dev_lines + k - 1, which the x kernel adds.
template <int K0_, int PART = 0> struct Dev {
    static constexpr int K0 = K0_;
    // base lines, and the spec slot of base line i
    static constexpr int NB = PART == 0 ? 3 * K0 - 1 : PART == 1 ? 2 * K0 : 2 * K0 - 1;
    __host__ __device__ static constexpr int base(int i)
    {
        return PART == 1 ? (i < K0 ? i : i + K0 - 1) : PART == 3 ? i + K0 : i;
    }
    static constexpr int NR = PART == 0 ? 5 * K0 - 3 : PART == 1 ? K0 + 1 : 2 * K0 - 2; // real rows
    static constexpr int NL = PART == 0 ? dev_lines(K0) : dev_lines_split(K0);          // lines of NL
    enum { UV, UW, VVUU, VW, VVWW, WWUU };
    __host__ __device__ static constexpr int k(int r) { return r < 2 ? 0 : 1 + (r - 2) / 5; }
    __host__ __device__ static constexpr int type(int r) { return r < 2 ? (r == 0 ? UW : WWUU) : (r - 2) % 5; }
    // row at forward position q (two per complex sequence), -1 = padding.  Rounded
    // twiddles leak a few 1e-8 of one row of a sequence into the other in FP32, alike in
    // every step.  At small a and g, psi weights uv and vw by ak, uw and uu by a and g only,
    // and the laminar profile makes uw and uu the larger rows: so uv and vw share a
    // sequence, and vw does not share uu's.  (State after 50 steps against FP64, with uv, uw /
    // vv - uu, vw / ... and now: M6 MM = 64, NN = 1024 6.4e-8 and 5.7e-8, NN = 512 5.1e-8 and
    // 4.7e-8, M6 2048^2 7.7e-8 and 6.9e-8; the advective form 6.0e-8, 6.3e-8 for the first
    // two.)  The three lines' worth of vw, vv - ww and vv - uu follow one another, so that
    // few accumulators are live.
    __host__ __device__ static constexpr int order(int q)
    {
        if (q >= NR) return -1;
        if (PART == 0) {
            constexpr int odd[] = {UV, VW, VVWW, VVUU, UW}, even[] = {UW, UV, VW, VVWW, VVUU};
            return q < 2 ? q : 2 + 5 * ((q - 2) / 5) + (((q - 2) / 5) % 2 ? even : odd)[(q - 2) % 5];
        }
        if (PART == 1) return q < 2 ? q : 2 + 5 * (q - 2) + UW;
        return 2 + 5 * (q / 2) + (PART == 2 ? (q & 1 ? VVUU : UV) : (q & 1 ? VVWW : VW));
    }
    // uses of row r: line, kind
    enum { ROW, G_ROW, UU_E, VW_E, VW_F, WW_E, WW_F }; // row, g row, and the multiples of DevMul
    __host__ __device__ static constexpr int nuse(int r) { return type(r) == VW || type(r) == VVWW ? 2 : 1; }
    __host__ __device__ static constexpr int use_line(int r, int u)
    {
        const int t = type(r);
        const bool e = (t == VW || t == VVWW) && u == 0; // the vw or ww share of DEV_E
        if (PART != 0 && e) return dev_lines(K0) + k(r) - 1;
        return dev_line(k(r)) + (t == UW ? DEV_UW : t == UV ? DEV_UV : t == VVUU || e ? DEV_E : DEV_F);
    }
    __host__ __device__ static constexpr int use_kind(int r, int u)
    {
        const int t = type(r);
        return t == WWUU ? G_ROW : t == VVUU ? UU_E : t == VW ? (u == 0 ? VW_E : VW_F) : t == VVWW ? (u == 0 ? WW_E : WW_F) : ROW;
    }
    // forward positions of the first and the last row of line L
    __host__ __device__ static constexpr int first(int L)
    {
        for (int q = 0; q < NR; q++)
            for (int u = 0; u < nuse(order(q)); u++)
                if (use_line(order(q), u) == L) return q;
        return -1;
    }
    __host__ __device__ static constexpr int last(int L)
    {
        int at = -1;
        for (int q = 0; q < NR; q++)
            for (int u = 0; u < nuse(order(q)); u++)
                if (use_line(order(q), u) == L) at = q;
        return at;
    }
};

template <int LOGNN> constexpr int zc_threads() { return (1 << LOGNN) > ZT ? (1 << LOGNN) : ZT; }

// Lane-group transforms where their registers fit (NN <= 512, and FP32 or
// the two-buffer form), with seven-entry pass tables; otherwise block-wide
// Stockham passes (ip_fft) with three-entry ones.
template <typename R, int LOGNN, bool PP> constexpr bool zc_wave() { return LOGNN <= 9 && (PP || sizeof(R) == 4); }
template <typename R, int LOGNN, bool PP> constexpr int zc_pw() { return zc_wave<R, LOGNN, PP>() ? 7 : 3; }
// LDS layout of the sequences: padded (lslot shift 4) for the FP32 lane-group
// transforms, XOR-swizzled otherwise (padding with shift 3 made FP64 k_zc 2 %
// slower at M4 1024^2)
template <typename R, int LOGNN, bool PP> constexpr int zc_ls() { return zc_wave<R, LOGNN, PP>() && sizeof(R) == 4 ? 4 : 0; }

// Sequence-granular forward batches: with one x-row per block, lane-group
// transforms and two buffers, a forward batch takes the next T/G (8)
// sequences in the order (pair q, phase b) -> 3 q + b, so that every lane
// group transforms; a pair whose three phases straddle two batches keeps its
// partial sums in registers.  Pair-granular batches of ZP pairs (3 ZP = 6
// sequences) leave two of the eight groups idle.  FP64 keeps batches of 6
// (its transforms are bound by LDS bandwidth, 16-byte values, and eight at
// once made FP64 k_zc 2 % slower at M4 1024^2 despite one batch in nine
// fewer; FP32 1 % faster), except that a tail of up to 2 sequences joins the
// last batch.
template <typename R, int LOGNN, bool PP> constexpr bool zc_sg()
{
    return PP && zc_wave<R, LOGNN, PP>() && zc_threads<LOGNN>() == (1 << LOGNN);
}
// forward sequences per batch (the last batch may take up to 8)
template <typename R> constexpr int zc_spb() { return sizeof(R) == 4 ? 8 : 6; }
// forward batches of NSF sequences, SPB a batch, a tail of at most 8 - SPB
// sequences joining the last full batch
template <int NSF, int SPB> constexpr int zc_nbf()
{
    const int nb = (NSF + SPB - 1) / SPB;
    return nb > 1 && NSF - (nb - 1) * SPB <= 8 - SPB ? nb - 1 : nb;
}
// sequences per buffer
template <typename R, int LOGNN, int ZP, bool PP> constexpr int zc_bseq()
{
    constexpr int NN = 1 << LOGNN, T = zc_threads<LOGNN>(), SEQ = T / NN * ZP * 3;
    constexpr int SPB = zc_sg<R, LOGNN, PP>() ? T / group_lanes<NN>() : SEQ;
    return SEQ > SPB ? SEQ : SPB;
}

// transform buffer(s), then the pass twiddle table of the NN-point
// transforms and the first NN entries of exp(2 pi i j/Q) (twq2 extends them)
template <typename R, int LOGNN, int ZP, bool PP> constexpr size_t zc_lds_bytes()
{
    constexpr int NN = 1 << LOGNN;
    constexpr int LPZ = lspan<NN, zc_ls<R, LOGNN, PP>()>();
    return sizeof(cplx_t<R>) * ((PP ? 2 : 1) * (size_t)zc_bseq<R, LOGNN, ZP, PP>() * LPZ +
                                ptw_size<NN, 1, zc_pw<R, LOGNN, PP>()>() + (size_t)NN);
}

// the pass of block row xt (XB x-rows) over the rows of Dev<K0, PART>
template <typename R, int K0, int PART, int LOGNN, int ZP, bool PP>
__device__ __forceinline__ void zc_pass(const Geo& g, int xt, const cplx_t<R>* __restrict__ U, cplx_t<R>* __restrict__ NL,
                                        const cplx_t<R>* __restrict__ twNN, const cplx_t<R>* __restrict__ twQ)
{
    using CT = cplx_t<R>;
    using FX = Dev<K0, PART>;
    using FR = FluxRows<K0>;
    constexpr int KK = 3 * K0 - 1;
    constexpr int NB = FX::NB;
    constexpr int NN = 1 << LOGNN;
    constexpr int T = zc_threads<LOGNN>();
    constexpr int XB = T / NN;
    constexpr int H = NN / 2;
    constexpr int NPI = (NB + 1) / 2;                 // inverse pairs: base lines 2p, 2p + 1
    constexpr int NBI = (NPI + ZP - 1) / ZP;
    constexpr int NR = FX::NR;
    constexpr int NPO = (NR + 1) / 2;                 // forward pairs: rows order(2p), order(2p + 1)
    constexpr int NBO = (NPO + ZP - 1) / ZP;
    constexpr int SEQ = XB * ZP * 3;
    constexpr int FT = XB * ZP * H / T;               // fold tasks per thread
    static_assert(FT * T == XB * ZP * H, "fold tasks must tile the block");
    extern __shared__ unsigned char smem_raw[];
    constexpr int LS = zc_ls<R, LOGNN, PP>(), LPZ = lspan<NN, LS>(); // sequence layout and span
    constexpr bool SG = zc_sg<R, LOGNN, PP>();
    constexpr int BSEQ = zc_bseq<R, LOGNN, ZP, PP>(); // sequences per buffer
    CT* bufA = reinterpret_cast<CT*>(smem_raw);       // [BSEQ][LPZ]: the sequences of a batch
    CT* bufB = bufA + (PP ? BSEQ * LPZ : 0);          // [BSEQ][LPZ]: those of the next batch (PP)
    constexpr int PW = zc_pw<R, LOGNN, PP>();
    CT* twNl = bufB + BSEQ * LPZ;                     // [ptw_size<NN, 1, PW>()] pass twiddles
    // buffer of batch k (inverse batches first, then forward ones)
    auto buf_of = [&](int k) { return (PP && (k & 1)) ? bufB : bufA; };
    // transforms of the first S sequences of b, in place, natural order in
    // and out; ends with a block barrier.  Lane-group transforms where their
    // registers fit (NN <= 512, and FP32 or the two-buffer form); otherwise
    // Stockham passes over the whole block (ip_fft, a barrier per half-pass).
    constexpr bool WAVE = zc_wave<R, LOGNN, PP>();
    auto transform = [&](auto sign, int S, CT* b, int t) {
        if constexpr (!WAVE) {
            ip_fft<CT, LOGNN, decltype(sign)::value, T, SEQ, true>(b, S, twNl, t);
            return;
        }
        constexpr int G = group_lanes<NN>(), PL = NN / G;
        const int gi = t / G, gl = t % G;
        if (gi < S) {
            CT* sq = b + gi * LPZ;
            CT v[PL];
            const int pg = lslot<LS>(gl);
            static_for<0, PL>([&](auto qi) { v[qi] = lsw<decltype(qi)::value * G, LS>(sq, pg); });
            group_fft<CT, LOGNN, decltype(sign)::value, true, PW, 1, 0, LS>(v, sq, gl, twNl);
            static_for<0, PL>([&](auto qi) { lsw<decltype(qi)::value * G, LS>(sq, pg) = v[qi]; });
        }
        __syncthreads();
    };
    static_assert(!WAVE || BSEQ * group_lanes<NN>() <= T, "one lane group per sequence");
    CT* twQl = twNl + ptw_size<NN, 1, PW>();          // [NN]: w^k, k < NN

    const int tid = threadIdx.x;
    const int xl = tid >> LOGNN, r = tid & (NN - 1);
    const int x0 = xt * XB;
    const int x = x0 + xl;
    const bool valid = x < g.P;
    const bool wide = g.NTs * (int)sizeof(CT) >= 64;
    // with one x-row per block the sequences of the valid pairs of a batch
    // come first, so a part-padding batch transforms only those
    auto nseq = [](int nv) { return XB == 1 ? 3 * nv : SEQ; };

    // fold task f of this thread: tau = tid + T f -> (row fx, pair fp, index fr);
    // its four values of the next batch are loaded while this one transforms
    CT pf[FT][4];
    auto prefetch = [&](int batch) {
#pragma unroll
        for (int f = 0; f < FT; f++) {
            const int tau = tid + T * f;
            const int fx = tau / (ZP * H), fp = (tau / H) % ZP, fr = tau % H;
            const int xg = x0 + fx;
            const int pr = batch * ZP + fp;
            const int r2 = fr == 0 ? H : NN - fr;
            const CT z{(R)0, (R)0};
            pf[f][0] = pf[f][1] = pf[f][2] = pf[f][3] = z;
            if (xg < g.P && pr < NPI) {
                // U[x][line][n] with KK lines of NN (uidx, with the flux form's sizes)
                const CT* u0 = U + ((size_t)(xg * KK + FX::base(2 * pr)) << LOGNN);
                pf[f][0] = u0[fr];
                pf[f][1] = u0[r2];
                if (2 * pr + 1 < NB) {
                    const CT* u1 = PART == 1 ? U + ((size_t)(xg * KK + FX::base(2 * pr + 1)) << LOGNN) : u0 + NN;
                    pf[f][2] = u1[fr];
                    pf[f][3] = u1[r2];
                }
            }
        }
    };

    R vb[3][KK];
    prefetch(0);
    ptw_fill<CT, LOGNN, 1, PW>(twNl, twNN, tid, T);
    for (int i = tid; i < NN; i += T) twQl[i] = twQ[i];
    __syncthreads();

    // In FP64, thread-derived indices are recomputed per batch from an opaque
    // copy of the thread index, so that the compiler does not hoist the LDS
    // addresses of every batch's passes into registers next to the point
    // values (hoisted, FP64 k_zc is 2 % slower at M4 1024^2).  The FP32
    // kernels have the registers to hold them (at most 119 VGPRs, no spills):
    // hoisted, they issue 9 % (NN = 512) to 22 % (NN = 1024) fewer VALU
    // instructions.
    auto opaque_tid = [] {
        int t = threadIdx.x;
        if constexpr (sizeof(R) == 8) asm volatile("" : "+v"(t));
        return t;
    };

    // A thread's fold tasks have one index fr, its output one r: where registers
    // allow, the twiddles of the folds and then of the unfolds are looked up once
    constexpr bool HT = PP && T % H == 0;
    CT tf[4];
    if constexpr (HT) {
        const int fr = tid % H, fm = fr == 0 ? H : NN - fr;
        tf[0] = twQl[fr];
        tf[1] = twQl[fm];
        tf[2] = twq2<R>(twQl, NN, 2 * fr);
        tf[3] = twq2<R>(twQl, NN, 2 * fm);
    }

    // ---- inverse z transforms of the base lines (c2r, +1) ----
    static_for<0, NBI>([&](auto bi) {
        constexpr int BN = decltype(bi)::value;
        constexpr int NV = NPI - BN * ZP < ZP ? NPI - BN * ZP : ZP; // valid pairs
        const int tid = opaque_tid();
        const int xl = tid >> LOGNN, r = tid & (NN - 1);
        CT* buf = buf_of(BN);
#pragma unroll
        for (int f = 0; f < FT; f++) {
            const int tau = tid + T * f;
            const int fx = tau / (ZP * H), fp = (tau / H) % ZP, fr = tau % H;
            if (XB == 1 && fp >= NV) continue;
            const int fm = fr == 0 ? H : NN - fr;
            CT* seq = buf + ((fx * ZP + fp) * 3) * LPZ;
            const CT one{(R)1, (R)0};
            zfold_bw<R, LS>(seq, 0, fr, NN, pf[f][0], pf[f][1], pf[f][2], pf[f][3], one, one);
            if constexpr (HT) {
                zfold_bw<R, LS>(seq + LPZ, 1, fr, NN, pf[f][0], pf[f][1], pf[f][2], pf[f][3], tf[0], tf[1]);
                zfold_bw<R, LS>(seq + 2 * LPZ, 2, fr, NN, pf[f][0], pf[f][1], pf[f][2], pf[f][3], tf[2], tf[3]);
            } else {
                zfold_bw<R, LS>(seq + LPZ, 1, fr, NN, pf[f][0], pf[f][1], pf[f][2], pf[f][3], twQl[fr], twQl[fm]);
                zfold_bw<R, LS>(seq + 2 * LPZ, 2, fr, NN, pf[f][0], pf[f][1], pf[f][2], pf[f][3],
                                twq2<R>(twQl, NN, 2 * fr), twq2<R>(twQl, NN, 2 * fm));
            }
        }
        if constexpr (BN + 1 < NBI) prefetch(BN + 1);
        __syncthreads();
        transform(std::integral_constant<int, +1>{}, nseq(NV), buf, tid);
        static_for<0, NV>([&](auto pi) {
            constexpr int p = decltype(pi)::value;
            constexpr int s1 = 2 * (BN * ZP + p);
#pragma unroll
            for (int b = 0; b < 3; b++) {
                const CT zv = buf[((xl * ZP + p) * 3 + b) * LPZ + lslot<LS>(r)];
                vb[b][FX::base(s1)] = zv.x;
                if constexpr (s1 + 1 < NB) vb[b][FX::base(s1 + 1)] = zv.y;
            }
        });
        // with one buffer the next batch overwrites this one's results
        if constexpr (!PP) __syncthreads();
    });

    // ---- products, forward z transforms (r2c, -1), line assembly ----
    const double gn = g.gamma * r, rgn = 1.0 / gn; // gamma n at the thread's output n = r
    const R lu = (R)g.cth, lw = (R)g.sth; // laminar u_1, w_1
    if constexpr (HT) {
        tf[0] = cconj(twQl[r]);
        tf[1] = cconj(twq2<R>(twQl, NN, 2 * r));
    }
    auto unfold_tw = [&](int b, int rv) { return HT ? tf[b - 1] : cconj(twq2<R>(twQl, NN, rv * b)); };
    constexpr int NLN = FX::NL;          // lines of NL
    CT acc[NLN];
    // line assembly of the two rows q1, q1 + 1 of a forward pair from their
    // transforms X: each row's terms go into the accumulators of its lines,
    // and a line is stored after its last row
    auto assemble = [&](auto q1c, const CT* X, CT* nlr, size_t nls) {
        constexpr int q1 = decltype(q1c)::value;
        static_for<0, 2>([&](auto hi) {
            constexpr int q = q1 + decltype(hi)::value;
            constexpr int row = FX::order(q);
            if constexpr (row >= 0) {
                const CT xs = X[decltype(hi)::value];
                static_for<0, FX::nuse(row)>([&](auto ui) {
                    constexpr int u = decltype(ui)::value;
                    constexpr int L = FX::use_line(row, u), kind = FX::use_kind(row, u);
                    constexpr int k = FX::k(row);
                    CT term = xs;
                    if constexpr (kind == FX::G_ROW) term = cscale(xs, (R)gn);
                    else if constexpr (kind != FX::ROW) {
                        const DevMul<R> m = dev_mul<R>(gn, rgn, ak1_of(k, g.beta));
                        if constexpr (kind == FX::VW_E) term = CT{xs.y * m.e, -(xs.x * m.e)};
                        else if constexpr (kind == FX::VW_F) term = CT{-(xs.y * m.h), xs.x * m.h};
                        else if constexpr (kind == FX::UU_E) term = cscale(xs, m.ak);
                        else if constexpr (kind == FX::WW_E) term = cscale(xs, m.far ? -m.ak : (R)0);
                        else term = cscale(xs, m.f);
                    }
                    if constexpr (FX::first(L) == q) acc[L] = term;
                    else acc[L] = cadd(acc[L], term);
                    if constexpr (FX::last(L) == q) {
                        if (valid) st_piece(nlr + L * nls, acc[L], wide);
                    }
                });
            }
        });
    };
    if constexpr (SG) {
        constexpr int SPB = zc_spb<R>();             // sequences per forward batch
        static_assert(T / group_lanes<NN>() >= 8, "a batch of up to 8 sequences");
        // forward sequences: pair q, phase b at 3 q + b.  With an odd number
        // of rows the last pair holds one row, whose three phases take two
        // sequences (phases 0 and 1 as the real and imaginary parts of the
        // first, phase 2 in the second): M4's 17 rows are 26 sequences
        // instead of 27 (FP64: 4 batches instead of 5)
        constexpr bool LONE = NR % 2 == 1;
        constexpr int QL = NPO - 1;                  // the last pair
        constexpr int NSF = 3 * NPO - (LONE ? 1 : 0);
        constexpr int NBF = zc_nbf<NSF, SPB>();
        CT X[2];                                      // transforms of the current pair's two rows
        static_for<0, NBF>([&](auto ri) {
            constexpr int RD = decltype(ri)::value;
            constexpr int J0 = RD * SPB, J1 = RD == NBF - 1 ? NSF : J0 + SPB;
            const int tid = opaque_tid();
            const int r = tid & (NN - 1); // one x-row per block
            const int rm = (NN - r) & (NN - 1);
            CT* buf = buf_of(NBI + RD);
            CT* nlr = NL + ((((size_t)(r >> g.lgNS) * NLN * g.P) + x0) << g.lgNS) + (r & (g.NTs - 1));
            const size_t nls = (size_t)g.P << g.lgNS;
#pragma unroll
            for (int b = 0; b < 3; b++)
#pragma unroll
                for (int sl = 0; sl < NB; sl++) asm volatile("" : "+v"(vb[b][FX::base(sl)]));
            static_for<J0, J1>([&](auto ji) {
                constexpr int j = decltype(ji)::value, q = j / 3, b = j % 3;
                constexpr int r1 = FX::order(2 * q), r2 = FX::order(2 * q + 1);
                R v1 = (R)0, v2 = (R)0;
                if constexpr (LONE && q == QL) { // b = 0: phases 0 and 1; b = 1: phase 2
                    v1 = FR::template row<r1>(vb[2 * b], lu, lw);
                    if constexpr (b == 0) v2 = FR::template row<r1>(vb[1], lu, lw);
                } else {
                    if constexpr (r1 >= 0) v1 = FR::template row<r1>(vb[b], lu, lw);
                    if constexpr (r2 >= 0) v2 = FR::template row<r2>(vb[b], lu, lw);
                }
                buf[(j - J0) * LPZ + lslot<LS>(r)] = CT{v1, v2};
            });
            __syncthreads();
            transform(std::integral_constant<int, -1>{}, J1 - J0, buf, tid);
            static_for<J0, J1>([&](auto ji) {
                constexpr int j = decltype(ji)::value, q = j / 3, b = j % 3;
                const CT zn = buf[(j - J0) * LPZ + lslot<LS>(r)];
                const CT zm = buf[(j - J0) * LPZ + lslot<LS>(rm)];
                const CT F1 = CT{zn.x + zm.x, zn.y - zm.y};
                const CT F2 = CT{zn.y + zm.y, zm.x - zn.x};
                if constexpr (LONE && q == QL) {
                    if constexpr (b == 0) { // phase 0 (F1) and phase 1 (F2) of the one row
                        X[0] = cadd(F1, cmul(F2, unfold_tw(1, r)));
                        X[1] = CT{(R)0, (R)0};
                    } else { // phase 2
                        X[0] = cadd(X[0], cmul(F1, unfold_tw(2, r)));
                        assemble(std::integral_constant<int, 2 * q>{}, X, nlr, nls);
                    }
                } else {
                    if constexpr (b == 0) {
                        X[0] = F1;
                        X[1] = F2;
                    } else {
                        const CT w = unfold_tw(b, r);
                        X[0] = cadd(X[0], cmul(F1, w));
                        X[1] = cadd(X[1], cmul(F2, w));
                    }
                    if constexpr (b == 2) assemble(std::integral_constant<int, 2 * q>{}, X, nlr, nls);
                }
            });
        });
        return;
    }
    static_for<0, NBO>([&](auto ri) {
        constexpr int RD = decltype(ri)::value;
        constexpr int NV = NPO - RD * ZP < ZP ? NPO - RD * ZP : ZP; // valid output pairs
        const int tid = opaque_tid();
        const int xl = tid >> LOGNN, r = tid & (NN - 1);
        CT* buf = buf_of(NBI + RD);
        // this thread's element of NL line L is nlr[L * nls] (nidx with the
        // flux form's lines): one base per batch instead of the full
        // index per store
        CT* nlr = NL + ((((size_t)(r >> g.lgNS) * NLN * g.P) + (x0 + xl)) << g.lgNS) + (r & (g.NTs - 1));
        const size_t nls = (size_t)g.P << g.lgNS;
        // the base values pass through an empty asm per batch: products shared
        // by rows of different batches are formed again in each batch instead
        // of being computed once and held in registers across all of them
#pragma unroll
        for (int b = 0; b < 3; b++)
#pragma unroll
            for (int sl = 0; sl < NB; sl++) asm volatile("" : "+v"(vb[b][FX::base(sl)]));
        static_for<0, NV>([&](auto pi) {
            constexpr int p = decltype(pi)::value;
            constexpr int q1 = 2 * (RD * ZP + p);
            constexpr int r1 = FX::order(q1), r2 = FX::order(q1 + 1);
#pragma unroll
            for (int b = 0; b < 3; b++) {
                R v1 = (R)0, v2 = (R)0;
                if constexpr (r1 >= 0) v1 = FR::template row<r1>(vb[b], lu, lw);
                if constexpr (r2 >= 0) v2 = FR::template row<r2>(vb[b], lu, lw);
                buf[((xl * ZP + p) * 3 + b) * LPZ + lslot<LS>(r)] = CT{v1, v2};
            }
        });
        __syncthreads();
        transform(std::integral_constant<int, -1>{}, nseq(NV), buf, tid);
        static_for<0, NV>([&](auto pi) {
            constexpr int p = decltype(pi)::value;
            constexpr int q1 = 2 * (RD * ZP + p);
            const int rm = (NN - r) & (NN - 1);
            CT X[2] = {CT{(R)0, (R)0}, CT{(R)0, (R)0}};
#pragma unroll
            for (int b = 0; b < 3; b++) {
                const CT zn = buf[((xl * ZP + p) * 3 + b) * LPZ + lslot<LS>(r)];
                const CT zm = buf[((xl * ZP + p) * 3 + b) * LPZ + lslot<LS>(rm)];
                const CT F1 = CT{zn.x + zm.x, zn.y - zm.y};
                const CT F2 = CT{zn.y + zm.y, zm.x - zn.x};
                if (b == 0) {
                    X[0] = F1;
                    X[1] = F2;
                } else {
                    const CT w = unfold_tw(b, r);
                    X[0] = cadd(X[0], cmul(F1, w));
                    X[1] = cadd(X[1], cmul(F2, w));
                }
            }
            assemble(std::integral_constant<int, q1>{}, X, nlr, nls);
        });
        if constexpr (!PP) __syncthreads();
    });
}

template <typename R, int K0, int LOGNN, int ZP, int WAVES, bool PP>
__global__ __launch_bounds__(zc_threads<LOGNN>(), WAVES) void k_zc(Batch bt, const cplx_t<R>* __restrict__ U,
                                                                   cplx_t<R>* __restrict__ NL,
                                                                   const cplx_t<R>* __restrict__ twNN,
                                                                   const cplx_t<R>* __restrict__ twQ)
{
    const Geo g = bt.geo[blockIdx.z];
    zc_pass<R, K0, 0, LOGNN, ZP, PP>(g, xcd_tile(blockIdx.x, gridDim.x), U + blockIdx.z * bt.u_stride,
                                     NL + blockIdx.z * bt.nl_stride, twNN, twQ);
}

// Rows of 1024 points in FP64: the points of a row hold more base values (M6:
// 418 KB) than the registers of a block can keep beside its transforms, so three
// blocks take the row, one for each pair of velocity components (Dev, PART 1 to
// 3: 12, 11 and 11 base lines of M6).  They run back to back on one XCD (block B
// on XCD B % 8; there part (B / 8) % 3 of row B / 24, each XCD a contiguous run
// of rows) and read the row's U lines through its L2 once.  The 34 inverse line
// transforms instead of 17 cost less than what the phase-sequential advective
// kernel pays for reading and adding three partial sums of NL in memory.
template <typename R, int K0, int LOGNN, int ZP>
__global__ __launch_bounds__(zc_threads<LOGNN>(), 4) void k_zc3(Batch bt, const cplx_t<R>* __restrict__ U,
                                                                cplx_t<R>* __restrict__ NL,
                                                                const cplx_t<R>* __restrict__ twNN,
                                                                const cplx_t<R>* __restrict__ twQ)
{
    const Geo g = bt.geo[blockIdx.z];
    U += blockIdx.z * bt.u_stride;
    NL += blockIdx.z * bt.nl_stride;
    const int idx = blockIdx.x >> 3, nb = gridDim.x / 3, part = idx % 3;
    const int xt = (blockIdx.x & 7) * (nb >> 3) + idx / 3;
    if (part == 0) zc_pass<R, K0, 1, LOGNN, ZP, false>(g, xt, U, NL, twNN, twQ);
    else if (part == 1) zc_pass<R, K0, 2, LOGNN, ZP, false>(g, xt, U, NL, twNN, twQ);
    else zc_pass<R, K0, 3, LOGNN, ZP, false>(g, xt, U, NL, twNN, twQ);
}
