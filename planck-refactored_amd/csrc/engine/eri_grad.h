// eri_grad.h — two-electron part of the nuclear gradient on the device.
//
// First derivatives of the contracted Cartesian ERIs (the shift rule of
// src/integrals/os.cpp:1296-1420) contracted on the fly with the two-particle
// density of the closed- or open-shell determinant,
//   Gamma_ijkl = 2 Pj_ij Pj_kl - kx (Pk1_ik Pk1_jl + Pk2_ik Pk2_jl),
// into dE2/dR for the centre of every shell, E2 = 1/4 sum Gamma_ijkl (ij|kl)
// (the ERI loop of src/gradient/gradient.cpp:209-232 with its permutation
// rule, gradient.cpp:70-118).
//
// Every ordered pair of shell pairs is visited once and differentiated on its
// bra only: the derivatives of (ab|cd) on C and D are those of (cd|ab) on its
// bra, and eight-fold symmetry leaves, for every ordered (bra, ket),
//   2 d_bra d_ket sum_abcd Gs d(ab|cd)/dR_A  (and R_B),   d = 1/2 for a shell with itself,
//   Gs = 2 Pj_ab Pj_cd - kx/2 (Pk_ac Pk_bd + Pk_ad Pk_bc)  (summed over Pk1, Pk2).
// The bra of a wave is fixed, so its six sums stay in registers over all kets of
// a work item: six atomics per item.  A long contraction is cut along the bra's
// primitives (the sums are linear in them), so that no item is a serial chain
// of thousands of primitive quartets.
//
// Layout as in eri_rows.h: one wave owns QW quartets of one bra at a time.
//   Phase A, lane = (quartet, root, axis): 2-D integrals I[e][f], e <= la+lb+1,
//   f <= lc+ld, the A -> B transfer, and per (a, b) three rows over f:
//     G,  dA = 2 alpha G[a+1][b] - a G[a-1][b],  dB = 2 beta G[a][b+1] - b G[a][b-1]
//   (alpha, beta the primitive exponents on A and B), to LDS.
//   Phase B, lane = row (a, b): sum_f W_f dAx Gy Gz and the like, W the row of Gs
//   carried from (cd) back to |f0] by the transposed C -> D transfer, in
//   registers from the densities of the quartet.
// Work per primitive quartet, root, row and f: six products and six FMAs, nine
// rows of LDS: bound by LDS and VALU alike; small molecules by the longest chain
// of primitives.  n-C3H8 / cc-pVDZ (85 functions) 3.8 ms per gradient, 11.4 ms
// without cutting the bra's primitives; 1213 ms with one quartet per wave, every
// factor and component through LDS and a serial chain of up to 6561 primitive
// quartets.
#pragma once

#include "eri_rows.h"

namespace pk {

struct GradArgs {
    const int *__restrict__ item_bra;    // work items: bra pair, and count kets from order[start]
    const int *__restrict__ item_start;
    const int *__restrict__ item_count;
    const int *__restrict__ item_prim;   // bra primitives [p & 0xffff, p >> 16)
    const int *__restrict__ order;       // pairs by class, ordering group and Schwarz bound
    const PairDev *__restrict__ pairs;
    const PrimDev *__restrict__ prims;
    const double *__restrict__ palpha;   // exponent on the pair's first shell, per primitive pair
    const double *__restrict__ hz;       // 1/(2 zeta) per primitive pair
    const int *__restrict__ pair_sh;     // [2 * npairs]: first and second shell of each pair
    const double *__restrict__ Pj;       // densities scaled by component norms, internal order
    const double *__restrict__ Pk1;
    const double *__restrict__ Pk2;      // two exchange densities only
    const double *__restrict__ Q;
    double *g;  // [3 * nshells] dE2/dR per shell centre
    double tol, kx;
    int nb;
    int nitems;
};

// Shape of one class: RC row chunks (blockIdx.y) of RN rows, QW quartets per wave.
template <int LA, int LB, int LC, int LD>
struct GradCls {
    using K = Cls<LA, LB, LC, LD>;
    static constexpr int E = K::E, F = K::F, NF = K::NF, NAB = K::NAB, NCD = K::NCD;
    static constexpr int NR = (K::L + 1) / 2 + 1;
    static constexpr int RC = NAB > 64 ? 2 : 1, RN = (NAB + RC - 1) / RC;
    static constexpr int RL = (F + 1) | 1;                              // doubles of one row of one axis, odd (banks)
    static constexpr int NGP = ((LA + 1) * (LB + 1) * 3 * RL) | 1;      // three kinds of rows
    static constexpr int QW = [] {
        const int q = 64 / RN, qa = 64 / (3 * NR);
        return q < qa ? q : qa;
    }();
    static constexpr int NX = (K::NA + K::NB) * (K::NC + K::ND);
    static constexpr int pe(int nk) { return 2 * NCD + nk * NX; }       // staged densities of a quartet
    static constexpr int gd(int nk) {
        const int f = QW * 3 * NR * NGP, j = QW * pe(nk);
        return f > j ? f : j;
    }
};

// Rows G, dA, dB of one axis for every (a, b), into g[((a (LB+1) + b) 3 + kind) RL + f].
template <int LA, int LB, int F, int RL>
__device__ __forceinline__ void axis_grad(double seed, double C00, double D00, double B00, double B10, double B01,
                                          double AB, double a2, double b2, double *g) {
    constexpr int E = LA + LB + 1;
    double I[E + 1][F + 1];
    I[0][0] = seed;
    sfor<1, E + 1>([&](auto e_) {
        constexpr int e = PK_CI(e_);
        I[e][0] = C00 * I[e - 1][0];
        if constexpr (e >= 2) I[e][0] = fma((double)(e - 1) * B10, I[e - 2][0], I[e][0]);
    });
    sfor<1, F + 1>([&](auto f_) {
        constexpr int f = PK_CI(f_);
        I[0][f] = D00 * I[0][f - 1];
        if constexpr (f >= 2) I[0][f] = fma((double)(f - 1) * B01, I[0][f - 2], I[0][f]);
        sfor<1, E + 1>([&](auto e_) {
            constexpr int e = PK_CI(e_);
            double t = fma(D00, I[e][f - 1], (double)e * B00 * I[e - 1][f - 1]);
            if constexpr (f >= 2) t = fma((double)(f - 1) * B01, I[e][f - 2], t);
            I[e][f] = t;
        });
    });
    // per f: (a|b) for b ascending, two columns of b at a time
    sfor<0, F + 1>([&](auto f_) {
        constexpr int f = PK_CI(f_);
        double c[E + 1], p[E + 1];  // (a|b) and (a|b-1)
        sfor<0, E + 1>([&](auto e_) {
            c[PK_CI(e_)] = I[PK_CI(e_)][f];
            p[PK_CI(e_)] = 0.0;
        });
        sfor<0, LB + 1>([&](auto b_) {
            constexpr int b = PK_CI(b_);
            sfor<0, LA + 1>([&](auto a_) {
                constexpr int a = PK_CI(a_);
                double *o = g + (a * (LB + 1) + b) * 3 * RL + f;
                o[0] = c[a];
                double da = a2 * c[a + 1];
                if constexpr (a > 0) da = fma(-(double)a, c[a - 1], da);
                double db = b2 * fma(AB, c[a], c[a + 1]);
                if constexpr (b > 0) db = fma(-(double)b, p[a], db);
                o[RL] = da;
                o[2 * RL] = db;
            });
            if constexpr (b < LB)
                sfor<0, E - b>([&](auto a_) {
                    constexpr int a = PK_CI(a_);
                    p[a] = c[a];
                    c[a] = fma(AB, c[a], c[a + 1]);
                });
        });
    });
}

// Transpose of hrr_step: w over (a levels LA..LA+LB-K) x (b level K), the sum of
// out (a, b) of levels (LA, LB) carried back.
template <int LA, int LB, int K>
__device__ __forceinline__ void hrr_adjoint(const double (&out)[ncart(LA) * ncart(LB)], const double ab[3],
                                            double (&w)[nlev(LA, LA + LB - K) * ncart(K)]) {
    if constexpr (K == LB) {
        sfor<0, ncart(LA) * ncart(LB)>([&](auto i_) { w[PK_CI(i_)] = out[PK_CI(i_)]; });
    } else {
        constexpr int NK = ncart(K), NK1 = ncart(K + 1);
        constexpr int NAL = nlev(LA, LA + LB - K - 1);
        double nxt[NAL * NK1];
        hrr_adjoint<LA, LB, K + 1>(out, ab, nxt);
        sfor<0, nlev(LA, LA + LB - K) * NK>([&](auto i_) { w[PK_CI(i_)] = 0.0; });
        sfor<0, NK1>([&](auto bp_) {
            constexpr int bp = PK_CI(bp_);
            constexpr int bx = cart_x(K + 1, bp), by = cart_y(K + 1, bp), bz = cart_z(K + 1, bp);
            constexpr int ax = build_axis(bx, by, bz);
            constexpr int b = cart_index(bx - (ax == 0), by - (ax == 1), bz - (ax == 2));
            sfor<0, NAL>([&](auto ia_) {
                constexpr int ia = PK_CI(ia_);
                constexpr int la = flat_level(LA, ia), ka = flat_k(LA, ia);
                constexpr int iap = flat(LA, cart_x(la, ka) + (ax == 0), cart_y(la, ka) + (ax == 1),
                                         cart_z(la, ka) + (ax == 2));
                w[ia * NK + b] = fma(ab[ax], nxt[ia * NK1 + bp], w[ia * NK + b]);
                w[iap * NK + b] += nxt[ia * NK1 + bp];
            });
        });
    }
}

// NK exchange densities.  One wave per workgroup and work item.
template <int LA, int LB, int LC, int LD, int NK>
__global__ __launch_bounds__(64) void k_grad(GradArgs a) {
    using K = Cls<LA, LB, LC, LD>;
    using S = GradCls<LA, LB, LC, LD>;
    constexpr int NA = K::NA, NB = K::NB, NC = K::NC, ND = K::ND, NAB = K::NAB, NCD = K::NCD, NF = K::NF, NR = S::NR;
    constexpr int QW = S::QW, RN = S::RN, RL = S::RL, NGP = S::NGP, NCX = NC + ND;
    constexpr int PE = S::pe(NK), EPL = (QW * PE + 63) / 64;
    extern __shared__ double smem[];
    double *G = smem;
    const int item = blockIdx.x;
    if (item >= a.nitems) return;
    const int lane = threadIdx.x;
    const int nb = a.nb;
    const int bra = uload(a.item_bra + item);
    const int kbeg = uload(a.item_start + item);
    const int kend = kbeg + uload(a.item_count + item);
    const PairDev *pbp = a.pairs + bra;
    const int bprim = uload(a.item_prim + item);
    const int bf0 = uload(&pbp->f0), bf1 = uload(&pbp->f1), np = (bprim >> 16) - (bprim & 0xffff);
    const int bpo = uload(&pbp->prim_off) + (bprim & 0xffff);
    const double bqmin = uload(&pbp->qmin);
    const double bdeg = uload(&pbp->diag) ? 1.0 : 2.0;  // 2 d

    // phase A role: slot, root, axis
    const int sa = lane / (3 * NR), ra = lane - sa * 3 * NR;
    const int r_a = ra / 3, ax = ra - 3 * r_a;
    const bool live_a = sa < QW;
    double *Ga = G + (live_a ? (sa * 3 * NR + ra) : 0) * NGP;
    const double ABq = sel3d(ax, uload(&pbp->ab[0]), uload(&pbp->ab[1]), uload(&pbp->ab[2]));
    const int cw = ((ax == 1 ? NR : 0) + r_a) * (PK_RYS_DEG + 1);  // this lane's series: node (axes 0, 2) or weight (1)
    const double lim = ax == 1 ? pk_rys_aw[pk_rys_abase[NR] + r_a] : pk_rys_ax2[pk_rys_abase[NR] + r_a];

    // phase B role: slot and row (a, b)
    const int row0 = S::RC > 1 ? (int)blockIdx.y * RN : 0;
    const int sl = lane / RN;
    const bool live = sl < QW && row0 + lane - sl * RN < NAB;
    const int sb = live ? sl : 0, row = live ? row0 + lane - sl * RN : 0;
    const int ia = row / NB, ib = row - ia * NB;
    int ro[3];
    {
        auto ex = [](int l, int i, int *x) {  // exponents of component i
            int lx = l;
            while (i > l - lx) {
                i -= l - lx + 1;
                --lx;
            }
            x[0] = lx;
            x[2] = i;
            x[1] = l - lx - i;
        };
        int xa[3], xb[3];
        ex(LA, ia, xa);
        ex(LB, ib, xb);
        sfor<0, 3>([&](auto q_) {
            constexpr int q = PK_CI(q_);
            ro[q] = sb * 3 * NR * NGP + q * NGP + (xa[q] * (LB + 1) + xb[q]) * 3 * RL;
        });
    }
    const size_t abi = (size_t)(bf0 + ia) * nb + bf1 + ib;
    const double Pab = 2.0 * a.Pj[abi], Qab = a.Q[abi];
    double gA[3] = {0.0, 0.0, 0.0}, gB[3] = {0.0, 0.0, 0.0};

    for (int g0 = kbeg; g0 < kend; g0 += QW) {
        const int idb = a.order[min(g0 + sb, kend - 1)];
        const PairDev *pk = a.pairs + idb;
        const int cf0 = pk->f0, df0 = pk->f1;
        const double kqmin = pk->qmin;
        const double cd[3] = {pk->ab[0], pk->ab[1], pk->ab[2]};
        double deg = pk->diag ? 0.5 * bdeg : bdeg;
        if (!live || g0 + sb >= kend) deg = 0.0;
        const PairDev *pa = a.pairs + a.order[min(g0 + (live_a ? sa : 0), kend - 1)];
        const int nqa = live_a && g0 + sa < kend ? pa->nprim : 0;
        const int qoff = nqa > 0 ? pa->prim_off : 0;
        // densities of the group's quartets, [slot][PE], over the factors: Q_cd,
        // Pj_cd, then the rows a and b of the exchange densities at columns c, d
        wave_fence();
        sfor<0, EPL>([&](auto i_) {
            constexpr int i = PK_CI(i_);
            const int e = min(lane + 64 * i, QW * PE - 1);
            const int s = e / PE, t = e - s * PE;
            const int c0 = __shfl(cf0, s * RN, 64), d0 = __shfl(df0, s * RN, 64);
            const double *M;
            size_t off;
            if (t < 2 * NCD) {
                const int j = t < NCD ? t : t - NCD;
                M = t < NCD ? a.Q : a.Pj;
                off = elem(c0 + j / ND, nb, d0 + j % ND);
            } else {
                int x = t - 2 * NCD;
                const bool second = NK == 2 && x >= S::NX;
                if (second) x -= S::NX;
                M = second ? a.Pk2 : a.Pk1;
                const int r = x / NCX, col = x - r * NCX;
                off = elem(r < NA ? bf0 + r : bf1 + r - NA, nb, col < NC ? c0 + col : d0 + col - NC);
            }
            const double x = M[off];
            if (64 * (i + 1) <= QW * PE || lane + 64 * i < QW * PE) G[lane + 64 * i] = x;
        });
        wave_fence();
        // W_f: the row of Gs over (cd), carried back to |f0]
        double W[NF];
        {
            const double *D = G + sb * PE;
            double w[NCD];
            sfor<0, NCD>([&](auto j_) {
                constexpr int j = PK_CI(j_), c = j / ND, d = j % ND;
                double x = 0.0;
                sfor<0, NK>([&](auto s_) {
                    const double *Xa = D + 2 * NCD + PK_CI(s_) * S::NX + ia * NCX;
                    const double *Xb = D + 2 * NCD + PK_CI(s_) * S::NX + (NA + ib) * NCX;
                    x = fma(Xa[c], Xb[NC + d], fma(Xa[NC + d], Xb[c], x));
                });
                const bool pass = bqmin * kqmin >= a.tol || Qab * D[j] >= a.tol;
                w[j] = (pass ? deg : 0.0) * fma(Pab, D[NCD + j], -0.5 * a.kx * x);
                if constexpr (j % 16 == 15) __builtin_amdgcn_sched_barrier(0);
            });
            hrr_adjoint<LC, LD, 0>(w, cd, W);
        }
        // primitive quartets (kq, kp)
        bool more = np > 0 && __any(nqa > 0);  // a pair can have lost all its primitives to the screening
        double qz = 1.0, qx = 0.0, qy = 0.0, qw = 0.0, hq = 0.0, qpa = 0.0, qkc = 0.0;
        for (int kq = 0, kp = 0; more;) {
            if (kp == 0) {
                const int qi = nqa > 0 ? qoff + min(kq, nqa - 1) : 0;
                const PrimDev *qp = a.prims + qi;
                qz = qp->zeta;
                qx = qp->p[0];
                qy = qp->p[1];
                qw = qp->p[2];
                qpa = qp->pa[ax];
                qkc = kq < nqa ? qp->kc : 0.0;
                hq = a.hz[qi];
            }
            const PrimDev *pp = a.prims + (bpo + kp);
            const double pz = uload(&pp->zeta), hp = uload(a.hz + bpo + kp);
            const double a2 = 2.0 * uload(a.palpha + bpo + kp), b2 = 2.0 * pz - a2;
            const double rs = rsqrt_nr(pz + qz), inv_de = rs * rs;
            const double x = uload(&pp->p[0]) - qx, y = uload(&pp->p[1]) - qy, z = uload(&pp->p[2]) - qw;
            const double T = pz * qz * inv_de * fma(x, x, fma(y, y, z * z));
            double val;
            {
                const bool small = T < pk_rys_tmax[NR];
                const double Tc = small ? T : 0.0;
                const int i = (int)Tc;
                val = cheb<double>(pk_rys_coef + pk_rys_base[NR] + i * (2 * NR * (PK_RYS_DEG + 1)) + cw,
                                   2.0 * (Tc - (double)i) - 1.0);
                if (!small) {
                    const double s = rsqrt_nr(T);
                    val = lim * (ax == 1 ? s : s * s);
                }
            }
            const double u = __shfl(val, lane - ax, 64);
            const double w = __shfl(val, lane - ax + 1, 64);
            wave_fence();  // the staged densities, or the rows of the previous primitive quartet, have been read
            if (live_a) {
                const double roz = qz * inv_de, roe = pz * inv_de;
                const double PQa = sel3d(ax, x, y, z);
                const double ppa = sel3d(ax, uload(&pp->pa[0]), uload(&pp->pa[1]), uload(&pp->pa[2]));
                axis_grad<LA, LB, S::F, RL>(ax == 0 ? uload(&pp->kc) * qkc * rs * w : 1.0, fma(-u * roz, PQa, ppa),
                                            fma(u * roe, PQa, qpa), 0.5 * inv_de * u, hp * (1.0 - roz * u),
                                            hq * (1.0 - roe * u), ABq, a2, b2, Ga);
            }
            wave_fence();
            if (++kp == np) {
                kp = 0;
                ++kq;
                more = __any(kq < nqa);
            }
#pragma unroll 1
            for (int r = 0; r < NR; ++r) {
                const double *Gr = G + r * 3 * NGP;
                double v[3][3][S::F + 1];  // [axis][G, dA, dB][f]
                sfor<0, 9>([&](auto q_) {
                    constexpr int q = PK_CI(q_) / 3, k = PK_CI(q_) % 3;
                    const double *src = Gr + ro[q] + k * RL;
                    sfor<0, S::F + 1>([&](auto i_) { v[q][k][PK_CI(i_)] = src[PK_CI(i_)]; });
                });
                sfor<0, NF>([&](auto j_) {
                    constexpr int j = PK_CI(j_);
                    constexpr int lf = flat_level(LC, j), kf = flat_k(LC, j);
                    constexpr int fx = cart_x(lf, kf), fy = cart_y(lf, kf), fz = cart_z(lf, kf);
                    const double wx = W[j] * v[0][0][fx], yz = W[j] * v[1][0][fy] * v[2][0][fz];
                    const double xz = wx * v[2][0][fz], xy = wx * v[1][0][fy];
                    gA[0] = fma(v[0][1][fx], yz, gA[0]);
                    gA[1] = fma(v[1][1][fy], xz, gA[1]);
                    gA[2] = fma(v[2][1][fz], xy, gA[2]);
                    gB[0] = fma(v[0][2][fx], yz, gB[0]);
                    gB[1] = fma(v[1][2][fy], xz, gB[1]);
                    gB[2] = fma(v[2][2][fz], xy, gB[2]);
                });
            }
        }
    }
    const int sA = uload(a.pair_sh + 2 * bra), sB = uload(a.pair_sh + 2 * bra + 1);
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        const double x = wave_sum(live ? gA[q] : 0.0), y = wave_sum(live ? gB[q] : 0.0);
        if (lane == 0) {
            unsafeAtomicAdd(&a.g[3 * sA + q], x);
            unsafeAtomicAdd(&a.g[3 * sB + q], y);
        }
    }
}

}  // namespace pk
