// eri_generic.h — cooperative shell-quartet kernel for any class up to (ff|ff).
//
// One 64-lane workgroup owns one contracted shell quartet at a time; the class
// (la, lb, lc, ld) is a runtime value, so one compiled kernel serves every
// ERI-output request (Schwarz table, ERI tensor) and the autotuner's alternative
// of a per-lane Rys class.
//
// Per primitive quartet: lanes r < n evaluate the Rys roots; lanes t < 3n build
// the 2-D integrals of root t/3 and axis t%3 into LDS; all lanes then form the
// transferred 1-D factors G[a][b][c][d] (closed-form transfers
//   (a|b) = sum_k C(b,k) (A-B)^(b-k) (a+k|0),  (c|d) likewise with C-D)
// and add sum_r Gx Gy Gz for their share of the (ab|cd) components into LDS
// accumulators.  J/K digestion reduces each output element
// in one lane (no atomic contention inside the quartet), then FP64 atomics.
// Reference semantics as in eri_prim.h (rys.cpp:250-485, os.cpp:837-879).
#pragma once

#include "eri_prim.h"

namespace pk {

constexpr int GEN_MAX_L = 3;  // per shell
constexpr int GEN_NR = 7;     // roots for L <= 12; also the 2-D extent E + 1 <= 7

struct GenArgs {
    // JK mode: wave lists of one class (as JKArgs); ERI mode: explicit quartets
    const int *__restrict__ wave_bra;
    const int *__restrict__ wave_start;
    const int *__restrict__ wave_count;
    const int *__restrict__ wave_mol;
    const int *__restrict__ kets;
    const long long *__restrict__ mol_off;  // JK mode: packed matrices per molecule
    const int *__restrict__ mol_nb;
    const int *__restrict__ qbra;  // ERI mode
    const int *__restrict__ qket;
    const PairDev *__restrict__ pairs;
    const PrimDev *__restrict__ prims;
    const double *__restrict__ hz;   // 1/(2 zeta) per primitive pair
    const double *__restrict__ P;    // density, scaled
    const double *__restrict__ Q;
    double *A;
    double *B;
    double *out;  // ERI mode: [nitems][NA NB NC ND]
    double tol;
    int nitems;  // waves (JK) or quartets (ERI)
    int la, lb, lc, ld;
    int eri_mode;
};

// C(n, k) for 0 <= k <= n <= 3
__device__ __forceinline__ double binom(int n, int k) {
    return (n == 3 && (k == 1 || k == 2)) ? 3.0 : ((n == 2 && k == 1) ? 2.0 : 1.0);
}

__device__ __forceinline__ double sel3(int ax, double x, double y, double z) {
    return ax == 0 ? x : (ax == 1 ? y : z);
}

// Rys rule with a runtime root count (the kernels' tables)
__device__ __forceinline__ void rys_root_rt(int n, double T, int r, double &u, double &w) {
    if (T >= pk_rys_tmax[n]) {
        const double s = rsqrt_nr(T);
        u = pk_rys_ax2[pk_rys_abase[n] + r] * s * s;
        w = pk_rys_aw[pk_rys_abase[n] + r] * s;
    } else {
        const int i = (int)T;
        const double x = 2.0 * (T - (double)i) - 1.0;
        const double *c = pk_rys_coef + pk_rys_base[n] + i * (2 * n * (PK_RYS_DEG + 1));
        u = cheb(c + r * (PK_RYS_DEG + 1), x);
        w = cheb(c + (n + r) * (PK_RYS_DEG + 1), x);
    }
}

// Sums of nterm terms for nout outputs over the 64 lanes of the workgroup:
// lpo lanes (a power of two) per output each add a strided share, then a
// butterfly inside the aligned lane group; the group's first lane emits.
// Every lane calls it (the shuffles need the whole wave).
template <typename Term, typename Emit>
__device__ __forceinline__ void seg_reduce(int lane, int nout, int nterm, Term term, Emit emit) {
    int sh = 0;  // lpo = 2^sh lanes per output
    while (sh < 6 && (2 << sh) * nout <= 64) ++sh;
    const int lpo = 1 << sh, opp = 64 >> sh;
    const int sl = lane & (lpo - 1);
    for (int o0 = 0; o0 < nout; o0 += opp) {
        const int o = o0 + (lane >> sh);
        double s = 0.0;
        if (o < nout)
            for (int t = sl; t < nterm; t += lpo) s += term(o, t);
        for (int off = lpo >> 1; off >= 1; off >>= 1) s += __shfl_xor(s, off, 64);
        if (o < nout && sl == 0) emit(o, s);
    }
}

// Cartesian exponents (x, y, z) of component k of a shell of angular momentum
// l <= 3, in the order lx descending, then ly descending
static __device__ const unsigned char kCartTab[4][10][3] = {
    {{0, 0, 0}},
    {{1, 0, 0}, {0, 1, 0}, {0, 0, 1}},
    {{2, 0, 0}, {1, 1, 0}, {1, 0, 1}, {0, 2, 0}, {0, 1, 1}, {0, 0, 2}},
    {{3, 0, 0}, {2, 1, 0}, {2, 0, 1}, {1, 2, 0}, {1, 1, 1}, {1, 0, 2}, {0, 3, 0}, {0, 2, 1}, {0, 1, 2}, {0, 0, 3}}};

// Index tables of one class, built once per workgroup so that the hot loops
// decode their indices by lookups instead of integer divisions: at most 100
// component pairs of two shells, 256 transferred 1-D factors per (root, axis).
struct GenTabs {
    static constexpr int NPR = 100, NGT = 256;
    unsigned char ab_a[NPR], ab_b[NPR], cd_c[NPR], cd_d[NPR];  // ab -> (a, b), cd -> (c, d)
    unsigned char ac_a[NPR], ac_c[NPR], bd_b[NPR], bd_d[NPR];  // pairs of the exchange sums
    unsigned char bc_b[NPR], bc_c[NPR], ad_a[NPR], ad_d[NPR];
    unsigned short ab_g[NPR][3];                               // G offset of (a, b) per axis
    unsigned char cd_g[NPR][3];                                // G offset of (c, d) per axis
    unsigned char g_a[NGT], g_b[NGT], g_c[NGT], g_d[NGT];      // G index -> exponents
};

__global__ __launch_bounds__(64) void k_generic(GenArgs a) {
    constexpr int NL = 64, NPR = GenTabs::NPR;
    extern __shared__ double smem[];
    __shared__ double su[GEN_NR], sw[GEN_NR];
    __shared__ double hab[3][10], hcd[3][10];  // C(b,k) AB^(b-k) per axis at [b(b+1)/2 + k]; ket likewise
    __shared__ double sP[6][NPR];              // density blocks ab, cd, ac, ad, bc, bd
    __shared__ double sQ[2][NPR];              // Schwarz blocks ab, cd
    __shared__ GenTabs tb;
    const int lane = threadIdx.x;
    const int item = blockIdx.x;
    if (item >= a.nitems) return;
    const int la = a.la, lb = a.lb, lc = a.lc, ld = a.ld;
    const int NA = (la + 1) * (la + 2) / 2, NB = (lb + 1) * (lb + 2) / 2;
    const int NC = (lc + 1) * (lc + 2) / 2, ND = (ld + 1) * (ld + 2) / 2;
    const int NAB = NA * NB, NCD = NC * ND, NABCD = NAB * NCD;
    const int E = la + lb, F = lc + ld, n = (E + F) / 2 + 1;
    const int F1 = F + 1, NI = (E + 1) * F1;
    const int D2 = lb + 1, D3 = lc + 1, D4 = ld + 1, D34 = D3 * D4;
    const int NG = (la + 1) * D2 * D34;  // transferred 1-D factors per (root, axis)
    double *I2 = smem;                   // [n * 3][E + 1][F + 1]
    double *G = I2 + n * 3 * NI;         // [n * 3][la + 1][lb + 1][lc + 1][ld + 1]
    double *acc = G + n * 3 * NG;        // [NABCD]

    for (int i = lane; i < NAB; i += NL) {
        const int ia = i / NB, ib = i % NB;
        tb.ab_a[i] = ia;
        tb.ab_b[i] = ib;
        for (int q = 0; q < 3; ++q) tb.ab_g[i][q] = (kCartTab[la][ia][q] * D2 + kCartTab[lb][ib][q]) * D34;
    }
    for (int i = lane; i < NCD; i += NL) {
        const int ic = i / ND, id = i % ND;
        tb.cd_c[i] = ic;
        tb.cd_d[i] = id;
        for (int q = 0; q < 3; ++q) tb.cd_g[i][q] = kCartTab[lc][ic][q] * D4 + kCartTab[ld][id][q];
    }
    for (int i = lane; i < NA * NC; i += NL) tb.ac_a[i] = i / NC, tb.ac_c[i] = i % NC;
    for (int i = lane; i < NB * ND; i += NL) tb.bd_b[i] = i / ND, tb.bd_d[i] = i % ND;
    for (int i = lane; i < NB * NC; i += NL) tb.bc_b[i] = i / NC, tb.bc_c[i] = i % NC;
    for (int i = lane; i < NA * ND; i += NL) tb.ad_a[i] = i / ND, tb.ad_d[i] = i % ND;
    for (int g = lane; g < NG; g += NL) {
        int t = g;
        tb.g_d[g] = t % D4;
        t /= D4;
        tb.g_c[g] = t % D3;
        t /= D3;
        tb.g_b[g] = t % D2;
        tb.g_a[g] = t / D2;
    }
    // this lane's first (ab, cd) in the flattened component loops, and the
    // step of 64 components in (ab, cd); likewise (root-axis, g) of the
    // transfer loop
    const int ab0 = lane / NCD, cd0 = lane % NCD, sab = NL / NCD, scd = NL % NCD;
    const int ra0 = lane / NG, g0 = lane % NG, sra = NL / NG, sg = NL % NG;
    __syncthreads();

    int bra, kbeg, kcnt, nb = 0;
    const double *P = nullptr, *Qm = nullptr;
    double *Am = nullptr, *Bm = nullptr;
    if (a.eri_mode) {
        bra = a.qbra[item];
        kbeg = item;
        kcnt = 1;
    } else {
        bra = a.wave_bra[item];
        kbeg = a.wave_start[item];
        kcnt = a.wave_count[item];
        const int mol = a.wave_mol[item];
        const long long moff = a.mol_off[mol];
        nb = a.mol_nb[mol];
        P = a.P + moff;
        Qm = a.Q + moff;
        Am = a.A + moff;
        Bm = a.B + moff;
    }
    const PairDev pb = a.pairs[bra];
    if (lane < 30) {
        // bra transfer coefficients C(b,k) AB^(b-k), b <= 3
        const int ax = lane / 10, t = lane % 10;
        const int b = t >= 6 ? 3 : (t >= 3 ? 2 : (t >= 1 ? 1 : 0)), k = t - b * (b + 1) / 2;
        const double x = sel3(ax, pb.ab[0], pb.ab[1], pb.ab[2]);
        double p = binom(b, k);
        for (int e = 0; e < b - k; ++e) p *= x;
        hab[ax][t] = p;
    }

    for (int kk = 0; kk < kcnt; ++kk) {
        const int ket = a.eri_mode ? a.qket[item] : a.kets[kbeg + kk];
        const PairDev pk = a.pairs[ket];
        for (int i = lane; i < NABCD; i += NL) acc[i] = 0.0;
        if (lane < 30) {
            const int ax = lane / 10, t = lane % 10;
            const int b = t >= 6 ? 3 : (t >= 3 ? 2 : (t >= 1 ? 1 : 0)), k = t - b * (b + 1) / 2;
            const double x = sel3(ax, pk.ab[0], pk.ab[1], pk.ab[2]);
            double p = binom(b, k);
            for (int e = 0; e < b - k; ++e) p *= x;
            hcd[ax][t] = p;
        }
        __syncthreads();
        for (int kq = 0; kq < pk.nprim; ++kq) {
            const PrimDev q = a.prims[pk.prim_off + kq];
            const double hq = a.hz[pk.prim_off + kq];
            for (int kp = 0; kp < pb.nprim; ++kp) {
                const PrimDev p = a.prims[pb.prim_off + kp];
                const double hp = a.hz[pb.prim_off + kp];
                const double rs = rsqrt_nr(p.zeta + q.zeta);
                const double inv_de = rs * rs;
                const double rho = p.zeta * q.zeta * inv_de;
                const double PQ[3] = {p.p[0] - q.p[0], p.p[1] - q.p[1], p.p[2] - q.p[2]};
                const double T = rho * fma(PQ[0], PQ[0], fma(PQ[1], PQ[1], PQ[2] * PQ[2]));
                const double pref = p.kc * q.kc * rs;
                if (lane < n) {
                    double u, w;
                    rys_root_rt(n, T, lane, u, w);
                    su[lane] = u;
                    sw[lane] = w;
                }
                __syncthreads();
                // 2-D integrals I[e][f] of root r, axis ax (lane 3r + ax), one
                // column f at a time with the previous two columns in registers
                if (lane < 3 * n) {
                    const int r = lane / 3, ax = lane - 3 * r;
                    const double ur = su[r];
                    const double B00 = 0.5 * inv_de * ur;
                    const double B10 = hp * (1.0 - q.zeta * inv_de * ur);  // rho / zeta = eta / (zeta + eta)
                    const double B01 = hq * (1.0 - p.zeta * inv_de * ur);
                    const double PQa = sel3(ax, PQ[0], PQ[1], PQ[2]);
                    const double C00 = fma(ur * (-q.zeta * inv_de), PQa, sel3(ax, p.pa[0], p.pa[1], p.pa[2]));
                    const double D00 = fma(ur * (p.zeta * inv_de), PQa, sel3(ax, q.pa[0], q.pa[1], q.pa[2]));
                    double *I = I2 + lane * NI;
                    double c2[GEN_NR], c1[GEN_NR], c0[GEN_NR];
                    c1[0] = ax == 0 ? pref * sw[r] : 1.0;
#pragma unroll
                    for (int e = 1; e < GEN_NR; ++e) {
                        double t = C00 * c1[e - 1];
                        if (e >= 2) t = fma((double)(e - 1) * B10, c1[e - 2], t);
                        c1[e] = e <= E ? t : 0.0;
                    }
#pragma unroll
                    for (int e = 0; e < GEN_NR; ++e) {
                        if (e <= E) I[e * F1] = c1[e];
                        c2[e] = 0.0;
                    }
                    for (int f = 1; f <= F; ++f) {
                        const double bf = (double)(f - 1) * B01;
#pragma unroll
                        for (int e = 0; e < GEN_NR; ++e) {
                            double t = fma(D00, c1[e], bf * c2[e]);
                            if (e >= 1) t = fma((double)e * B00, c1[e - 1], t);
                            c0[e] = e <= E ? t : 0.0;
                        }
#pragma unroll
                        for (int e = 0; e < GEN_NR; ++e) {
                            if (e <= E) I[e * F1 + f] = c0[e];
                            c2[e] = c1[e];
                            c1[e] = c0[e];
                        }
                    }
                }
                __syncthreads();
                // transferred factors G[a][b][c][d] = sum_k sum_l C(b,k) AB^(b-k)
                // C(d,l) CD^(d-l) I[a+k][c+l] for every (root, axis) and G index,
                // spread over the lanes
                int ra = ra0, g = g0;
                for (int t = lane; t < 3 * n * NG; t += NL) {
                    const int ax = ra % 3;
                    const int ia = tb.g_a[g], ib = tb.g_b[g], ic = tb.g_c[g], id = tb.g_d[g];
                    const double *I = I2 + ra * NI + ia * F1 + ic;
                    const double *hb = hab[ax] + ib * (ib + 1) / 2, *hd = hcd[ax] + id * (id + 1) / 2;
                    double s = 0.0;
                    for (int k = 0; k <= ib; ++k) {
                        double scd = 0.0;
                        for (int l = 0; l <= id; ++l) scd = fma(hd[l], I[k * F1 + l], scd);
                        s = fma(hb[k], scd, s);
                    }
                    G[ra * NG + g] = s;
                    g += sg;
                    ra += sra;
                    if (g >= NG) g -= NG, ++ra;
                }
                __syncthreads();
                int ab = ab0, cd = cd0;
                for (int i = lane; i < NABCD; i += NL) {
                    const int o0 = tb.ab_g[ab][0] + tb.cd_g[cd][0], o1 = tb.ab_g[ab][1] + tb.cd_g[cd][1],
                              o2 = tb.ab_g[ab][2] + tb.cd_g[cd][2];
                    double s = 0.0;
                    for (int r = 0; r < n; ++r)
                        s = fma(G[(r * 3) * NG + o0] * G[(r * 3 + 1) * NG + o1], G[(r * 3 + 2) * NG + o2], s);
                    acc[i] += s;
                    cd += scd;
                    ab += sab;
                    if (cd >= NCD) cd -= NCD, ++ab;
                }
                __syncthreads();
            }
        }
        if (a.eri_mode) {
            double *o = a.out + (size_t)item * NABCD;
            for (int i = lane; i < NABCD; i += NL) o[i] = acc[i];
            __syncthreads();
            continue;
        }
        // ---- J/K digestion of the quartet (bra pb, ket pk)
        double deg = 1.0;
        if (pb.diag) deg *= 0.5;
        if (pk.diag) deg *= 0.5;
        if (pb.f0 == pk.f0 && pb.f1 == pk.f1) deg *= 0.5;
        const bool all_pass = pb.qmin * pk.qmin >= a.tol;
        // density (and Schwarz) blocks of the quartet into LDS: independent
        // loads issued together, read many times by the reductions below
        auto Pv = [&](int r, int c) { return P[(size_t)r * nb + c]; };
        for (int i = lane; i < NAB; i += NL) {
            const int af = pb.f0 + tb.ab_a[i], bf = pb.f1 + tb.ab_b[i];
            sP[0][i] = Pv(af, bf);
            if (!all_pass) sQ[0][i] = Qm[(size_t)af * nb + bf];
        }
        for (int i = lane; i < NCD; i += NL) {
            const int cf = pk.f0 + tb.cd_c[i], df = pk.f1 + tb.cd_d[i];
            sP[1][i] = Pv(cf, df);
            if (!all_pass) sQ[1][i] = Qm[(size_t)cf * nb + df];
        }
        for (int i = lane; i < NA * NC; i += NL) sP[2][i] = Pv(pb.f0 + tb.ac_a[i], pk.f0 + tb.ac_c[i]);
        for (int i = lane; i < NA * ND; i += NL) sP[3][i] = Pv(pb.f0 + tb.ad_a[i], pk.f1 + tb.ad_d[i]);
        for (int i = lane; i < NB * NC; i += NL) sP[4][i] = Pv(pb.f1 + tb.bc_b[i], pk.f0 + tb.bc_c[i]);
        for (int i = lane; i < NB * ND; i += NL) sP[5][i] = Pv(pb.f1 + tb.bd_b[i], pk.f1 + tb.bd_d[i]);
        __syncthreads();
        // apply degeneracy and the function-level Schwarz test in place
        {
            int ab = ab0, cd = cd0;
            for (int i = lane; i < NABCD; i += NL) {
                double m = deg;
                if (!all_pass && sQ[0][ab] * sQ[1][cd] < a.tol) m = 0.0;
                acc[i] *= m;
                cd += scd;
                ab += sab;
                if (cd >= NCD) cd -= NCD, ++ab;
            }
        }
        __syncthreads();
        auto at = [&](int ia, int ib, int ic, int id) { return acc[(ia * NB + ib) * NCD + ic * ND + id]; };
        // A_ab += 2 sum_cd v P_cd ; A_cd += 2 sum_ab v P_ab
        seg_reduce(lane, NAB, NCD, [&](int ab, int cd) { return acc[ab * NCD + cd] * sP[1][cd]; },
                   [&](int ab, double v) {
                       unsafeAtomicAdd(&Am[(size_t)(pb.f0 + tb.ab_a[ab]) * nb + pb.f1 + tb.ab_b[ab]], 2.0 * v);
                   });
        seg_reduce(lane, NCD, NAB, [&](int cd, int ab) { return acc[ab * NCD + cd] * sP[0][ab]; },
                   [&](int cd, double v) {
                       unsafeAtomicAdd(&Am[(size_t)(pk.f0 + tb.cd_c[cd]) * nb + pk.f1 + tb.cd_d[cd]], 2.0 * v);
                   });
        // B_ac += sum_bd v P_bd ; B_bc += sum_ad v P_ad ; B_ad += sum_bc v P_bc ; B_bd += sum_ac v P_ac
        const double(*S)[NPR] = sP + 2;  // ac, ad, bc, bd
            seg_reduce(lane, NA * NC, NB * ND, [&](int o, int t) {
                return at(tb.ac_a[o], tb.bd_b[t], tb.ac_c[o], tb.bd_d[t]) * S[3][t];
            }, [&](int o, double v) { unsafeAtomicAdd(&Bm[(size_t)(pb.f0 + tb.ac_a[o]) * nb + pk.f0 + tb.ac_c[o]], v); });
            seg_reduce(lane, NB * NC, NA * ND, [&](int o, int t) {
                return at(tb.ad_a[t], tb.bc_b[o], tb.bc_c[o], tb.ad_d[t]) * S[1][t];
            }, [&](int o, double v) { unsafeAtomicAdd(&Bm[(size_t)(pb.f1 + tb.bc_b[o]) * nb + pk.f0 + tb.bc_c[o]], v); });
            seg_reduce(lane, NA * ND, NB * NC, [&](int o, int t) {
                return at(tb.ad_a[o], tb.bc_b[t], tb.bc_c[t], tb.ad_d[o]) * S[2][t];
            }, [&](int o, double v) { unsafeAtomicAdd(&Bm[(size_t)(pb.f0 + tb.ad_a[o]) * nb + pk.f1 + tb.ad_d[o]], v); });
            seg_reduce(lane, NB * ND, NA * NC, [&](int o, int t) {
                return at(tb.ac_a[t], tb.bd_b[o], tb.ac_c[t], tb.bd_d[o]) * S[0][t];
            }, [&](int o, double v) { unsafeAtomicAdd(&Bm[(size_t)(pb.f1 + tb.bd_b[o]) * nb + pk.f1 + tb.bd_d[o]], v); });
        __syncthreads();
    }
}

// dynamic LDS of the generic kernel for a class: 2-D integrals and transferred
// factors for n roots x 3 axes, and the quartet's accumulators
inline size_t generic_lds_bytes(int la, int lb, int lc, int ld) {
    const size_t nabcd = (size_t)ncart(la) * ncart(lb) * ncart(lc) * ncart(ld);
    const size_t n = (la + lb + lc + ld) / 2 + 1;
    const size_t ni = (size_t)(la + lb + 1) * (lc + ld + 1), ng = (size_t)(la + 1) * (lb + 1) * (lc + 1) * (ld + 1);
    return (n * 3 * (ni + ng) + nabcd) * sizeof(double);
}

}  // namespace pk
