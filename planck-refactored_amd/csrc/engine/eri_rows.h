// eri_rows.h — row kernel: the shell-quartet kernel of the classes whose
// integrals do not fit one lane (d and f classes).
//
// One wave owns QW quartets (one bra pair, QW ket pairs) at a time; a lane owns
// row(s) (ab) of the integral matrices (ab|cd) and keeps all NCD ket components
// of its rows in registers from the first primitive to the last J/K sum.
//   Phase A, lane = (quartet, root, axis): the Rys root, the 2-D integrals and
//   the A -> B transfer of one axis,
//     G[a][b][f] = sum_k C(b,k) AB^(b-k) I[a+k][f],
//   entirely in registers, then one run of LDS stores.
//   Phase B, lane = row (a, b): per root the three rows G_x[ax][bx][..],
//   G_y[ay][by][..], G_z[az][bz][..] (lc+ld+1 contiguous doubles each) come from
//   LDS and every ket component f of |f0], lc <= |f| <= lc+ld, adds Gx Gy Gz.
//   After the primitives the C -> D transfer turns the row [ab|f0] into (ab|cd)
//   in the lane's registers.
// A workgroup takes a work item: one bra pair and up to about a thousand of its
// kets.  J/K digestion from the registers: J_ab is kept over the whole item; the
// exchange sums into the ket's second shell go to LDS exchange rows (the bra's
// functions x the functions of that shell type), flushed once per item; those
// into its first shell to a small LDS block per slot, flushed when that shell
// changes; J_cd is summed over the rows through LDS, one global atomic per ket
// component.
//
// What bounds it: the LDS pipe (phase B reads 3 (lc+ld+1) doubles per row and
// root, the digestion about as much again), 55-70% busy on (dp|dp) and (fd|dp)
// of n-C10H22 / cc-pVTZ, with the VALU at 30%; two waves per SIMD by registers.
// Hence the layout: the C -> D transfer after the contraction (16 doubles per
// row instead of 18 for (dp| kets, 46 instead of 60 for (fd|, and (lc+ld+1)
// instead of (lc+1)(ld+1) factors per axis), odd strides, the exchange sums of
// the first ket shell held over the run of kets that share it (LDS exchange rows
// only for the second shell's columns), and the densities of a group staged once
// by coalesced loads.  Serial kernel times against the per-lane and the
// one-quartet-per-wave kernels they replace: see rows_class in eri_classes.h.
// Reference semantics as in eri_prim.h (rys.cpp:250-485, os.cpp:837-879) and
// eri_kernels.h (digestion).
#pragma once

#include "eri_kernels.h"

namespace pk {

// Shape of one class: RC row chunks (blockIdx.y) of RN rows, RPL rows per lane,
// QW quartets per wave.
template <int LA, int LB, int LC, int LD>
struct RowCls {
    using K = Cls<LA, LB, LC, LD>;
    static constexpr int NR = K::NR, NAB = K::NAB, NCD = K::NCD;
    static constexpr int RC = NAB > 64 ? 2 : 1, RN = (NAB + RC - 1) / RC;
    static constexpr int E = K::E, F = K::F, NF = K::NF;
    static constexpr int RL = (F + 1) | 1;                         // doubles of one (a, b) row of one axis, odd (banks)
    static constexpr int NGP = ((LA + 1) * (LB + 1) * RL) | 1;     // odd stride: the lanes' stores hit all banks
    static constexpr int qw(int rpl) {
        int q = 64 * rpl / RN;
        const int qa = 64 / (3 * NR);
        q = q < qa ? q : qa;
        return q < 1 ? 1 : q;
    }
    static constexpr int gdoubles(int rpl) { return qw(rpl) * 3 * NR * NGP; }
    static constexpr int RPL = (RC == 1 && qw(2) > qw(1) && 2 * NF <= 18 && gdoubles(2) * 8 <= 16384) ? 2 : 1;
    static constexpr int QW = qw(RPL);
    static constexpr int NRT = QW * RN;  // rows of a wave
    // staged densities of a quartet: Schwarz and J density of (cd), then the
    // rows a and b of the exchange density (twice for two) at the columns c, d
    static constexpr int NX = (K::NA + K::NB) * (K::NC + K::ND);
    static constexpr int pe(int nk) { return 2 * NCD + nk * NX; }
    static constexpr int JS = NRT | 1;  // stride of the J_cd buffer
    // doubles of LDS per wave: the factors, or the staged densities and at least
    // a few components of the J_cd buffer
    static constexpr int gd(int nk) {
        const int f = gdoubles(RPL), j = QW * pe(nk) + JS * (NCD < 4 ? NCD : 4);
        return ((f > j ? f : j) + 1) / 2 * 2;
    }
    // exchange sums of the current first ket shell of each slot
    static constexpr int NROW = K::NA + K::NB;
    static constexpr int cb(int nk) { return (QW * nk * NROW * K::NC + 1) / 2 * 2; }
    // held in registers over the run of kets that share it, where they are few
    static constexpr bool run(int nk) { return nk * RPL * 2 * K::NC <= 20; }
    static constexpr int wave_doubles(int nk) { return gd(nk) + cb(nk); }
    static constexpr int jc(int nk) {  // ket components per J_cd pass
        const int c = (gd(nk) - QW * pe(nk)) / JS;
        return c < NCD ? c : NCD;
    }
};

__device__ __forceinline__ void wave_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

__device__ __forceinline__ double sel3d(int ax, double x, double y, double z) { return ax == 0 ? x : (ax == 1 ? y : z); }

// All G[a][b][f] of one axis into g (LDS, [(a (LB+1) + b) RL + f]).
template <int LA, int LB, int F, int RL>
__device__ __forceinline__ void axis_rows(double seed, double C00, double D00, double B00, double B10, double B01,
                                          double AB, double *g) {
    constexpr int E = LA + LB;
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
    // A -> B, b ascending in place: I[a] holds (a|b)
    sfor<0, LB + 1>([&](auto b_) {
        constexpr int b = PK_CI(b_);
        if constexpr (b > 0)
            sfor<0, E - b + 1>([&](auto a_) {
                constexpr int a = PK_CI(a_);
                sfor<0, F + 1>([&](auto f_) { I[a][PK_CI(f_)] = fma(AB, I[a][PK_CI(f_)], I[a + 1][PK_CI(f_)]); });
            });
        sfor<0, LA + 1>([&](auto a_) {
            sfor<0, F + 1>([&](auto f_) { g[(PK_CI(a_) * (LB + 1) + b) * RL + PK_CI(f_)] = I[PK_CI(a_)][PK_CI(f_)]; });
        });
    });
}

// Uniform loads through the constant address space: scalar loads, although the
// kernel also writes memory (pairs, primitives and lists never change during it).
template <typename T>
__device__ __forceinline__ T uload(const T *p) {
    return *(const __attribute__((address_space(4))) T *)(unsigned long long)p;
}

// Work item blk, row chunk chunk_y, on all waves of the workgroup; smem: its LDS.
template <int LA, int LB, int LC, int LD, int NK>
__device__ __forceinline__ void rows_run(const JKArgs &a, int blk, int chunk_y, double *smem) {
    using K = Cls<LA, LB, LC, LD>;
    using S = RowCls<LA, LB, LC, LD>;
    constexpr int NA = K::NA, NB = K::NB, NC = K::NC, ND = K::ND, NAB = K::NAB, NCD = K::NCD, NF = K::NF, NR = K::NR;
    constexpr int RPL = S::RPL, QW = S::QW, RN = S::RN, RL = S::RL, NGP = S::NGP, NROW = NA + NB, GD = S::wave_doubles(NK);
    constexpr bool RUN = S::run(NK);
    constexpr int CB = QW * NK * NROW * NC;
    const int lane = threadIdx.x & 63;
    const int wid = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int nwg = (int)(blockDim.x >> 6);
    const int bra = uload(a.wave_bra + blk);
    const unsigned kbeg = uload(a.wave_start + blk);
    const unsigned kend = kbeg + uload(a.wave_count + blk);
    const int mol = uload(a.wave_mol + blk);
    const long long moff = uload(a.mol_off + mol);
    const int nb = uload(a.mol_nb + mol);
    const double *__restrict__ P = a.P + moff;
    const double *__restrict__ KD[2] = {NK == 2 ? a.PK + moff : P, NK == 2 ? a.PK2 + moff : P};
    const double *__restrict__ Qm = a.Q + moff;
    double *Am = a.A + moff;
    double *Bg[2] = {a.B + moff, NK == 2 ? a.B2 + moff : a.B + moff};
    double *G = smem + (size_t)wid * GD;
    double *krow = smem + (size_t)nwg * GD;  // [NK][NA + NB][kcols], then J_ab
    const bool segmode = a.segmode != 0;
    const int kc = segmode ? a.kcols : 0;
    double *jrow = krow + NK * NROW * kc;
    const int *tb = a.tblk + 5 * mol;
    const int dbase = uload(tb + LD), ncols = uload(tb + LD + 1) - dbase;  // columns: the kets' second shells
    double *cblk = G + S::gd(NK);  // [QW][NK][NA + NB][NC] of this wave
    for (int i = lane; i < CB; i += 64) cblk[i] = 0.0;
    for (int i = threadIdx.x; i < NK * NROW * kc + NAB; i += blockDim.x) krow[i] = 0.0;
    __syncthreads();

    const PairDev *pbp = a.pairs + bra;
    const int bf0 = uload(&pbp->f0), bf1 = uload(&pbp->f1), np = uload(&pbp->nprim), bpo = uload(&pbp->prim_off);
    const double bqmin = uload(&pbp->qmin);
    const double bdeg = uload(&pbp->diag) ? 0.5 : 1.0;

    // phase A role: slot, root, axis
    const int sa = lane / (3 * NR), ra = lane - sa * 3 * NR;
    const int r_a = ra / 3, ax = ra - 3 * r_a;
    const bool live_a = sa < QW;
    double *Ga = G + (live_a ? (sa * 3 * NR + ra) : 0) * NGP;
    const double ABq = sel3d(ax, uload(&pbp->ab[0]), uload(&pbp->ab[1]), uload(&pbp->ab[2]));
    const int cw = ((ax == 1 ? NR : 0) + r_a) * (PK_RYS_DEG + 1);  // Chebyshev series of this lane: the node
                                                                   // (axes 0, 2) or the weight (1)
    const double lim = ax == 1 ? pk_rys_aw[pk_rys_abase[NR] + r_a] : pk_rys_ax2[pk_rys_abase[NR] + r_a];

    // phase B role: rows idx = lane + 64 k of (slot, row)
    const int row0 = S::RC > 1 ? chunk_y * RN : 0;
    int sb[RPL], ro[RPL][3], af_[RPL], bf_[RPL], ka_[RPL], kb_[RPL];
    bool live[RPL];
    double Pab[RPL], Qab[RPL], jab[RPL];
    sfor<0, RPL>([&](auto k_) {
        constexpr int k = PK_CI(k_);
        const int idx = lane + 64 * k;
        const int s = idx / RN;
        int row = row0 + idx - s * RN;
        live[k] = s < QW && row < NAB;
        sb[k] = live[k] ? s : 0;
        if (!live[k]) row = 0;
        const int ia = row / NB, ib = row - ia * NB;
        af_[k] = bf0 + ia;
        bf_[k] = bf1 + ib;
        ka_[k] = ia * kc;
        kb_[k] = (NA + ib) * kc;
        // exponents of component i of a shell of angular momentum l
        auto ex = [](int l, int i, int *x) {
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
            ro[k][q] = sb[k] * 3 * NR * NGP + q * NGP + (xa[q] * (LB + 1) + xb[q]) * RL;
        });
        const size_t abi = (size_t)af_[k] * nb + bf_[k];
        Pab[k] = P[abi];
        Qab[k] = Qm[abi];
        jab[k] = 0.0;
    });

    // staged elements of this lane: e = lane + 64 i of [slot][pe]; the address is
    // base + ket-dependent part: kind 0 (cd): (c0 + c) nb + d0 + d, kinds 1, 2: row
    // + c0 + col or row + d0 + col
    constexpr int PE = S::pe(NK), EPL = (QW * PE + 63) / 64, NCX = NC + ND;
    // groups of a wave: chunks of a.chunk groups dealt to the waves in turn (kets
    // with the same first shell are neighbours, and their cost falls along the list)
    int left = a.chunk;  // groups of the current chunk after the one that next() left
    unsigned g0 = kbeg + wid * a.chunk * QW;
    auto next = [&](unsigned g) {
        if (--left > 0) return g + QW;
        left = a.chunk;
        return g + QW + (nwg - 1) * a.chunk * QW;
    };

    // ---- software pipeline over the groups: the ket indices are loaded two
    // groups ahead, the pair fields one group ahead (ket primitives and the
    // coefficients of their roots where they are used: loading them one primitive
    // quartet ahead changed nothing, the LDS pipe and the vector unit set the time)
    auto slot_ket = [&](unsigned g, int s) { return a.kets[ket_pos(g, s, kend)]; };
    int ida = 0, idb[RPL];                      // kets of the next group (phase A slot, rows)
    int n_qoff, n_nq, n_c0[RPL], n_d0[RPL], n_diag[RPL];
    double n_qmin[RPL], n_cd[RPL][3];
    auto load_fields = [&](unsigned g) {             // from ida, idb of group g
        const PairDev *pk = a.pairs + ida;
        const bool on = live_a && g + sa < kend;
        n_nq = on ? pk->nprim : 0;
        n_qoff = pk->prim_off;
        sfor<0, RPL>([&](auto k_) {
            constexpr int k = PK_CI(k_);
            const PairDev *pr = a.pairs + idb[k];
            n_c0[k] = pr->f0;
            n_d0[k] = pr->f1;
            n_diag[k] = pr->diag;
            n_qmin[k] = pr->qmin;
            sfor<0, 3>([&](auto q_) { n_cd[k][PK_CI(q_)] = pr->ab[PK_CI(q_)]; });
        });
    };
    auto load_ids = [&](unsigned g) {
        ida = slot_ket(g, live_a ? sa : 0);
        sfor<0, RPL>([&](auto k_) { idb[PK_CI(k_)] = slot_ket(g, sb[PK_CI(k_)]); });
    };
    // ket primitive kq of the lane's slot, and the roots' coefficients of (kq, kp)
    int qoff = 0, nqa = 0;
    double qz, qx, qy, qw, hq, qpa, qkc;
    auto load_q = [&](int kq) {
        const int qi = nqa > 0 ? qoff + min(kq, nqa - 1) : 0;
        const PrimDev *qp = a.prims + qi;
        qz = qp->zeta;
        qx = qp->p[0];
        qy = qp->p[1];
        qw = qp->p[2];
        qpa = qp->pa[ax];
        qkc = kq < nqa ? qp->kc : 0.0;
        hq = a.hz[qi];
    };
    double rs, T, xc, cc[PK_RYS_DEG + 1], PQa;
    auto prep = [&](int kp) {
        const PrimDev *pp = a.prims + (bpo + kp);
        const double pz = uload(&pp->zeta);
        rs = rsqrt_nr(pz + qz);
        const double x = uload(&pp->p[0]) - qx, y = uload(&pp->p[1]) - qy, z = uload(&pp->p[2]) - qw;
        T = pz * qz * (rs * rs) * fma(x, x, fma(y, y, z * z));
        PQa = sel3d(ax, x, y, z);
        const double Tc = T < pk_rys_tmax[NR] ? T : 0.0;
        const int i = (int)Tc;
        xc = 2.0 * (Tc - (double)i) - 1.0;
        const double *c = pk_rys_coef + pk_rys_base[NR] + i * (2 * NR * (PK_RYS_DEG + 1)) + cw;
#pragma unroll
        for (int j = 0; j <= PK_RYS_DEG; ++j) cc[j] = c[j];
    };
    bool more = false;  // primitives left in the group
    unsigned g1 = next(g0);
    if (g0 < kend) {
        load_ids(g0);
        load_fields(g0);
        load_ids(g1);
        qoff = n_qoff, nqa = n_nq;
        // a pair can have lost all its primitives to the screening
        more = np > 0 && __any(nqa > 0);
    }
    // exchange sums (rows a and b, columns of the first ket shell) of the current
    // run, and their way to the global accumulator when the shell changes
    int cur[RPL];
    double kca[RUN ? NK : 1][RUN ? RPL : 1][RUN ? NC : 1], kcb[RUN ? NK : 1][RUN ? RPL : 1][RUN ? NC : 1];
    auto clear_run = [&]() {
        if constexpr (RUN)
            sfor<0, NK * RPL * NC>([&](auto i_) {
                constexpr int i = PK_CI(i_);
                kca[i / (RPL * NC)][i / NC % RPL][i % NC] = kcb[i / (RPL * NC)][i / NC % RPL][i % NC] = 0.0;
            });
    };
    sfor<0, RPL>([&](auto k_) { cur[PK_CI(k_)] = -1; });
    clear_run();
    // value of x at the lane of the first row of slot s
    auto at_slot = [&](const int (&x)[RPL], int s) {
        const int idx = s * RN;
        if constexpr (RPL == 1) {
            return __shfl(x[0], idx, 64);
        } else {
            const int u = __shfl(x[0], idx & 63, 64), v = __shfl(x[1], idx & 63, 64);
            return idx < 64 ? u : v;
        }
    };
    auto cadd = [&](int sp, int k, int r, int c, double x) {
        __hip_atomic_fetch_add(&cblk[((sb[k] * NK + sp) * NROW + r) * NC + c], x, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_WAVEFRONT);
    };
    auto flush_run = [&]() {
        if constexpr (RUN) {
            sfor<0, NK * RPL>([&](auto i_) {
                constexpr int sp = PK_CI(i_) / RPL, k = PK_CI(i_) % RPL;
                if (live[k])
                    sfor<0, NC>([&](auto c_) {
                        cadd(sp, k, af_[k] - bf0, PK_CI(c_), kca[sp][k][PK_CI(c_)]);
                        cadd(sp, k, NA + bf_[k] - bf1, PK_CI(c_), kcb[sp][k][PK_CI(c_)]);
                    });
            });
            clear_run();
        }
        wave_fence();
        int ln = lane;
        asm volatile("" : "+v"(ln));
        sfor<0, (CB + 63) / 64>([&](auto i_) {
            const int e = ln + 64 * PK_CI(i_);
            const int s = min(e / (NK * NROW * NC), QW - 1), t = e - s * (NK * NROW * NC);
            const int c0 = at_slot(cur, s);
            if (e < CB) {
                const double x = cblk[e];
                cblk[e] = 0.0;
                const int sp = NK == 2 && t >= NROW * NC ? 1 : 0, rc = t - sp * NROW * NC;
                const int r = rc / NC, rf = r < NA ? bf0 + r : bf1 + r - NA;
                if (x != 0.0) unsafeAtomicAdd(&(sp ? Bg[1] : Bg[0])[(size_t)rf * nb + c0 + rc - r * NC], x);
            }
        });
        wave_fence();
    };
    while (g0 < kend) {
        {
            bool changed = false;
            sfor<0, RPL>([&](auto k_) { changed = changed || (cur[PK_CI(k_)] >= 0 && cur[PK_CI(k_)] != n_c0[PK_CI(k_)]); });
            if (__any(changed)) flush_run();
            sfor<0, RPL>([&](auto k_) { cur[PK_CI(k_)] = n_c0[PK_CI(k_)]; });
        }
        // this group's rows
        int cf0[RPL], df0[RPL];
        double deg[RPL], kqmin[RPL], cd[RPL][3];
        sfor<0, RPL>([&](auto k_) {
            constexpr int k = PK_CI(k_);
            cf0[k] = n_c0[k];
            df0[k] = n_d0[k];
            kqmin[k] = n_qmin[k];
            sfor<0, 3>([&](auto q_) { cd[k][PK_CI(q_)] = n_cd[k][PK_CI(q_)]; });
            double d = n_diag[k] ? 0.5 * bdeg : bdeg;
            if (cf0[k] == bf0 && df0[k] == bf1) d *= 0.5;
            deg[k] = live[k] && g0 + sb[k] < kend ? d : 0.0;  // 0 for lanes and slots without a quartet
        });
        // densities of the group's quartets, one element of [slot][PE] per lane and load
        double st[EPL];
        {
            int ln = lane;
            asm volatile("" : "+v"(ln));  // the element's indices are recomputed here, not held over the loop
            sfor<0, EPL>([&](auto i_) {
                constexpr int i = PK_CI(i_);
                const int e = min(ln + 64 * i, QW * PE - 1);
                const int s = e / PE, t = e - s * PE;
                const int c0 = at_slot(cf0, s), d0 = at_slot(df0, s);
                const double *M;
                size_t off;
                if (t < 2 * NCD) {
                    const int j = t < NCD ? t : t - NCD;
                    M = t < NCD ? Qm : P;
                    off = elem(c0 + j / ND, nb, d0 + j % ND);
                } else {
                    int x = t - 2 * NCD;
                    const bool second = NK == 2 && x >= S::NX;
                    if (second) x -= S::NX;
                    M = second ? KD[1] : KD[0];
                    const int r = x / NCX, col = x - r * NCX;
                    off = elem(r < NA ? bf0 + r : bf1 + r - NA, nb, col < NC ? c0 + col : d0 + col - NC);
                }
                st[i] = M[off];
            });
        }
        const unsigned g2 = next(g1);
        load_fields(g1);
        load_ids(g2);

        double acc[RPL][NF];
        sfor<0, RPL>([&](auto k_) { sfor<0, NF>([&](auto j_) { acc[PK_CI(k_)][PK_CI(j_)] = 0.0; }); });
        for (int kq = 0, kp = 0; more;) {
            {
                if (kp == 0) load_q(kq);
                prep(kp);
                const PrimDev *pp = a.prims + (bpo + kp);
                const double pz = uload(&pp->zeta), pkc = uload(&pp->kc), hp = uload(a.hz + bpo + kp);
                double val = cheb<double>(cc, xc);
                if (!(T < pk_rys_tmax[NR])) {
                    const double s = rsqrt_nr(T);
                    val = lim * (ax == 1 ? s : s * s);
                }
                const double u = __shfl(val, lane - ax, 64);
                const double w = __shfl(val, lane - ax + 1, 64);
                const double inv_de = rs * rs, roz = qz * inv_de, roe = pz * inv_de;
                const double ppa = sel3d(ax, uload(&pp->pa[0]), uload(&pp->pa[1]), uload(&pp->pa[2]));
                wave_fence();  // the rows of the previous primitive quartet have been read
                if (live_a)
                    axis_rows<LA, LB, S::F, RL>(ax == 0 ? pkc * qkc * rs * w : 1.0, fma(-u * roz, PQa, ppa),
                                            fma(u * roe, PQa, qpa), 0.5 * inv_de * u, hp * (1.0 - roz * u),
                                            hq * (1.0 - roe * u), ABq, Ga);
                wave_fence();
            }
            if (++kp == np) {
                kp = 0;
                ++kq;
                more = __any(kq < nqa);
            }
#pragma unroll 1
            for (int r = 0; r < NR; ++r) {
                const double *Gr = G + r * 3 * NGP;
                sfor<0, RPL>([&](auto k_) {
                    constexpr int k = PK_CI(k_);
                    double gq[3][S::F + 1];
                    sfor<0, 3>([&](auto q_) {
                        const double *src = Gr + ro[k][PK_CI(q_)];
                        sfor<0, S::F + 1>([&](auto i_) { gq[PK_CI(q_)][PK_CI(i_)] = src[PK_CI(i_)]; });
                    });
                    sfor<0, NF>([&](auto j_) {
                        constexpr int j = PK_CI(j_);
                        constexpr int lf = flat_level(LC, j), kf = flat_k(LC, j);
                        constexpr int x = cart_x(lf, kf), y = cart_y(lf, kf), z = cart_z(lf, kf);
                        acc[k][j] = fma(gq[0][x] * gq[1][y], gq[2][z], acc[k][j]);
                    });
                });
            }
        }
        // the staged densities into LDS, over the factors
        wave_fence();
        sfor<0, EPL>([&](auto i_) {
            constexpr int i = PK_CI(i_);
            if (64 * (i + 1) <= QW * PE || lane + 64 * i < QW * PE) G[lane + 64 * i] = st[i];
        });
        wave_fence();
        qoff = n_qoff, nqa = n_nq;
        more = np > 0 && g1 < kend && __any(nqa > 0);
        // ---- digestion
        double *JB = G + QW * PE;
        sfor<0, RPL>([&](auto k_) {
            constexpr int k = PK_CI(k_);
            const double *D = G + sb[k] * PE;
            double v[NCD];
            hrr_step<double, LC, LD, 0>(acc[k], cd[k], v);
            if (__all(bqmin * kqmin[k] >= a.tol)) {
                sfor<0, NCD>([&](auto j_) { v[PK_CI(j_)] *= deg[k]; });
            } else {
                sfor<0, NCD>([&](auto j_) { v[PK_CI(j_)] *= Qab[k] * D[PK_CI(j_)] >= a.tol ? deg[k] : 0.0; });
            }
            // J_ab
            sfor<0, NCD>([&](auto j_) { jab[k] = fma(v[PK_CI(j_)], D[NCD + PK_CI(j_)], jab[k]); });
            // exchange: rows a and b of the bra, columns of the ket's shells
            auto exch = [&](auto sp_, auto emit) {
                constexpr int sp = PK_CI(sp_);
                const double *Xa = D + 2 * NCD + sp * S::NX + (af_[k] - bf0) * NCX;
                const double *Xb = D + 2 * NCD + sp * S::NX + (NA + bf_[k] - bf1) * NCX;
                // B_ac += sum_bd v P_bd, B_bc += sum_ad v P_ad
                sfor<0, NC>([&](auto c_) {
                    constexpr int c = PK_CI(c_);
                    double x = 0.0, y = 0.0;
                    sfor<0, ND>([&](auto d_) {
                        constexpr int d = PK_CI(d_);
                        x = fma(v[c * ND + d], Xb[NC + d], x);
                        y = fma(v[c * ND + d], Xa[NC + d], y);
                    });
                    if constexpr (RUN) {
                        kca[sp][k][c] += x;
                        kcb[sp][k][c] += y;
                    } else {
                        cadd(sp, k, af_[k] - bf0, c, x);
                        cadd(sp, k, NA + bf_[k] - bf1, c, y);
                    }
                });
                __builtin_amdgcn_sched_barrier(0);
                // B_ad += sum_bc v P_bc, B_bd += sum_ac v P_ac
                sfor<0, ND>([&](auto d_) {
                    constexpr int d = PK_CI(d_);
                    double x = 0.0, y = 0.0;
                    sfor<0, NC>([&](auto c_) {
                        constexpr int c = PK_CI(c_);
                        x = fma(v[c * ND + d], Xb[c], x);
                        y = fma(v[c * ND + d], Xa[c], y);
                    });
                    emit(ka_[k], af_[k], d, x);
                    emit(kb_[k], bf_[k], d, y);
                });
                __builtin_amdgcn_sched_barrier(0);
            };
            if (deg[k] != 0.0) {
                sfor<0, NK>([&](auto s_) {
                    constexpr int sp = PK_CI(s_);
                    if (segmode)
                        exch(s_, [&](int r, int, int d, double x) {
                            __hip_atomic_fetch_add(&krow[sp * NROW * kc + r + df0[k] - dbase + d], x, __ATOMIC_RELAXED,
                                                   __HIP_MEMORY_SCOPE_WORKGROUP);
                        });
                    else
                        exch(s_, [&](int, int rf, int d, double x) {
                            unsafeAtomicAdd(&Bg[sp][(size_t)rf * nb + df0[k] + d], x);
                        });
                });
            }
            sfor<0, NCD>([&](auto j_) { v[PK_CI(j_)] *= Pab[k]; });
            // J_cd: sum over the rows of each slot through LDS, JC components at a
            // time; the slots of this k are those whose rows lie in [64 k, 64 k + 64)
            // (RPL = 1), or summed by partial rows
            constexpr int JC = S::jc(NK), JS = S::JS, NJP = (NCD + JC - 1) / JC;
            int ln = lane;
            asm volatile("" : "+v"(ln));
            sfor<0, NJP>([&](auto p_) {
                constexpr int j0 = PK_CI(p_) * JC, jn = NCD - j0 < JC ? NCD - j0 : JC;
                constexpr int R0 = 64 * k, R1 = (S::NRT < 64 * (k + 1) ? S::NRT : 64 * (k + 1));  // rows of the wave held in this k
                wave_fence();
                if (live[k]) sfor<0, jn>([&](auto j_) { JB[PK_CI(j_) * JS + ln] = v[j0 + PK_CI(j_)]; });
                wave_fence();
                // slots with rows in this k
                constexpr int S0 = R0 / RN, S1 = (R1 + RN - 1) / RN;
                constexpr int OUT = (S1 - S0) * jn;
                constexpr int SH = OUT * 8 <= 64 ? 3 : (OUT * 4 <= 64 ? 2 : (OUT * 2 <= 64 ? 1 : 0));
                constexpr int LP = 1 << SH;
                sfor<0, (OUT * LP + 63) / 64>([&](auto o_) {
                    const int o = (ln + 64 * PK_CI(o_)) >> SH, part = ln & (LP - 1);
                    const bool on = o < OUT;
                    const int so = on ? o / jn : 0, j = on ? o - so * jn : 0, s = S0 + so;
                    // rows of slot s within this k
                    const int r0 = max(s * RN, R0) - R0;
                    const int r1 = min(s * RN + min(RN, NAB - row0), R1) - R0;
                    const int c0 = __shfl(cf0[k], r0, 64), d0 = __shfl(df0[k], r0, 64);
                    const double *src = JB + j * JS;
                    double x = 0.0;
                    for (int i = r0 + part; i < r1; i += LP) x += src[i];
                    sfor<0, SH>([&](auto h_) { x += __shfl_xor(x, 1 << PK_CI(h_), 64); });
                    if (on && part == 0 && g0 + s < kend) {
                        const int q = j0 + j;
                        unsafeAtomicAdd(&Am[(size_t)(c0 + q / ND) * nb + d0 + q % ND], 2.0 * x);
                    }
                });
            });
        });
        wave_fence();
        g0 = g1;
        g1 = g2;
    }
    flush_run();
    // J_ab of the wave's rows
    sfor<0, RPL>([&](auto k_) {
        constexpr int k = PK_CI(k_);
        if (live[k])
            __hip_atomic_fetch_add(&jrow[(af_[k] - bf0) * NB + bf_[k] - bf1], jab[k], __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_WORKGROUP);
    });
    __syncthreads();
    if (segmode) {
        const int per = NROW * ncols;
        for (int i = threadIdx.x; i < NK * per; i += blockDim.x) {
            const int sp = i / per, rc = i - sp * per;
            const int r = rc / ncols, col = rc - r * ncols;
            const double x = krow[(sp * NROW + r) * kc + col];
            if (x != 0.0) {
                const int rf = r < NA ? bf0 + r : bf1 + (r - NA);
                unsafeAtomicAdd(&Bg[sp][(size_t)rf * nb + dbase + col], x);
            }
        }
    }
    for (int i = threadIdx.x; i < NAB; i += blockDim.x) {
        const double x = jrow[i];
        if (x != 0.0) unsafeAtomicAdd(&Am[(size_t)(bf0 + i / NB) * nb + bf1 + i % NB], 2.0 * x);
    }
}

template <int LA, int LB, int LC, int LD, int NK>
__global__ __launch_bounds__(256, (RowCls<LA, LB, LC, LD>::NF > 36 ? 1 : 2)) void k_rows(JKArgs a) {
    extern __shared__ double smem[];
    int blk = blockIdx.x;
    if (a.remap) {
        const int per = gridDim.x >> 3;
        blk = (blk & 7) * per + (blk >> 3);
    }
    if (blk >= a.nwaves) return;  // the whole workgroup
    rows_run<LA, LB, LC, LD, NK>(a, blk, (int)blockIdx.y, smem);
}

}  // namespace pk
