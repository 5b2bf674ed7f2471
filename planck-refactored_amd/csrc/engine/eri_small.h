// eri_small.h — one launch for many short class lists.
//
// The build of a small molecule has twenty to fifty class lists of a few waves
// each; launched one by one, every list costs its own launch and the latency of
// its first loads, and the chip is empty in between (one water, 6-31G*: 21 lists
// of 12-30 us).  Here one workgroup of one wave takes one wave (per-lane
// Obara-Saika classes) or one work item (row kernels) of any of the lists: the
// class is a switch on a uniform value, the registers those of the largest class,
// which does not matter where the waves are few.  Plain mode: every exchange sum
// a global atomic.  H2O / 6-31G* 0.76 -> 0.08 ms per build.
#pragma once

#include "eri_classes.h"
#include "eri_rows.h"
#include "small_table.h"

namespace pk {

template <int A, int B, int C, int D>
__device__ __forceinline__ void small_item(const JKArgs &a, int item, double *smem) {
    if constexpr (small_os(A, B, C, D)) {
        jk_run<double, A, B, C, D, ALG_OS, 0, ncart(C) * ncart(D), 1, false>(a, item, item + 1, 1, item, smem);
    } else {
        constexpr int RC = RowCls<A, B, C, D>::RC;
        rows_run<A, B, C, D, 1>(a, item / RC, item % RC, smem);
    }
}

// SET 0: classes of s, p, d shells; 1: classes with an f shell.
template <int SET>
__global__ __launch_bounds__(64, 2) void k_small(JKArgs a, const SmallList *__restrict__ lists, SmallTab tab) {
    extern __shared__ double smem[];
    const int b = blockIdx.x;
    int l = 0;
    while (l + 1 < tab.n && b >= tab.first[l + 1]) ++l;
    const SmallList *s = lists + tab.list[l];
    const int item = b - tab.first[l], nw = uload(&s->nwaves);
    const int *wave = (const int *)uload(&s->wave);
    a.wave_bra = wave;
    a.wave_start = wave + nw;
    a.wave_count = wave + 2 * (size_t)nw;
    a.wave_mol = wave + 3 * (size_t)nw;
    a.kets = (const int *)uload(&s->kets);
    a.nwaves = nw;
    a.chunk = uload(&s->chunk);
    a.segmode = 0;
    switch (uload(&s->cls)) {
#define PK_CASE(A, B, C, D, shard)                                                                    \
    case pair_class(A, B) * (pair_class(A, B) + 1) / 2 + pair_class(C, D):                            \
        if constexpr (small_class(A, B, C, D) && (A == 3) == (SET == 1)) small_item<A, B, C, D>(a, item, smem); \
        break;
        PK_FOR_EACH_CLASS(PK_CASE)
#undef PK_CASE
    }
}

}  // namespace pk
