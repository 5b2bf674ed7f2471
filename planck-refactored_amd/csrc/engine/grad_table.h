// grad_table.h — the gradient kernels (eri_grad.h) as the host side sees them.
#pragma once

namespace pk {

struct GradEntry {
    const void *k1, *k2;  // kernels with one and two exchange densities
    int lds[2];           // LDS bytes of each
    int qw;               // quartets per wave
    int rc;               // row chunks (grid y)
};

// angular momenta (la >= lb) of pair class c
constexpr int pair_la(int c) {
    int l = 0;
    while ((l + 1) * (l + 2) / 2 <= c) ++l;
    return l;
}
constexpr int pair_lb(int c) { return c - pair_la(c) * (pair_la(c) + 1) / 2; }

}  // namespace pk

#define PK_GRAD_PAIRS 10  // pair classes of s, p, d, f shells
#define PK_NGRADSHARDS 8
// fills the entries (bra class * PK_GRAD_PAIRS + ket class) of one shard; defined in pk_grad.hip
template <int SHARD>
void pk_grad_register(pk::GradEntry *table);
