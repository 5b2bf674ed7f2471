// pk_grad.hip — instantiates the gradient kernels of the ordered classes (bra
// pair class, ket pair class) of shard PK_SHARD (compiled once per shard, see
// the Makefile).
#include "eri_grad.h"
#include "grad_table.h"

namespace {

template <int CB, int CK>
void add(pk::GradEntry *table) {
    if constexpr ((CB * PK_GRAD_PAIRS + CK) % PK_NGRADSHARDS == PK_SHARD) {
        constexpr int A = pk::pair_la(CB), B = pk::pair_lb(CB), C = pk::pair_la(CK), D = pk::pair_lb(CK);
        using S = pk::GradCls<A, B, C, D>;
        table[CB * PK_GRAD_PAIRS + CK] =
            pk::GradEntry{(const void *)pk::k_grad<A, B, C, D, 1>, (const void *)pk::k_grad<A, B, C, D, 2>,
                          {(int)(S::gd(1) * sizeof(double)), (int)(S::gd(2) * sizeof(double))}, S::QW, S::RC};
    }
}

}  // namespace

template <>
void pk_grad_register<PK_SHARD>(pk::GradEntry *table) {
    pk::sfor<0, PK_GRAD_PAIRS * PK_GRAD_PAIRS>(
        [&](auto i_) { add<PK_CI(i_) / PK_GRAD_PAIRS, PK_CI(i_) % PK_GRAD_PAIRS>(table); });
}
