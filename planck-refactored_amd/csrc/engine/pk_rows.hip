// pk_rows.hip — instantiates the row kernels of the classes of shard PK_SHARD
// (compiled once per shard, see the Makefile).
#include "eri_classes.h"
#include "eri_rows.h"
#include "rows_table.h"

namespace {

template <int A, int B, int C, int D, int CLS>
void add(pk::RowsEntry *table) {
    if constexpr (CLS % PK_NROWSHARDS == PK_SHARD && pk::small_rows(A, B, C, D)) {
        using S = pk::RowCls<A, B, C, D>;
        table[CLS] = pk::RowsEntry{(const void *)pk::k_rows<A, B, C, D, 1>, (const void *)pk::k_rows<A, B, C, D, 2>,
                                   {(int)(S::wave_doubles(1) * sizeof(double)), (int)(S::wave_doubles(2) * sizeof(double))},
                                   S::QW, S::RC};
    }
}

}  // namespace

template <>
void pk_rows_register<PK_SHARD>(pk::RowsEntry *table) {
#define PK_ADD(a, b, c, d, shard) \
    add<a, b, c, d, pk::pair_class(a, b) * (pk::pair_class(a, b) + 1) / 2 + pk::pair_class(c, d)>(table);
    PK_FOR_EACH_CLASS(PK_ADD)
#undef PK_ADD
}
