// rows_table.h — the row kernels (eri_rows.h) as the host side sees them.
#pragma once

#include "eri_kernels.h"

namespace pk {

struct RowsEntry {
    // kernels with one and two exchange densities (null: the class has none)
    const void *k1 = nullptr, *k2 = nullptr;
    int wave_bytes[2] = {0, 0};  // LDS of one wave, with one and two exchange densities
    int qw = 1;          // quartets per wave
    int rc = 1;          // row chunks (grid y)
};

}  // namespace pk

// fills the entries of one shard's classes; defined in pk_rows.hip
#define PK_NROWSHARDS 8
template <int SHARD>
void pk_rows_register(pk::RowsEntry *table);
