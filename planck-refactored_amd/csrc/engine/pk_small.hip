// pk_small.hip — instantiates k_small of set PK_SHARD (see the Makefile).
#include "eri_small.h"

template <>
const void *pk_small_kernel<PK_SHARD>() {
    return (const void *)pk::k_small<PK_SHARD>;
}
