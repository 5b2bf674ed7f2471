// small_table.h — the one-launch kernels for short lists (eri_small.h) as the
// host side sees them.
#pragma once

namespace pk {

// A list in device memory: its waves [4][nwaves], kets and class.
struct SmallList {
    const int *wave, *kets;
    int nwaves, cls, chunk;
};

// Lists of one launch: first block and index of each.
struct SmallTab {
    int n;
    int first[55], list[55];
};

// Obara-Saika class of the launch (as the engines os and auto run it)
constexpr bool small_os(int la, int lb, int lc, int ld) { return os_available(la, lb, lc, ld); }
// classes the launch covers: the Obara-Saika classes, and rows of up to 36
// components (fd and ff kets would cost all of them registers)
constexpr bool small_class(int la, int lb, int lc, int ld) {
    return small_os(la, lb, lc, ld) || (small_rows(la, lb, lc, ld) && nlev(lc, lc + ld) <= 36);
}

}  // namespace pk

// kernel of a set (0: s, p, d shells; 1: with f shells); defined in pk_small.hip
template <int SET>
const void *pk_small_kernel();
