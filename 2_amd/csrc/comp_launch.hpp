// comp_launch.hpp -- what the launchers of the composite-radix passes share.
#pragma once

#include <algorithm>

#include "comp_tiles.hpp"

namespace mmx {

// x and y passes: 256 threads, two waves per SIMD at least.
#define MMX_COMP_KERNEL __global__ void __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(2)))

template <typename K> static void comp_lds(K kernel, size_t bytes)
{
    if (bytes > 65536)
        (void)hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
}

constexpr size_t kCompLds = 64 * 1024;
constexpr size_t kLdsMax = 160 * 1024;

// Workgroups wanted resident at once: four per CU.
constexpr long kCompSlots = 1024;

// DFTs of the stage that has most of them (smallest radix)
inline int comp_tasks(const CompFFT &f, int lines)
{
    int t = 1;
    for (int s = 0; s < f.ns; s++) t = std::max(t, lines * (f.L / f.R[s]));
    return t;
}
// Columns per workgroup (log2): 16, 128 bytes of a row, within 64 KB (two take
// what they need: films of 1000 and 1024 rows 66 and 77 us, with one column 90
// and 101).  Fewer
// while a stage has more than 256 DFTs and all workgroups are still resident
// at once (several small ones overlap better on a CU), and while there are
// fewer workgroups than CUs.
template <typename F> static int comp_cols(const CompFFT &f, int ncomp, F lds, long nlines, int h2)
{
    auto blocks = [&](int lw) { return nlines * div_up(h2, 1 << lw); };
    int lw = 4;
    while (lw > 1 && lds(lw) > kCompLds) lw--;
    while (lw > 0 && lds(lw) > kLdsMax) lw--;
    while (lw > 2 && comp_tasks(f, ncomp << lw) > kBlock && blocks(lw - 1) <= kCompSlots) lw--;
    while (lw > 2 && blocks(lw) < 256) lw--;
    return lw;
}

} // namespace mmx
