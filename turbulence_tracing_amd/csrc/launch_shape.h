// Arithmetic of launch shapes, apart from the kernels (plain C++).
#pragma once

namespace tt {

// LDS of a CU, and the unit in which a block's share of it is given out.
constexpr int kLdsBytes = 160 * 1024, kLdsGranule = 1280;

// Dynamic LDS that keeps a CU to at most `blocks` blocks of a kernel without
// static LDS: the largest number of whole units of which `blocks` requests fit.
// Where blocks + 1 of them fit too (13 blocks, 15), one unit more, so that fewer
// stay resident rather than more.  160 KB / blocks as it is, rounded up to units
// by the hardware, left one block fewer at 3, 5, 6 and 7.
constexpr int lds_for_residency(int blocks) {
    constexpr int units = kLdsBytes / kLdsGranule;
    int u = units / blocks;
    if ((blocks + 1) * u <= units) ++u;
    return u * kLdsGranule;
}

}  // namespace tt
