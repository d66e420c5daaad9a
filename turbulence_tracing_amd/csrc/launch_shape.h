// Arithmetic of launch shapes, apart from the kernels (plain C++).
#pragma once
#include <cstdint>

namespace tt {

// A launch holds fewer than 2^32 threads along each axis of its grid: of one that
// asks for more, blocks go missing without an error.  More blocks than that go in
// rows of equal length; block (x, y) takes part
// y * gridDim.x + x, if there is one (some of the last row's may have none).
struct Blocks {
    uint32_t x, y;
};
constexpr Blocks spread(int64_t blocks, int threads) {
    const int64_t most = 0xffffffffll / threads;
    const int64_t rows = (blocks + most - 1) / most;
    return rows <= 1 ? Blocks{(uint32_t)blocks, 1u} : Blocks{(uint32_t)((blocks + rows - 1) / rows), (uint32_t)rows};
}

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
