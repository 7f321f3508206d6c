// coo_entries.hpp -- places of an element's COO entries (build_system_elemStorage.f90:260-293): node b's row
// of blocks (a, b), a <= b, follows those of the nodes before it, a block column-major, of the diagonal
// block the 6 upper entries.
#pragma once

#include <cstdint>

namespace yeti {

// first entry of node b's row
__host__ __device__ constexpr int coo_start(int b) { return (9 * b * b + 3 * b) / 2; }

// dofs of entry x of an element of up to 64 nodes: 3 a + kk | (3 b + ll) << 8
constexpr int ENTRY_NODES = 64;

struct EntryTab {
    alignas(16) uint16_t v[coo_start(ENTRY_NODES)];
    constexpr EntryTab() : v() {
        int x = 0;
        for (int b = 0; b < ENTRY_NODES; ++b)
            for (int a = 0; a <= b; ++a)
                for (int l = 0; l < 3; ++l)
                    for (int k = 0; k < (a < b ? 3 : l + 1); ++k) v[x++] = (uint16_t)((3 * a + k) | (3 * b + l) << 8);
    }
};
__device__ constexpr EntryTab entry_tab{};

}  // namespace yeti
