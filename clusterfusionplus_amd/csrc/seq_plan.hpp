// What the kernels of a portion of the sequence models are launched with, from sizes alone.  Plain C++ without the device's headers, so
// that the choices can be looked at on the host.
#pragma once
#include <stddef.h>

#include <algorithm>

namespace cfpp {

inline int up_to(int a, int b) { return (a + b - 1) / b * b; }
inline int ceil_div(int a, int b) { return (a + b - 1) / b; }

// Attention of a portion of T tokens at positions pos0 and on: R query heads for each of G key / value heads, `keys` of them in a tile.
struct AttnSizes {
    int T, R, G, pos0, chunk, keys;
    bool pairs;              // bf16: two column tiles per wave are possible
    int per_cu;              // workgroups that share a compute unit
    size_t floats;           // of a split's partial results
};
// Columns of a workgroup and splits of the keys.  bf16: two column tiles per wave share the reads of keys and values; one, where that
// leaves fewer columns empty or where two workgroups per compute unit are not reached.  Splits fill the chip: two workgroups per
// compute unit, with two tiles at least in each split of the longest walk, which begins at the chunk of the portion's first token (that
// chunk counts and not the context: 37 tokens just behind a chunk of 8192 see one tile; shared by 16 splits, eight layers of 32 / 8 heads
// of 128 took 1005 us, and take 957).
struct AttnPlan { bool two; int splits; };
inline AttnPlan plan_attn(const AttnSizes& a, int cus, size_t room) {
    const int cols = a.T * a.R, behind = a.pos0 + a.T - (a.chunk > 0 ? a.pos0 / a.chunk * a.chunk : 0);
    const int tiles = ceil_div(a.chunk > 0 ? std::min(behind, a.chunk) : behind, a.keys);
    const bool two = a.pairs && ceil_div(cols, 128) * a.G >= 2 * cus;
    const int wgs = ceil_div(cols, two ? 128 : 64) * a.G;
    return {two, std::max(1, (int)std::min<size_t>({(size_t)16, (size_t)(a.per_cu * cus / wgs), (size_t)(tiles / 2), room / a.floats}))};
}

}  // namespace cfpp
