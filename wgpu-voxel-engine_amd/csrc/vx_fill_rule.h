// vx_fill_rule.h -- which chunks the fast density fill takes, and with which
// compiled variant.  Plain C++ (no HIP), shared by the host runtime and the
// kernels and checked on the CPU.
#pragma once

#include <stdint.h>

namespace vx {

// Octaves the fast fill is compiled for: the variants.  Octaves a terrain
// does not have get amplitude 0.
constexpr int kFastVariants[] = {2, 3, 4, 6, 8};

// Columns a lane holds at once, by edge, the kernel's largest edge and
// variant: four columns share a row's terms while their coefficients (4 per
// octave and column) leave four waves per SIMD.  Terrains of more octaves
// have fine cells, whose tables fit more rows with one column per lane.
constexpr int fast_cols(int edge, int max_edge, int variant) {
    return edge == 16 || variant > 4 ? 1 : edge == 64 || max_edge == 64 ? 2 : 4;
}

// Table entries (16 B each) of a wave: 23 KB of tables per workgroup (13 KB
// beside a 64^3 slab) let four workgroups share a CU's 160 KB of LDS.
constexpr int fast_tab(int max_edge) { return max_edge == 64 ? 208 : 368; }

// Rows (layers times lines) of a chunk that a workgroup holds at once: a
// quarter of a 64^3 chunk's (8 KB instead of 32 KB), a smaller chunk's all.
constexpr int fast_rows(int max_edge) { return max_edge == 64 ? 1024 : max_edge * max_edge; }

// Workgroups per 64^3 chunk of the fast fill in a batch of n chunks, 4 at least
// (fast_rows).  1,024 run at once: at 323 chunks 4 are 1,292, a second round
// that is nearly empty; 8 take 103 us, 16 107 us.  A ragged batch of 2,048
// takes 73 us with 4 and 13 us more with 8: nothing is left to even out, and
// each workgroup lays its terms out anew.
constexpr int fill64_parts_for(int n) { return n >= 1024 ? 4 : n >= 128 ? 8 : 16; }

// The variant that takes a density chunk, or 0 for the general kernels.  The
// fast fill needs
//   - octave frequencies up to 0.75: above, nearly every row enters a new
//     cell and tables of cells do not pay;
//   - |coordinate * frequency| below 2^22: lattice cells are then exact
//     integers whose differences count table entries;
//   - finite amplitudes whose sum stays far from overflow: no infinity or NaN
//     then enters the comparisons;
//   - the tables of one row within a wave's share of LDS, in a kernel of any
//     largest edge: the variants above 4 octaves hold half the columns, so a
//     terrain of few octaves whose finest is dense may take one of those.
inline int32_t fast_variant(int32_t octaves, float frequency, float lacunarity, float gain,
                            int32_t cx, int32_t cy, int32_t cz, int32_t edge) {
    const int32_t c[3] = {cx, cy, cz};
    float reach = 0.0f;
    for (int32_t v : c) {
        const float a = (float)((int64_t)v * edge), m = a < 0 ? -a : a;
        reach = m > reach ? m : reach;
    }
    reach += (float)edge;
    float f = frequency, amp = 1.0f, sum = 0.0f;
    int points = 0;  // lattice points of a line, all octaves
    for (int o = 0; o < octaves; o++) {
        if (!(f <= 0.75f) || !(reach * f < 4194304.0f)) return 0;
        // the cells a line spans: one more for its position within a cell,
        // one for the coordinates' rounding, and the far corner
        points += (int)((float)edge * f) + 3;
        sum += amp < 0 ? -amp : amp;
        f = f * lacunarity;
        amp = amp * gain;
    }
    if (!(sum < 1e30f)) return 0;
    for (int v : kFastVariants) {
        if (v < octaves) continue;
        const int p = points + 2 * (v - octaves);
        bool fits = true;
        for (int m = edge; m <= 64; m *= 2)
            fits &= 2 * p * (64 / edge) * fast_cols(edge, m, v) <= fast_tab(m);
        if (fits) return v;
    }
    return 0;
}

}  // namespace vx
