// vx_fill_rule.h -- which chunks the fast density fill takes, with which
// compiled variant, and how many workgroups fill a chunk.  Plain C++ (no HIP),
// shared by the host runtime and the kernels and checked on the CPU.
#pragma once

#include <stdint.h>

#include <initializer_list>

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

// True if every voxel coordinate of the frequency lies on one of at most 64
// positions in a cell (f is a multiple of 1/q), or cells are larger than 64 voxels.
inline bool on_lattice(float f) {
    if (f < 1.0f / 64) return true;
    for (int q = 1; q <= 64; q++) {
        const float p = f * (float)q, d = p - (float)(int)(p + 0.5f);
        if (d < 1e-5f && d > -1e-5f) return true;
    }
    return false;
}

// Whether a chunk that fast_variant accepts gains from it in a batch of n
// chunks of edges up to max_edge (one chunk alone always does: the general
// kernel has one workgroup for it).  zero: the threshold is zero at every
// layer (reference rule, y_scale 0).  From the fill times of 1 to 2,000 chunks
// of each edge, general / fast:
//   - above 4 octaves the general kernels evaluate octave by octave: 1.1 to 30.
//   - Up to 4, their rows share a column's terms while its cell lasts, and
//     tables gain less the more cells a chunk has.  At a finest frequency of
//     0.32 / 0.35 / 0.41 / 0.45 / 0.5: 32^3 of 1 and 2 octaves 1.05 / 1.0 / 0.9 / 0.75 /
//     0.8; of 3 0.95 / 1.0 / 1.0 / 1.0 / 0.8 (1.2 at 0.35 from 512 chunks on), of 4 1.15 /
//     1.2 / 1.1 / 1.15 / 0.85 (0.9 at 0.45 from 1,024 on); 64^3 of 1, 3 and 4 1.3 to 2 /
//     1.0 to 2 / 1.0 to 1.9 / 0.75 to 1.3 / 0.6 to 1.2, of 2 1.5 / 1.4 / 1.1 / 1.25 / 0.6.
//   - A zero threshold meets noise that is exactly zero wherever a voxel lies
//     on a lattice plane of every octave, and those rows are evaluated twice:
//     one octave 0.4 to 1.05 (off the lattice 1.0 to 1.8 up to 0.25, at 64^3 up to
//     0.35), two 0.95 to 1.25 up to 0.1, at 0.125 0.85 to 0.95 (1.2 from 1,024 chunks
//     on) and 0.4 to 0.75 from 0.25 on (64^3 1.0 to 1.3), three and four as other
//     terrains.  Where all cells are larger than 50,000 voxels it is zero nearly
//     everywhere: 0.85.
//   - 16^3 chunks pay for a chunk's tables over a quarter of the lines: 0.6 to
//     1.05 below 384 chunks (one octave 0.8 to 1.0 at any number; four octaves of
//     1 to 8 chunks 1.05 to 1.2), then 0.95 to 1.3, on a lattice at threshold zero
//     0.5 to 1.0 below 1,024.
inline bool fast_pays(int32_t octaves, float frequency, float lacunarity, bool zero, int32_t edge,
                      int32_t max_edge, int32_t n) {
    float f = frequency, fine = 0.0f;
    bool lattice = zero && octaves <= 4;
    for (int o = 0; o < octaves; o++) {
        fine = f > fine ? f : fine;
        lattice = lattice && on_lattice(f);
        f = f * lacunarity;
    }
    if (zero && fine < 2e-5f) return false;
    if (octaves > 4) return true;
    if (max_edge <= 16) {
        if (octaves == 1) return false;
        if (octaves == 4 && !zero && n <= 8) return true;
        return lattice ? octaves == 4 && n >= 1024 : n >= 384;
    }
    if (edge == 64) {
        if (zero && octaves == 1) return !lattice && fine <= 0.36f;
        return fine <= (octaves == 2 || n <= 16 ? 0.47f : 0.42f);
    }
    if (zero && octaves == 1) return !lattice && fine <= 0.25f;
    if (lattice && octaves == 2) return fine <= (n >= 1024 ? 0.125f : 0.1f);
    if (octaves == 4) return fine <= (n >= 1024 ? 0.42f : 0.46f);
    return fine <= (octaves == 3 && n >= 512 ? 0.38f : 0.325f);
}

// ---- workgroups per chunk
constexpr int kFillGrid = 1024;  // fill workgroups that fill the GPU (4 per CU)

// Chunks of a batch by kernel: fast ones (a variant set), general ones.
struct FillMix {
    int32_t fast = 0, general = 0;
    void add(int32_t variant) { (variant ? fast : general)++; }
};

// Workgroups per chunk of n chunks: one for kFillGrid or more; below that 2, 4
// or 8 so that the grid still covers about kFillGrid workgroups (8 only for at
// most kFillGrid / 8 chunks that hold 64^3 ones).  `hint` (1, 2, 4 or 8; 0 =
// this rule) replaces the rule where it would split.
constexpr int fill_parts_for(int32_t n, int32_t max_edge, int32_t hint = 0) {
    if (n >= kFillGrid) return 1;
    if (hint > 0) return hint;
    return 2 * n >= kFillGrid ? 2 : (max_edge > 32 && 8 * n <= kFillGrid) ? 8 : 4;
}

// Workgroups per chunk that each fill kernel takes on a batch of n chunks (0 =
// it has none): the fast one by all n, with 64^3 chunks fill64_parts_for or a
// hint of 4 at least; the general one as a batch of its chunks alone would (64
// of them among 512 filled in 70 us with the batch's two, in 41 with their four).
// Batches of kFillGrid chunks and more ignore the hint.
struct FillShape {
    int fast, general;
};
constexpr FillShape fill_shape(int32_t n, int32_t max_edge, FillMix mix, int32_t hint) {
    const int32_t h = n < kFillGrid ? hint : 0, general = mix.general < n ? mix.general : n;
    const int fast = max_edge <= 32 ? fill_parts_for(n, max_edge, h)
                     : h            ? (h > 4 ? h : 4)
                                    : fill64_parts_for(n);
    return FillShape{mix.fast > 0 ? fast : 0, general > 0 ? fill_parts_for(general, max_edge, h) : 0};
}

// True iff each chunk of a batch of edges up to 32 gets one workgroup, so that
// FillWork.count_out is honoured for every chunk (whatever the hint).
constexpr bool fill_whole_chunks(int32_t n, FillMix mix) {
    return n >= kFillGrid && (mix.general == 0 || mix.general >= kFillGrid);
}

// Hints worth timing on a batch: half and twice what the rule gives each of its
// kernels (four at most up to edge 32, eight beyond), without those that come
// to a shape that another, or the rule, has already.  At most 4; their number.
constexpr int tune_fill_hints(int32_t n, int32_t max_edge, FillMix mix, int32_t hints[4]) {
    if (n >= kFillGrid) return 0;
    FillShape seen[5] = {fill_shape(n, max_edge, mix, 0)};
    int k = 0;
    for (const int parts : {seen[0].general, seen[0].fast})
        for (const int h : {parts / 2, parts * 2}) {
            if (h < 1 || h > (max_edge > 32 ? 8 : 4)) continue;
            const FillShape s = fill_shape(n, max_edge, mix, h);
            bool known = false;
            for (int i = 0; i <= k; i++) known |= seen[i].fast == s.fast && seen[i].general == s.general;
            if (known) continue;
            hints[k++] = h;
            seen[k] = s;
        }
    return k;
}

}  // namespace vx
