// vx_internal.h -- structures shared by the host runtime (vx_api.cpp) and the
// gfx950 kernels (vx_kernels.hip).  Plain-old-data only: every struct here is
// copied byte-for-byte into device memory.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "vx_fill_rule.h"

namespace vx {

constexpr int kBlock = 256;        // threads per workgroup (4 wave64)
constexpr int kMaxOctaves = 8;     // fBm octaves supported by the noise tables
constexpr int kDescTile = 4096;    // face descriptors staged in LDS per emit tile
constexpr int kEmitGrid = 2560;    // emit workgroups that fill the GPU twice (5 per CU at once)
constexpr int kEmitThree = 1792;   // chunks of edge 32 up to which three workgroups each pay
constexpr int kEmitGrid64 = 6144;  // the same over slabs of 64^3 chunks (4 per CU at once)

// Terrain kinds (mirror of vx_terrain.kind in include/voxel.h).
enum : int32_t { kAir = 0, kSolid = 1, kHeightmap = 2, kDensity = 3, kReference = 4 };

// Block ids stored in the u8 voxel array: 0 air, 1 grass, 2 dirt.  The
// reference's CubeType is {GRASS=0, DIRT=1, AIR=2} (src/cube.rs:16-21).
enum : uint32_t { kBlockAir = 0, kBlockGrass = 1, kBlockDirt = 2, kBlockMixed = 0xFFu };

// Output formats (mirror of VX_FMT_* in include/voxel.h).
enum : uint32_t { kFmtInstances = 1u, kFmtVertices = 2u };

// Per-terrain constants, resident in device memory.  The permutation is the
// splitmix64/Fisher-Yates shuffle of 0..255 for the seed, doubled to 512.
struct TerrainDev {
    int32_t kind;
    int32_t octaves;
    float frequency;
    float lacunarity;
    float gain;
    float height_scale;
    int32_t height_max;
    float y_scale;
    int32_t perm[512];
};

// Per-hash gradient coefficients for the column-hoisted noise evaluation,
// indexed [corner k][hash & 15] with corner k = x | row << 1 | col << 2 (row
// = world y, the per-row axis; col = world z).  grad_k = fma(yr, g_row,
// a_x*xr + a_col*zr); the +-1 entries select and sign an operand, the zero
// entries are the signed zero that makes the product vanish exactly (-0
// when the operand is >= 0, +0 when it is < 0), so the sum equals Perlin's
// (+-u) + (+-v) bit for bit.
struct GradLut {
    float4 c[8][16];  // noise at (wx, wy, wz): (a_x, a_col, g_row) = (gx, gz, gy)
    float4 r[8][16];  // noise at (wx, wz, wy), the reference's axes: (gx, gy, gz)
};

// Meshing constants computed on the host from the rotation of each face
// direction (nalgebra from_euler_angles restated) and the translation sign:
//   P[d][r][s][corner] = ((M(r,0)*cx + M(r,1)*cy) + M(r,2)*cz)
//   Mb[d][s][r][c]     = M(r,c) of T*R for a translation component of sign s
//                        (c = 3 unused, zero)
// where s = 1 iff that translation component is negative.  The innermost
// four floats of each are what one face reads for one coordinate r: a
// single 16-byte LDS read.
struct MeshTables {
    alignas(16) float P[6][3][2][4];
    alignas(16) float Mb[6][2][3][4];
    uint32_t tex[3][6];  // [block id][dir] -> texture layer (row 0 unused)
};

// One chunk to fill: terrain -> ids, occupancy rows, boundary planes, meta.
struct FillWork {
    int32_t cx, cy, cz, edge;
    int32_t terrain;       // index into the terrain table
    int32_t variant;       // fill_variant: 0 = the general kernels, else the fast one's
    uint8_t *ids;          // edge^3
    uint32_t *occ;         // edge^2 rows * W words (W = 1 for edge <= 32, 2 for 64)
    uint32_t *planes;      // 4 planes * edge * W words: x=0, x=N-1, z=0, z=N-1
    uint32_t *meta;        // [0] solid block id (or kBlockMixed)
    float *noise_out;      // optional raw noise (density: edge^3, heightmap: edge^2)
    // Optional (one workgroup per chunk, edges up to 32): the fill also counts
    // the chunk's visible faces, for chunks whose every neighbour is absent
    // or was written before the launch.  cnb[k] = the plane of neighbour k
    // (-x, +x, -z, +z) facing this chunk, null = absent; count_out[0] = the
    // face count.
    const uint32_t *cnb[4];
    uint32_t *count_out;   // null: the count kernel counts
};

// One chunk to mesh.  nb[k] points at the neighbour's plane facing this
// chunk (k = -x, +x, -z, +z -> its x=N-1, x=0, z=N-1, z=0 plane) or is null
// when the neighbour is absent (chunk.rs:89-107: absent -> emit).
struct MeshWork {
    int32_t ox, oy, oz, edge;  // world origin of the chunk
    const uint32_t *occ;
    const uint8_t *ids;
    const uint32_t *nb[4];
    uint32_t solid_type;       // block id of every solid voxel, or kBlockMixed
    uint32_t pad0;
};

// Batch-wide mesh outputs.
struct MeshOut {
    float *vertices;      // 20 floats per face (4 x {pos xyz, uv})
    uint32_t *indices;    // 6 per face, chunk-local
    uint32_t *instances;  // 17 dwords per face (InstanceRaw)
    uint64_t capacity;    // faces
    uint32_t formats;
    uint32_t pad0;
};

// Fused noise -> cull -> compact: per-side source of the neighbour plane.
enum : uint32_t { kHaloAbsent = 0u, kHaloResident = 1u, kHaloRecompute = 2u };

// One chunk of the fused kernel: its fill outputs, its mesh description
// (m.nb[k] read for resident sides) and how each neighbour plane is obtained.
// kHaloRecompute is only used when that neighbour is the adjacent chunk of
// the same batch with the same terrain and edge, so the recomputed plane is
// bit-identical to the one the neighbour writes itself.
struct FusedWork {
    FillWork f;
    MeshWork m;
    uint32_t halo[4];
    int32_t nbi[4];  // batch index of each in-batch (kHaloRecompute) neighbour, else -1
};

// Control words of one fused run; zeroed by the reset kernel.
struct FusedCtl {
    uint32_t *ticket;    // next chunk to hand out (processing order = output order)
    uint64_t *status;    // per chunk: flag(2 bits) | face count or inclusive prefix
    uint32_t *counts;    // per chunk face count (for the host)
    uint64_t *bases;     // per chunk first face (for the host)
    uint64_t *total;     // faces of the whole batch
    uint32_t *overflow;  // set when a chunk did not fit the arena
    uint32_t *error;     // set when a look-back wait exceeded its bound
    uint32_t *filled;    // per chunk: its fill has published (pipelined form; may be null)
    uint32_t *mesh_ticket;  // next chunk to mesh (pipelined form; may be null)
};

// Frustum job carried by a fused launch: planes in device memory (updated
// per frame without re-capturing the graph), n chunk coordinates, edge,
// one mask byte per chunk.  n = 0 disables it.
struct CullJob {
    const float *planes;
    const int32_t *coords;
    uint8_t *mask;
    int32_t n;
    int32_t edge;
};

// Six frustum planes [near far left right top bottom] x (a b c d), passed
// to the cull kernel by value.
struct Planes {
    float p[24];
};

// Indirect draw arguments (the layout of vx_draw_indexed in include/voxel.h
// and of WebGPU's drawIndexedIndirect buffer).
struct DrawArgs {
    uint32_t index_count, instance_count, first_index;
    int32_t base_vertex;
    uint32_t first_instance;
};
enum : uint32_t { kDrawInstanced = 1u, kDrawExpanded = 2u };

// Variant of the fast fill for a chunk of terrain T (vx_fill_rule.h), 0 for
// the general kernels; chunks without 3-D noise always take the fast one.
inline int32_t fill_variant(const TerrainDev &T, int32_t cx, int32_t cy, int32_t cz, int32_t edge) {
    if (T.kind != kDensity && T.kind != kReference) return 1;
    return fast_variant(T.octaves, T.frequency, T.lacunarity, T.gain, cx, cy, cz, edge);
}

inline int words_per_row(int edge) { return (edge + 31) / 32; }

// ---- kernel launchers (vx_kernels.hip) --------------------------------
// Schedules: `order` (fill, emit) lists the n items in launch order, or is
// null for 0..n-1.  An entry outside [0, n) makes its workgroup do nothing
// and sets a sticky error word: `error` for the fill, overflow[1] for the
// emit, whose overflow[0] is the arena-overflow flag the scan clears.
// Workgroups per emit item, so that the last round of the 1,280 workgroups
// that run at once is short without many that only repeat an item's set-up.
// Edge 16 (700 faces an item, the set-up is most of it): one round, and at
// most four or a workgroup per CU; emits of 132 / 256 / 400 / 600 / 800 chunks
// take 15 / 17 / 18 / 19 / 23 us at 4 / 4 / 3 / 2 / 1 parts, against 22 / 21 / 24 /
// 25 / 31 at the rule of edge 32.  Edge 32: kEmitGrid workgroups, at most 15
// parts (512 chunks at 1 / 3 / 5 / 8 parts 127 / 95 / 94 / 101 us a pass), three up
// to kEmitThree, but for chunks of many faces (emit_shares; 1,640 chunks of
// instances at 1 / 3 parts 171 / 170 us density, 184 / 174 reference rule, 139 / 133
// heightmap), one beyond (with vertices 1 / 3 parts tie at 1,740 to 1,815 chunks, then
// three lose: 2,048 of the reference rule 232 / 244, density 225 / 232).  Slabs of 64^3 chunks hold more faces: kEmitGrid64 (1,292 slabs at 1 / 3 /
// 5 / 8 parts 430 / 386 / 364 / 416); without vertices seven at most from 256 slabs
// on (600 slabs at 3 / 7 / 11 parts 156 / 146 / 159 us density, 490 / 496 / 523 with
// 22,000 faces each; with vertices the latter prefer 11, 582 / 552); one at
// kEmitGrid items or more (two at 4,100 mixed items lose 15%).  Odd numbers above two: workgroups go round the 8
// XCDs, and an even number puts the same parts and slabs, which are not alike,
// on the same ones (1,600 slabs at 2 / 3 / 4 parts 347 / 304 / 346).  `hint` (1..4;
// 0 = this rule) replaces the rule below kEmitGrid items.
inline int emit_parts_for(int32_t items, int32_t max_edge, bool vertices, int32_t hint = 0) {
    if (items >= kEmitGrid) return 1;
    if (hint > 0) return hint;
    if (max_edge <= 16) {
        const int round = kEmitGrid / 2 / items, cus = 256 / items, most = cus > 4 ? cus : 4;
        return round < 1 ? 1 : round < most ? round : most;
    }
    if (max_edge <= 32 && 2 * items >= kEmitGrid) return items < kEmitThree ? 3 : 1;
    const int p = ((max_edge > 32 ? kEmitGrid64 : kEmitGrid) + items - 1) / items;
    const int most = max_edge > 32 && items >= 256 && !vertices ? 7 : 15;
    return p <= most ? (p - 1) | 1 : most;
}
// Whether the parts of a batch of n items share an item of F faces.  Where the
// items alone fill the GPU, several parts even out a last round of unequal
// items, but writing vertices and indices of many faces (104 B each) from
// three workgroups at once loses more: 1,640 chunks of 32^3 at 1 / 3 parts, 2,700
// faces each 163 / 155 us, 11,500 663 / 689, 28,000 1,424 / 1,481 (instances, 68 B, gain:
// 555 / 501 and 1,078 / 980).
constexpr uint32_t kEmitDense = 8192;
constexpr bool emit_shares(int32_t n, uint32_t F, bool vertices) {
    return !vertices || F < kEmitDense || 2 * n < kEmitGrid;
}
// parts_hint, mix (of the batch that the launch is of): fill_shape.
hipError_t launch_fill(const FillWork *work, const int32_t *order, int32_t n, int32_t max_edge,
                       const TerrainDev *terrains, const GradLut *lut, uint32_t *error,
                       int32_t parts_hint, FillMix mix, hipStream_t s);
// Batches that hold 64^3 chunks emit by items: each 64^3 chunk is kSlabs
// y-slabs of kSlabLayers layers (face counts per slab in slabs[kSlabs * i
// ..], written by the count kernel), any other chunk one item.  With `items`
// (the batch's mesh work) the scan's order lists item codes chunk << 2 |
// slab, at most kSlabs * n of them; launch_emit takes their number.
constexpr int kSlabs = 4;
// clear (may be null): a word the count sets to 0 (the overflow word of an
// emit that follows without a scan).  cull: a frustum job run beside it.
hipError_t launch_count(const MeshWork *work, int32_t n, int32_t max_edge, uint32_t *counts,
                        uint32_t *slabs, uint32_t *clear, const CullJob &cull, hipStream_t s);
// base_in (device, may be null): faces before these chunks, added to every
// base and to the total (the second half of a split batch).
hipError_t launch_scan(const uint32_t *counts, int32_t n, const MeshWork *items, uint64_t *bases,
                       uint64_t *total, uint32_t *overflow, int32_t *order_out, hipStream_t s,
                       const uint64_t *base_in = nullptr);
hipError_t launch_fill_one(const FillWork &w, const TerrainDev *terrains, const GradLut *lut,
                           hipStream_t s);
// solid_type: FillWork.meta[0], from the host's reading of the ids.
hipError_t launch_pack_one(const FillWork &w, uint32_t solid_type, hipStream_t s);
// slabs: kSlabs face counts of a 64^3 chunk, written by the count and read by
// the emit (smaller chunks do not use them).
hipError_t launch_count_one(const MeshWork &w, uint32_t *count, uint32_t *slabs, hipStream_t s);
hipError_t launch_emit_one(const MeshWork &w, uint32_t faces, const uint32_t *slabs, MeshOut out,
                           const MeshTables *tables, uint32_t *overflow, hipStream_t s);
// parts_hint: emit_parts_for's hint.  total (null: bases come from the scan):
// the emit sums the counts before each chunk itself, in batch order (order =
// null), and writes bases and *total; for batches of at most kSelfScan chunks.
hipError_t launch_emit(const MeshWork *work, const int32_t *order, int32_t n, int32_t n_items,
                       int32_t max_edge, uint64_t *bases, const uint32_t *counts,
                       const uint32_t *slabs, MeshOut out, const MeshTables *tables,
                       uint32_t *overflow, int32_t parts_hint, uint64_t *total, hipStream_t s);
// 4 us of launch and scan against sums that grow with n and the scan's
// largest-first order: 32^3 batches gain 3 to 5 us a pass up to 128 chunks, 1 to 4
// at 200 to 450, 0.5 to 4 at 512 (density to heightmap); 64^3 ones gain up to 9,
// but 256 of them lose 3 to 8.  At 600 to 1,000 some gain and some lose 3, 1,640 lose 6.
constexpr int kSelfScan = 512;
// Emit items of a batch: its chunks, or for batches that hold 64^3 chunks
// kSlabs per 64^3 chunk and one per other chunk.
inline int32_t emit_items_of(int32_t n, int32_t n_items, int32_t max_edge) {
    return max_edge <= 32 ? n : n_items;
}
hipError_t launch_fused(const FusedWork *work, int32_t n, int32_t max_edge,
                        const TerrainDev *terrains, const GradLut *lut, const MeshTables *tables,
                        FusedCtl ctl, MeshOut out, const CullJob &cull, int32_t grid,
                        hipStream_t s);
// Pipelined form (edges up to 32): fill and mesh tasks from two ticket
// counters; one workgroup in `ratio` (2..kPipeRatioMax, 0 = kPipeRatio)
// meshes from the start, the others fill and then mesh; mesh m is served
// once fills up to m + lag are out (lag >= the farthest in-batch neighbour
// index minus the chunk's own).  Needs ctl.filled and ctl.mesh_ticket.
constexpr int kPipeRatio = 3;
constexpr int kPipeRatioMax = 8;
hipError_t launch_pipe(const FusedWork *work, int32_t n, int32_t max_edge, int32_t lag,
                       const TerrainDev *terrains, const GradLut *lut, const MeshTables *tables,
                       FusedCtl ctl, MeshOut out, const CullJob &cull, int32_t grid, int32_t ratio,
                       hipStream_t s);
hipError_t launch_cull(const CullJob &job, hipStream_t s);
hipError_t launch_set_planes(const Planes &planes, float *dst, hipStream_t s);
hipError_t launch_copy(void *dst, const void *src, uint64_t bytes, hipStream_t s);
hipError_t launch_frustum(const Planes &planes, const int32_t *coords, int32_t n, int32_t edge,
                          uint8_t *mask, hipStream_t s);
// Draw lists of up to kDrawOne meshes can take one launch; `state` holds
// kDrawStateWords words that no other launch uses at the same time, zero before
// the first use; `tag` is a number (1 to 2^48 - 1) that no earlier launch on them had.
constexpr int32_t kDrawOne = 65536;
constexpr int32_t kDrawStateWords = kDrawOne / 512;
hipError_t launch_draw_one(const Planes &planes, const int32_t *coords, const uint32_t *faces,
                           const uint64_t *first, int32_t n, int32_t edge, uint32_t mode,
                           uint64_t *state, uint64_t tag, DrawArgs *args, uint32_t *count,
                           hipStream_t s);
// Workgroups (and block_counts entries) a draw list of n meshes uses.
int32_t draw_blocks(int32_t n);
// The draw-list scratch array of the allocation-free entry point: device
// address of `device`'s copy (looked up once per device, with that device
// current at the first call), and the most meshes it serves.
constexpr int kMaxDevices = 64;
hipError_t draw_scratch_address(int device, uint32_t **ptr);
int32_t draw_scratch_max_meshes();
// Zeroes n <= 64 words with a kernel (capturable; no memset node).
hipError_t launch_clear_words(uint32_t *p, int32_t n, hipStream_t s);
hipError_t launch_draw_list(const Planes &planes, const int32_t *coords, const uint32_t *faces,
                            const uint64_t *first, int32_t n, int32_t edge, uint32_t mode,
                            uint32_t *block_counts, DrawArgs *args, uint32_t *count, hipStream_t s);

}  // namespace vx
