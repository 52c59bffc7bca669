"""Meshes of one chunk, whose faces are shared between workgroups in tiles of
at least 256: face counts on both sides of a tile, one face's worth of work,
none, and the worst case; block types found while the ids are read."""
import numpy as np
import pytest

import voxel_amd as V

pytestmark = pytest.mark.gpu


def isolated(edge, k):
    """k voxels without neighbours: 6 k faces."""
    ids = np.zeros((edge, edge, edge), np.uint8)
    at = [(y, z, x) for y in range(0, edge, 2) for z in range(0, edge, 2) for x in range(0, edge, 2)]
    for i in np.linspace(0, len(at) - 1, k).astype(int) if k else ():
        ids[at[i]] = V.GRASS if i % 3 else V.DIRT
    return ids.reshape(-1)


@pytest.mark.parametrize("edge", [16, 32, 64])
@pytest.mark.parametrize("voxels", [0, 1, 42, 43, 85, 86, 170, 171, 512])
def test_mesh_parts(ctx, oracle_mod, edge, voxels):
    print("[case]", edge, voxels, flush=True)
    ids = isolated(edge, voxels)
    ch = V.Chunk.from_ids(ctx, (1, 0, -1), edge, ids)
    assert (ch.ids() == ids).all()
    assert (ch.occupancy() == oracle_mod.occupancy(ids, edge)).all()
    mesh = ch.create_mesh()
    faces, inst, vert, idx = oracle_mod.mesh_buffers(ids, edge, (edge, 0, -edge), [None] * 4)
    assert mesh.faces == len(faces) == 6 * len(np.unique(np.nonzero(ids)[0]))
    got = mesh.instances()
    assert (got["m"].view(np.uint32) == inst["m"].view(np.uint32)).all()
    assert (got["tex"] == inst["tex"]).all()
    assert (mesh.vertices().view(np.uint32) == vert.view(np.uint32)).all()
    assert (mesh.indices() == idx).all()


@pytest.mark.parametrize("edge", [16, 32, 64])
def test_checkerboard_of_both_types(ctx, oracle_mod, edge):
    y, z, x = np.indices((edge,) * 3)
    ids = np.where((x + y + z) % 2, 1 + (x // 2 + y) % 2, 0).astype(np.uint8).reshape(-1)
    mesh = V.Chunk.from_ids(ctx, (0, 0, 0), edge, ids).create_mesh()
    faces, inst, _, _ = oracle_mod.mesh_buffers(ids, edge, (0, 0, 0), [None] * 4)
    assert mesh.faces == len(faces) == 3 * edge ** 3
    got = mesh.instances()
    assert (got["tex"] == inst["tex"]).all()
    assert (got["m"].view(np.uint32) == inst["m"].view(np.uint32)).all()


@pytest.mark.parametrize("bad", [3, 255])
def test_ids_out_of_range_are_refused(ctx, bad):
    for at in (0, 16 ** 3 - 1):
        ids = np.ones(16 ** 3, np.uint8)
        ids[at] = bad
        with pytest.raises(V.VoxelError) as e:
            V.Chunk.from_ids(ctx, (0, 0, 0), 16, ids)
        assert e.value.status == V.ERR_INVALID


@pytest.mark.parametrize("edge,n", [(16, 17), (16, 64), (16, 400), (16, 639), (16, 641), (16, 1281), (32, 700),
                                    (32, 1279), (32, 1281), (32, 1792), (64, 21), (64, 400)])
def test_batch_parts(ctx, oracle_mod, edge, n):
    """Batches on both sides of the rule for workgroups per emit item."""
    print("[case]", edge, n, flush=True)
    t = V.Terrain(kind=V.TERRAIN_HEIGHTMAP, seed=3, octaves=2, frequency=1 / 24, lacunarity=2.0, gain=0.5,
                  height_scale=14.0, height_max=15)
    ot = oracle_mod.terrain(kind=t.kind, seed=t.seed, octaves=t.octaves, frequency=t.frequency,
                            lacunarity=t.lacunarity, gain=t.gain, height_scale=t.height_scale,
                            height_max=t.height_max, y_scale=t.y_scale)
    coords = [(i % 31 - 15, 0, i // 31) for i in range(n)]
    b = V.Batch(ctx, coords, edge, ctx.terrain(t), None, formats=V.FMT_INSTANCES)
    b.run()
    b.wait()
    inst = b.mesh(V.FMT_INSTANCES)
    for i in [0, 1, 7, n // 2, n - 2, n - 1]:
        ids = oracle_mod.chunk_fill(ot, *coords[i], edge)
        faces, ei, _, _ = oracle_mod.mesh_buffers(ids, edge, tuple(v * edge for v in coords[i]), [None] * 4)
        first, cnt = b.chunk_faces(i)
        assert cnt == len(faces), i
        got = inst[first:first + cnt]
        assert (got["m"].view(np.uint32) == ei["m"].view(np.uint32)).all(), i
        assert (got["tex"] == ei["tex"]).all(), i
    b.close()


@pytest.mark.parametrize("formats", [V.FMT_VERTICES, V.FMT_INSTANCES, V.FMT_VERTICES | V.FMT_INSTANCES])
@pytest.mark.parametrize("n", [1279, 1280])
def test_batch_parts_by_faces(ctx, oracle_mod, n, formats):
    """Three workgroups an item, but one for an item of 8,192 faces and more
    that writes vertices: items on both sides of it, empty ones among them."""
    print("[case]", n, formats, flush=True)
    kw = dict(seed=7, lacunarity=2.0, gain=0.5)
    ts = [V.Terrain(kind=V.TERRAIN_REFERENCE, octaves=2, frequency=0.3, **kw),   # 28,000 faces
          V.Terrain(kind=V.TERRAIN_REFERENCE, octaves=3, frequency=0.057, **kw),  # about 8,000
          V.Terrain(kind=V.TERRAIN_DENSITY, octaves=4, frequency=1 / 64, y_scale=1 / 128, **kw),
          V.Terrain(kind=V.TERRAIN_AIR)]
    ots = [oracle_mod.terrain(kind=t.kind, seed=t.seed, octaves=t.octaves, frequency=t.frequency,
                              lacunarity=t.lacunarity, gain=t.gain, height_scale=t.height_scale,
                              height_max=t.height_max, y_scale=t.y_scale) for t in ts]
    pick = [(i // 32 if i % 32 == 5 else 3) % 4 for i in range(n)]
    coords = [(i % 31 - 15, 0, i // 31) for i in range(n)]
    b = V.Batch(ctx, coords, 32, [ctx.terrain(ts[k]) for k in pick], None, formats=formats)
    b.run()
    b.wait()
    inst = b.mesh(V.FMT_INSTANCES) if formats & V.FMT_INSTANCES else None
    vert, idx = (b.mesh(V.FMT_VERTICES), b.mesh(V.FMT_INDICES)) if formats & V.FMT_VERTICES else (None, None)
    counts = []
    for i in [k for k in range(n) if pick[k] != 3] + [0, n - 1]:
        ids = oracle_mod.chunk_fill(ots[pick[i]], *coords[i], 32)
        faces, ei, ev, ex = oracle_mod.mesh_buffers(ids, 32, tuple(v * 32 for v in coords[i]), [None] * 4)
        first, cnt = b.chunk_faces(i)
        assert cnt == len(faces), i
        counts.append(cnt)
        if inst is not None:
            got = inst[first:first + cnt]
            assert (got["m"].view(np.uint32) == ei["m"].view(np.uint32)).all(), i
            assert (got["tex"] == ei["tex"]).all(), i
        if vert is not None:
            assert (vert[4 * first:4 * (first + cnt)].view(np.uint32) == ev.view(np.uint32)).all(), i
            assert (idx[6 * first:6 * (first + cnt)] == ex).all(), i
    assert min(c for c in counts if c) < 8192 < max(counts)
    b.close()
