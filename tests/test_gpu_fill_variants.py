"""The fast density fill against the oracle, byte for byte, at the edges of its
rule: every compiled variant and the general kernels, each edge alone (the
one-chunk kernel, eight workgroups) and mixed in a batch of 64^3 chunks (the
64 kernel), cell boundaries inside and at the chunk's faces, tables that need
several row segments, voxels that lie exactly on their threshold."""
import dataclasses

import numpy as np
import pytest

import voxel_amd as V

pytestmark = pytest.mark.gpu


def dens(**kw):
    return V.Terrain(kind=V.TERRAIN_DENSITY, **{**dict(seed=7, octaves=4, frequency=1 / 64, lacunarity=2.0,
                                                       gain=0.5, y_scale=1 / 128), **kw})


REF = V.Terrain(kind=V.TERRAIN_REFERENCE, seed=1, octaves=3, frequency=0.09, lacunarity=0.5, gain=2.5)
CASES = {
    "one octave at the frequency limit": dens(octaves=1, frequency=0.75),
    "one octave past the limit": dens(octaves=1, frequency=0.8),
    "two octaves, odd ratio": dens(octaves=2, frequency=0.21, lacunarity=1.9, gain=0.7),
    "reference rule": REF,
    "reference rule, five octaves": dataclasses.replace(REF, octaves=5, frequency=1 / 40, lacunarity=2.0, gain=0.5),
    "four octaves": dens(),
    "four fine octaves": dens(frequency=0.04),
    "six octaves": dens(octaves=6, frequency=0.01),
    "seven octaves, slow": dens(octaves=7, frequency=1 / 300, lacunarity=1.8),
    "eight octaves past the limit": dens(octaves=8, frequency=1 / 64),
    "threshold zero": dens(octaves=3, frequency=1 / 16, y_scale=0.0),
    "negative gain, falling frequency": dens(frequency=0.2, lacunarity=0.5, gain=-1.5),
    "heightmap": V.Terrain(kind=V.TERRAIN_HEIGHTMAP, seed=5, octaves=5, frequency=0.07, height_scale=40.0,
                           height_max=70),
}
# the origin, negative coordinates, and on both sides of |coordinate * f| = 2^22
COORDS = [(0, 0, 0), (-3, -1, 7), (2 ** 20 - 2, 0, -5), (2 ** 21, 1, -2 ** 20)]


def oracle_terrain(O, t):
    return O.terrain(kind=t.kind, seed=t.seed, octaves=t.octaves, frequency=t.frequency,
                     lacunarity=t.lacunarity, gain=t.gain, height_scale=t.height_scale,
                     height_max=t.height_max, y_scale=t.y_scale)


def planes(ids, n):
    """x=0, x=N-1 as [y, z] and z=0, z=N-1 as [y, x]."""
    a = ids.reshape(n, n, n) != 0
    return a[:, :, 0], a[:, :, -1], a[:, 0, :], a[:, -1, :]


@pytest.mark.parametrize("name", CASES)
def test_fill_variants(ctx, oracle_mod, name):
    t = CASES[name]
    ot = oracle_terrain(oracle_mod, t)
    print("[case]", name, flush=True)
    ids = {}
    for edge in (16, 32, 64):
        for coord in COORDS if edge == 32 else COORDS[:2]:
            ref = ids[edge, coord] = oracle_mod.chunk_fill(ot, *coord, edge)
            ch = V.Chunk.new(ctx, t, coord, edge)
            assert (ch.ids() == ref).all(), (edge, coord)
            assert (ch.occupancy() == oracle_mod.occupancy(ref, edge)).all(), (edge, coord)
    keys = list(ids)
    for splits in ((0, 0), (8, 1)):
        b = V.Batch(ctx, [c for _, c in keys], [e for e, _ in keys], ctx.terrain(t))
        b.set_splits(*splits)
        b.run()
        b.wait()
        for i, k in enumerate(keys):
            assert (b.ids(i) == ids[k]).all(), (k, splits)
        # each chunk as the neighbour of an all-solid one: the faces that its
        # boundary planes leave are the voxels it has none at
        for i, (edge, _) in enumerate(keys[:4]):
            ch = b.chunk(i)
            solid = V.Chunk.from_ids(ctx, (0, 0, 0), edge, np.ones(edge ** 3, np.uint8))
            for side, facing in enumerate((1, 0, 3, 2)):
                adj = [None] * 4
                adj[side] = ch
                hidden = int(planes(ids[keys[i]], edge)[facing].sum())
                assert solid.create_mesh(adj).faces == 6 * edge * edge - hidden, (i, side)
            solid.release()
            ch.release()
        b.close()


@pytest.mark.parametrize("edge", [16, 32])
def test_whole_chunks(ctx, oracle_mod, edge):
    """1,024 chunks and more: one workgroup per chunk, counting in the fill."""
    t = dens(octaves=3, frequency=1 / 24)
    ot = oracle_terrain(oracle_mod, t)
    coords = [(x - 16, 0, z) for x in range(33) for z in range(32)]
    b = V.Batch(ctx, coords, edge, ctx.terrain(t))
    b.run()
    b.wait()
    for i in range(0, len(coords), 37):
        ref = oracle_mod.chunk_fill(ot, *coords[i], edge)
        assert (b.ids(i) == ref).all(), i
        faces = oracle_mod.mesh_buffers(ref, edge, (0, 0, 0), [None] * 4)[0]
        assert b.chunk_faces(i)[1] == len(faces), i
    b.close()


@pytest.mark.parametrize("n", [127, 130, 1030])
@pytest.mark.parametrize("kind", ["four octaves", "six octaves", "reference rule", "heightmap"])
def test_tiles_beside_64(ctx, oracle_mod, kind, n):
    """Batches with 64^3 chunks on both sides of their tiles' rule (16, 8 and
    4 workgroups a chunk), smaller chunks among them."""
    t = CASES[kind]
    ot = oracle_terrain(oracle_mod, t)
    edges = [64 if i % 8 == 3 else (32, 16)[i % 2] for i in range(n)]
    coords = [(i % 13 - 6, 0, i // 13) for i in range(n)]
    b = V.Batch(ctx, coords, edges, ctx.terrain(t))
    b.run()
    b.wait()
    for i in [0, 1, 2, 3, n // 2, n - 2, n - 1] + [k for k in range(3, n, 8)][-2:]:
        ref = oracle_mod.chunk_fill(ot, *coords[i], edges[i])
        assert (b.ids(i) == ref).all(), i
        ch = b.chunk(i)
        assert (ch.occupancy() == oracle_mod.occupancy(ref, edges[i])).all(), i
        ch.release()
        assert b.chunk_faces(i)[1] == len(oracle_mod.mesh_buffers(ref, edges[i], (0, 0, 0), [None] * 4)[0]), i
    b.close()


@pytest.mark.parametrize("n", [383, 384])
@pytest.mark.parametrize("name", ["16^3", "beside larger"])
def test_batch_rule(ctx, oracle_mod, name, n):
    """Batches on both sides of the rule that sends chunks to the general
    kernels: 16^3 chunks by their number, in larger batches each terrain by its
    finest octave, both kernels on one batch."""
    ts = [dens(octaves=3, frequency=1 / 60), dens(octaves=3, frequency=1 / 6), dens(octaves=1, frequency=0.25, y_scale=0.0),
          dens(octaves=6, frequency=1 / 80)]
    ots = [oracle_terrain(oracle_mod, t) for t in ts]
    edges = [16 if name == "16^3" else (16, 32)[i % 2] for i in range(n)]
    coords = [(i % 23 - 11, 0, i // 23) for i in range(n)]
    b = V.Batch(ctx, coords, edges, [ctx.terrain(ts[i % 4]) for i in range(n)])
    for splits in ((0, 0), (2, 1), (2, 1), (2, 1)):  # launched, captured, replayed twice
        b.set_splits(*splits)
        b.run()
        b.wait()
        for i in list(range(8)) + [n // 2, n // 2 + 1, n - 2, n - 1]:
            ref = oracle_mod.chunk_fill(ots[i % 4], *coords[i], edges[i])
            assert (b.ids(i) == ref).all(), (i, splits)
            assert b.chunk_faces(i)[1] == len(oracle_mod.mesh_buffers(ref, edges[i], (0, 0, 0), [None] * 4)[0]), i
    b.close()
