"""Face counts against the oracle on both sides of the count's rule: a
workgroup per chunk and a wave per chunk, each edge alone and mixed, batches
that do not fill the last workgroup, any subset of the four neighbours."""
import numpy as np
import pytest

import voxel_amd as V

pytestmark = pytest.mark.gpu

SIZES = {"16, workgroups": ([16], 37), "16, fewest waves": ([16], 514), "16, waves": ([16], 2049),
         "32, workgroups": ([32], 37),
         "32, waves": ([32], 2050), "32 and 16, waves": ([32, 16], 2051), "64": ([64], 9),
         "64, 32 and 16": ([64, 32, 16], 30)}


@pytest.mark.parametrize("name", SIZES)
def test_counts(ctx, oracle_mod, name):
    edges, n = SIZES[name]
    print("[case]", name, flush=True)
    t = V.Terrain(kind=V.TERRAIN_DENSITY, seed=11, octaves=2, frequency=0.3, lacunarity=2.0, gain=0.6,
                  y_scale=0.0)
    ot = oracle_mod.terrain(kind=t.kind, seed=t.seed, octaves=t.octaves, frequency=t.frequency,
                            lacunarity=t.lacunarity, gain=t.gain, height_scale=t.height_scale,
                            height_max=t.height_max, y_scale=t.y_scale)
    rng = np.random.default_rng(5)
    k = len(edges)
    e = [edges[i % k] for i in range(n)]
    coords = [(int(x), int(y), int(z)) for x, y, z in rng.integers(-40, 40, (n, 3))]
    # any other chunk of the same edge, or none, at each side
    nb = rng.integers(0, n // k, (n, 4)) * k + np.arange(n)[:, None] % k
    nb = np.where((rng.random((n, 4)) < 0.4) | (nb == np.arange(n)[:, None]), -1, nb).astype(np.int32)
    b = V.Batch(ctx, coords, e, ctx.terrain(t), neighbours=nb)
    b.run()
    b.wait()
    for i in list(range(8)) + list(range(n - 8, n)) + [int(v) for v in rng.integers(0, n, 12)]:
        ids = [oracle_mod.chunk_fill(ot, *coords[j], e[j]) if j >= 0 else None for j in (i, *nb[i])]
        faces = oracle_mod.mesh_buffers(ids[0], e[i], (0, 0, 0), ids[1:])[0]
        assert b.chunk_faces(i)[1] == len(faces), i
    b.close()


@pytest.mark.parametrize("edge", [16, 32, 64])
@pytest.mark.parametrize("density", [0.0, 0.02, 0.5, 1.0])
def test_count_of_ids(ctx, oracle_mod, edge, density):
    rng = np.random.default_rng(edge)
    ids = [(rng.random(edge ** 3) < density).astype(np.uint8)]
    ids += [(rng.random(edge ** 3) < 0.5).astype(np.uint8) for _ in range(4)]
    ch = [V.Chunk.from_ids(ctx, (0, 0, 0), edge, v) for v in ids]
    for sides in (0, 1, 2, 4, 8, 15):
        adj = [k if sides >> k & 1 else None for k in range(4)]
        faces = oracle_mod.mesh_buffers(ids[0], edge, (0, 0, 0),
                                        [None if k is None else ids[1 + k] for k in adj])[0]
        m = ch[0].create_mesh([None if k is None else ch[1 + k] for k in adj])
        assert m.faces == len(faces), sides
    for c in ch:
        c.release()
