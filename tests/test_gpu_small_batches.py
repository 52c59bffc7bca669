"""Batches on both sides of 512 chunks, up to which the emit takes its bases
from the counts itself: bases, total, whole mesh, a frustum job beside the
count (its workgroups follow the chunks'), an arena that has to grow, and
replays of the captured graph with a moved camera."""
import numpy as np
import pytest

import camera
import voxel_amd as V

pytestmark = pytest.mark.gpu

T = V.Terrain(kind=V.TERRAIN_DENSITY, seed=3, octaves=2, frequency=1 / 20, y_scale=1 / 64)


def frustum(eye, d):
    return V.Frustum(camera.colmajor(camera.perspective(np.radians(70), 1.6, 0.1, 512) @
                                     camera.look_at(eye, np.asarray(eye) + d)))


@pytest.mark.parametrize("edges", ["16", "mixed"])
@pytest.mark.parametrize("n", [1, 2, 65, 511, 512, 513])
def test_small_batches(ctx, oracle_mod, n, edges):
    O = oracle_mod
    print("[case]", n, edges, flush=True)
    if edges == "mixed" and n > 65:
        n = 40 + n % 3  # mixed edges: emit items, all kinds of chunk
    ot = O.terrain(kind=T.kind, seed=T.seed, octaves=T.octaves, frequency=T.frequency,
                   lacunarity=T.lacunarity, gain=T.gain, y_scale=T.y_scale)
    es = [16 if edges == "16" else (64, 16, 32, 16)[i % 4] for i in range(n)]
    coords = [(i % 23 - 11, 0, i // 23) for i in range(n)]
    tids = [ctx.terrain(T if i % 5 else V.Terrain(kind=V.TERRAIN_AIR)) for i in range(n)]
    boxes = np.array([(x, 0, z) for x in range(-20, 20) for z in range(-20, 20)][:n + 777], np.int32)
    cbuf, mbuf = V.DeviceBuffer.of(ctx, boxes), V.DeviceBuffer(ctx, len(boxes))
    b = V.Batch(ctx, coords, es, tids, None, formats=V.FMT_VERTICES | V.FMT_INSTANCES, face_capacity=100)
    expect, run = [], 0
    for c, e, i in zip(coords, es, range(n)):
        ids = O.chunk_fill(ot, *c, e) if i % 5 else np.zeros(e ** 3, np.uint8)
        expect.append(O.mesh_buffers(ids, e, tuple(v * e for v in c), [None] * 4))
    total = sum(len(x[0]) for x in expect)
    for rep in range(4):  # launched, captured, replayed
        f = frustum((10.0 * rep, 20.0, -30.0), (0.5, -0.1, 0.2 + rep))
        mbuf.upload(np.full(len(boxes), 7, np.uint8))
        b.set_cull(f, cbuf, len(boxes), 16, mbuf)
        b.run()
        assert b.wait() == total
        assert (mbuf.download(np.uint8, len(boxes)) == f.mask(ctx, boxes, 16)).all(), rep
    verts, idx, inst = b.mesh(V.FMT_VERTICES), b.mesh(V.FMT_INDICES), b.mesh(V.FMT_INSTANCES)
    for i, (faces, ei, ev, ex) in enumerate(expect):
        first, cnt = b.chunk_faces(i)
        assert (first, cnt) == (run, len(faces)), i
        s = slice(first, first + cnt)
        assert (verts[4 * first:4 * (first + cnt)].view(np.uint32) == ev.view(np.uint32)).all(), i
        assert (idx[6 * first:6 * (first + cnt)] == ex).all(), i
        assert (inst[s]["m"].view(np.uint32) == ei["m"].view(np.uint32)).all(), i
        run += cnt
    b.close()
    cbuf.free()
    mbuf.free()
