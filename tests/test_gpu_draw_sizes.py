"""Draw lists on both sides of every change of path: one launch up to 65,536
meshes, two passes of one mesh per thread up to 262,144, of four above; edges
of workgroups; nothing or everything visible; an offset past 32 bits; replays
of a captured call between eager ones.  Each against the host's own test of
every box."""
import ctypes as C

import numpy as np
import pytest

import camera
import voxel_amd as V

pytestmark = pytest.mark.gpu


def frustum(eye, d, far):
    return V.Frustum(camera.colmajor(camera.perspective(np.radians(70), 1.6, 0.1, far) @
                                     camera.look_at(eye, np.asarray(eye) + d)))


def expected(mask, faces, first, mode):
    i = np.nonzero(mask)[0]
    out = np.zeros(len(i), V.DRAW_DTYPE)
    if mode == V.DRAW_EXPANDED:
        out["index_count"], out["instance_count"] = 6 * faces[i], 1
        out["first_index"], out["base_vertex"] = 6 * first[i], 4 * first[i]
    else:
        out["index_count"], out["instance_count"], out["first_instance"] = 6, faces[i], first[i]
    return out


@pytest.mark.parametrize("n", [1, 511, 512, 513, 65535, 65536, 65537, 262144, 262145])
def test_draw_list_sizes(ctx, n):
    print("[case] draw list", n, flush=True)
    rng = np.random.default_rng(n)
    side = int(np.ceil(np.sqrt(n)))
    coords = np.stack(np.meshgrid(np.arange(side), [0], np.arange(side), indexing="ij"), -1).reshape(-1, 3)
    coords = np.ascontiguousarray(rng.permutation(coords)[:n], np.int32)
    faces = rng.integers(0, 900, n).astype(np.uint32)
    first = np.concatenate([[0], np.cumsum(faces[:-1], dtype=np.uint64)]).astype(np.uint64)
    mid = side * 16.0
    cams = [frustum((mid, 50.0, mid), (0.6, -0.2, 0.4), 600.0),         # some
            frustum((mid, 5000.0, mid), (0.0, 1.0, 0.001), 600.0),      # none: looks up from above
            frustum((mid, 1e6, mid), (0.0, -1.0, 0.001), 1e7)]          # all
    for f, least, most in zip(cams, (0, 0, n), (n, 0, n)):
        mask = f.mask(ctx, coords)
        assert least <= mask.sum() <= most
        for mode in (V.DRAW_INSTANCED, V.DRAW_EXPANDED):
            got = f.draw_list(ctx, coords, faces, first, mode=mode)
            assert (got == expected(mask, faces, first, mode)).all()
    # an offset past the draw's 32 bits is reported, and only by that call
    far = first.copy()
    far[-1] = 1 << 40
    with pytest.raises(V.VoxelError):
        cams[2].draw_list(ctx, coords, faces, far)
    assert len(cams[2].draw_list(ctx, coords, faces, first)) == n


def test_captured_draw_list(ctx):
    """vx_frustum_draw_list captured from the context's stream and replayed,
    with other boxes in the same buffer and eager calls between."""
    hip = C.CDLL("libamdhip64.so.7")
    s = V.P()
    ctx.check(ctx.L.vx_ctx_stream(ctx.h, C.byref(s)), "vx_ctx_stream")
    n, f = 4000, frustum((0.0, 40.0, 0.0), (0.5, -0.1, 0.7), 900.0)
    rng = np.random.default_rng(1)

    def boxes():
        return np.ascontiguousarray(rng.integers(-30, 30, (n, 3)) * [1, 0, 1], np.int32)
    faces = rng.integers(0, 900, n).astype(np.uint32)
    first = np.concatenate([[0], np.cumsum(faces[:-1], dtype=np.uint64)]).astype(np.uint64)
    a = boxes()
    f.draw_list(ctx, a, faces, first)  # the context's state exists
    bufs = [V.DeviceBuffer.of(ctx, v) for v in (a, faces, first)]
    args, cnt = V.DeviceBuffer(ctx, n * 20), V.DeviceBuffer(ctx, 8)
    graph, ex = V.P(), V.P()
    assert hip.hipStreamBeginCapture(s, 1) == 0
    st = ctx.L.vx_frustum_draw_list(ctx.h, C.byref(f.c), bufs[0].ptr, bufs[1].ptr, bufs[2].ptr, n, 32,
                                    V.DRAW_INSTANCED, args.ptr, cnt.ptr)
    assert hip.hipStreamEndCapture(s, C.byref(graph)) == 0 and st == V.OK
    assert hip.hipGraphInstantiate(C.byref(ex), graph, None, None, C.c_size_t(0)) == 0
    try:
        for _ in range(5):
            a = boxes()
            bufs[0].upload(a)
            assert hip.hipGraphLaunch(ex, s) == 0
            ctx.synchronize()
            want = expected(f.mask(ctx, a), faces, first, V.DRAW_INSTANCED)
            assert cnt.download(np.uint32, 2).tolist() == [len(want), 0]
            got = args.download(np.uint8, len(want) * 20).view(V.DRAW_DTYPE)
            assert (got == want).all()
            assert (f.draw_list(ctx, a, faces, first) == want).all()  # eager, same state
    finally:
        hip.hipGraphExecDestroy(ex)
        hip.hipGraphDestroy(graph)
        for b in bufs + [args, cnt]:
            b.free()


def test_captured_draw_list_beside_eager_ones(ctx):
    """Replays of a captured list on another stream, eager lists of other
    lengths meanwhile: both stay right, and so do later ones."""
    hip = C.CDLL("libamdhip64.so.7")
    s, s2 = V.P(), V.P()
    ctx.check(ctx.L.vx_ctx_stream(ctx.h, C.byref(s)), "vx_ctx_stream")
    assert hip.hipStreamCreateWithFlags(C.byref(s2), 1) == 0  # non-blocking
    n, f = 65536, frustum((0.0, 40.0, 0.0), (0.5, -0.1, 0.7), 900.0)
    rng = np.random.default_rng(3)
    coords = np.ascontiguousarray(rng.integers(-30, 30, (n, 3)) * [1, 0, 1], np.int32)
    faces = rng.integers(0, 900, n).astype(np.uint32)
    first = np.concatenate([[0], np.cumsum(faces[:-1], dtype=np.uint64)]).astype(np.uint64)
    mask = f.mask(ctx, coords)
    want = expected(mask, faces, first, V.DRAW_INSTANCED)
    bufs = [V.DeviceBuffer.of(ctx, v) for v in (coords, faces, first)]
    args, cnt = V.DeviceBuffer(ctx, n * 20), V.DeviceBuffer(ctx, 8)
    graph, ex = V.P(), V.P()
    assert hip.hipStreamBeginCapture(s, 1) == 0
    st = ctx.L.vx_frustum_draw_list(ctx.h, C.byref(f.c), bufs[0].ptr, bufs[1].ptr, bufs[2].ptr, n, 32,
                                    V.DRAW_INSTANCED, args.ptr, cnt.ptr)
    assert hip.hipStreamEndCapture(s, C.byref(graph)) == 0 and st == V.OK
    assert hip.hipGraphInstantiate(C.byref(ex), graph, None, None, C.c_size_t(0)) == 0
    try:
        for k, m in enumerate((65536, 512, 30000, 65536, 1, 65000, 4096, 65536)):
            print("[case] replay beside a list of", m, flush=True)
            for _ in range(3):
                assert hip.hipGraphLaunch(ex, s2) == 0
            got = f.draw_list(ctx, coords[:m], faces[:m], first[:m])
            assert hip.hipStreamSynchronize(s2) == 0
            assert (got == expected(mask[:m], faces[:m], first[:m], V.DRAW_INSTANCED)).all()
            assert cnt.download(np.uint32, 2).tolist() == [len(want), 0]
            assert (args.download(np.uint8, len(want) * 20).view(V.DRAW_DTYPE) == want).all()
    finally:
        hip.hipGraphExecDestroy(ex)
        hip.hipGraphDestroy(graph)
        hip.hipStreamDestroy(s2)
        for b in bufs + [args, cnt]:
            b.free()
