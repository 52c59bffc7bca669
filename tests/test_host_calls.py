"""What the library's host code queues, and in which order, without a GPU: its
HIP calls bind to tests/host_calls/hip_calls.cpp, which logs them.  Each
scenario runs in a process of its own."""
import os
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
STUB = os.path.join(ROOT, "tests", "host_calls", "hip_calls.cpp")

PRELUDE = r"""
import ctypes as C, sys
hip = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
hip.calls_log.restype = C.c_char_p
sys.path.insert(0, sys.argv[2])
import numpy as np
import voxel_amd as V
ctx = V.Context(0)
stream = V.P()
ctx.check(ctx.L.vx_ctx_stream(ctx.h, C.byref(stream)), "vx_ctx_stream")
def calls():
    "The calls since the last look."
    out = hip.calls_log().decode().split("\n")[:-1]
    hip.calls_clear()
    return out
def terrain(**k):
    return V.Terrain(**dict(dict(kind=V.TERRAIN_DENSITY, seed=7, octaves=4, frequency=1 / 64,
                                 lacunarity=2.0, gain=0.5, y_scale=1 / 128), **k))
def batch(n, edge=32, t=None, **k):
    return V.Batch(ctx, [(i, 0, 0) for i in range(n)], edge, ctx.terrain(t or terrain()), **k)
calls()
"""


@pytest.fixture(scope="module")
def scenario(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    so = tmp_path_factory.mktemp("calls") / "hip_calls.so"
    subprocess.run([cxx, "-std=c++17", "-O1", "-shared", "-fPIC", STUB, "-o", str(so)], check=True)

    def run(code, **env):
        p = subprocess.run([sys.executable, "-c", PRELUDE + code, str(so),
                            os.path.join(ROOT, "wgpu-voxel-engine_amd")],
                           capture_output=True, text=True, timeout=120, env=dict(os.environ, **env))
        assert p.returncode == 0, p.stdout + p.stderr
    return run


DRAW = r"""
frustum = V.Frustum(np.eye(4, dtype=np.float32).ravel())
def draw(n):
    return ctx.L.vx_frustum_draw_list(ctx.h, C.byref(frustum.c), bufs[0].ptr, bufs[1].ptr, bufs[2].ptr,
                                      n, 32, V.DRAW_INSTANCED, bufs[3].ptr, bufs[4].ptr)
bufs = [V.DeviceBuffer(ctx, b) for b in (100000 * 12, 100000 * 4, 100000 * 8, 100000 * 20, 8)]
calls()
"""


@pytest.mark.parametrize("mode", [1, 2])
@pytest.mark.parametrize("warm", [[], [100000]])
def test_captured_draw_list_records_kernels_only(scenario, mode, warm):
    """The first list of up to 65,536 meshes may be a captured one, after a
    longer list or none: nothing is allocated or cleared in its capture."""
    scenario(DRAW + f"""
for n in {warm}:
    assert draw(n) == V.OK
calls()
assert hip.hipStreamBeginCapture(stream, {mode}) == 0
assert draw(4000) == V.OK
got = [c for c in calls() if c != "hipStreamBeginCapture"]
assert got and all(c.startswith("captured:draw_") for c in got), got
""")


def test_captured_draw_list_keeps_no_state(scenario):
    """A list queued at once takes one launch, whose status words are that
    call's own; a captured one, whose replays would share them with later
    calls, the two passes that overwrite all they read."""
    scenario(DRAW + """
for _ in range(2):
    assert draw(4000) == V.OK
assert calls() == ["draw_one_kernel 8"] * 2
assert hip.hipStreamBeginCapture(stream, 1) == 0
assert draw(4000) == V.OK
graph = V.P()
assert hip.hipStreamEndCapture(stream, C.byref(graph)) == 0
assert calls() == ["hipStreamBeginCapture", "captured:draw_count_kernel 16", "captured:draw_write_kernel 16",
                   "hipStreamEndCapture"]
assert draw(4000) == V.OK
assert calls() == ["draw_one_kernel 8"]
""")


@pytest.mark.parametrize("mode", ["STAGED", "SPLIT"])
@pytest.mark.parametrize("call", ["hipStreamBeginCapture", "hipStreamEndCapture", "hipGraphInstantiate"])
def test_wait_outlives_a_failed_capture(scenario, mode, call):
    """A run that succeeded is waited for and its results are returned whether
    or not the graph of later runs can be captured; the next run tries again."""
    scenario(f"""
b = batch(4)
b.set_mode(V.BATCH_{mode})
b.run()
calls()
hip.calls_fail(b"{call}")
assert b.wait() == 0
assert "hipStreamSynchronize" in calls()
assert b.chunk_faces(3) == (0, 0)
b.run()
got = calls()
assert "hipGraphInstantiate" in got and got[-1] == "hipGraphLaunch", got
""")


def test_graphs_are_captured_on_a_private_stream(scenario):
    """A caller, or another thread, may queue work on the context's stream at
    any moment: no call captures that stream."""
    scenario("""
hip.calls_capture_stream.restype = C.c_void_p
for mode in (V.BATCH_STAGED, V.BATCH_SPLIT):
    b = batch(4)
    b.set_mode(mode)
    b.run()
    b.wait()
    assert hip.calls_capture_stream() not in (None, stream.value)
    got = [c for c in calls() if c.startswith("captured:")]
    assert any("emit_kernel" in c for c in got)
# and a run in the caller's own capture records work, with a graph or without
for runs in (0, 1, 2):
    b = batch(4)
    for _ in range(runs):
        b.run()
        b.wait()
    calls()
    assert hip.hipStreamBeginCapture(stream, 1) == 0
    b.run()
    graph = V.P()
    assert hip.hipStreamEndCapture(stream, C.byref(graph)) == 0
    got = calls()[1:-1]
    assert got and all(c.startswith("captured:") for c in got), (runs, got)
""")


@pytest.mark.parametrize("use", ["create_mesh", "neighbour", "ids", "occupancy"])
def test_chunk_of_another_context_is_waited_for(scenario, use):
    """A chunk made in one context and used through another: its pack or fill
    runs on the first one's stream, so the call waits for that first; within a
    context the stream orders them."""
    scenario(f"""
other = V.Context(0)
hip.calls_synced_stream.restype = C.c_void_p
chunk = V.Chunk.from_ids(ctx, (0, 0, 0), 32, np.ones(32 ** 3, np.uint8))
mine = V.Chunk.from_ids(other, (1, 0, 0), 32, np.ones(32 ** 3, np.uint8))
def use(c):
    if "{use}" == "create_mesh":
        c.create_mesh()
    elif "{use}" == "neighbour":
        mine.create_mesh((c, None, None, None))
    else:
        getattr(c, "{use}")()
seen = []
def sync_first(c):
    calls()
    hip.calls_fail(b"hipStreamSynchronize")  # ends the call at its first wait
    try:
        use(c)
        assert False
    except V.VoxelError:
        pass
    return calls()[0] == "hipStreamSynchronize" and hip.calls_synced_stream() == stream.value
foreign = V.Chunk(other, chunk.h)  # the same chunk through the other context
assert sync_first(foreign)
foreign.h = None
if "{use}" != "neighbour":
    assert not sync_first(chunk)
""")


def test_mixed_batch_fills_side_by_side(scenario):
    """A batch whose chunks take both fill kernels: the general ones on the
    second stream, with as many workgroups as a batch of them alone, joined
    before the count; a batch of one kind launches one fill."""
    scenario("""
fine = terrain(frequency=0.5, octaves=2)  # past the fast fill's frequencies
tids = [ctx.terrain(fine if i % 8 == 0 else terrain()) for i in range(512)]
b = V.Batch(ctx, [(i, 0, 0) for i in range(512)], 32, tids)
calls()
b.run()
got = calls()
at = [i for i, c in enumerate(got) if c == "hipStreamWaitEvent"]
names = [c.split()[0] for c in got if "_kernel" in c]
assert names[:3] == ["fill_split_kernel", "fill_fast_kernel", "count_kernel"], got
assert len(at) == 2 and at[1] < got.index("count_kernel 512"), got
assert "fill_split_kernel 2048" in got and "fill_fast_kernel 1024" in got, got
b.wait()
one = batch(64)
calls()
one.run()
got = calls()
assert [c.split()[0] for c in got if "fill" in c] == ["fill_fast_kernel"] and "hipStreamWaitEvent" not in got
""")


def test_autotuner_times_each_fill_shape_once(scenario):
    """64^3 chunks of the bounded fill: eight workgroups by the rule, four and
    not eight again among the candidates, and each launched as named."""
    scenario("""
b = batch(130, 64, face_capacity=64)
calls()
r = b.autotune(1)
fills = [c["splits"][0] for c in r["candidates"] if c["mode"] == "staged" and c["splits"][1] == 0]
assert fills == [0, 4], r
seen = {int(c.split()[1]) // 130 for c in calls() if c.startswith(("fill_fast", "captured:fill_fast"))}
assert seen == {4, 8}, seen
""")


def test_no_memory_for_a_form_is_an_error(scenario):
    """Host memory that a run needs for its form and cannot have is a status,
    not an exception through the C entry; the batch runs once there is some."""
    scenario("""
import resource
b = batch(20000, 16, face_capacity=64)
b.set_mode(V.BATCH_FUSED)
used = int(open("/proc/self/statm").read().split()[0]) * resource.getpagesize()
soft, hard = resource.getrlimit(resource.RLIMIT_AS)
resource.setrlimit(resource.RLIMIT_AS, (used + (1 << 20), hard))
try:
    b.run()
    status = V.OK
except V.VoxelError as e:
    status = e.status
resource.setrlimit(resource.RLIMIT_AS, (soft, hard))
assert status == -2, status  # VX_ERR_NOMEM
b.run()
""")
