"""VX_CHECK_SCHEDULES=1 (read once per process) passes whatever forms a batch
has run in: the emission order in memory is the last scan's, which the forms
without a scan (the persistent ones, the staged one of small batches) leave."""
import os
import subprocess
import sys
import textwrap

import pytest

import voxel_amd as V

pytestmark = pytest.mark.gpu

SCRIPT = textwrap.dedent("""
    import sys
    sys.path.insert(0, {pkg!r})
    import voxel_amd as V
    nx, nz = int(sys.argv[1]), int(sys.argv[2])
    ctx = V.Context(0)
    t = V.Terrain(kind=V.TERRAIN_DENSITY, seed=7, octaves=4, frequency=1 / 64, lacunarity=2.0,
                  gain=0.5, y_scale=1 / 128)
    b = V.Batch(ctx, [(x, 0, z) for x in range(nx) for z in range(nz)], 16, ctx.terrain(t),
                V.grid_neighbours(nx, nz), formats=V.FMT_INSTANCES, face_capacity=64)
    want = None
    for step in ("SPLIT", "wait", "STAGED", "FUSED", "SPLIT", "PIPELINED", "SPLIT", "chunks", "SPLIT", "STAGED",
                 "tune", "SPLIT", "AUTO"):
        print("[case]", step, flush=True)
        if step == "chunks":
            b.run_per_chunk()
        elif step == "tune":
            b.autotune(2)
        elif step != "wait":
            b.set_mode(getattr(V, "BATCH_" + step))
            b.run()
        got = b.wait()
        want = want or got
        assert got == want, (step, got, want)
        for _ in range(2):  # captured, replayed
            b.run()
            assert b.wait() == want, step
    b.close()
    ctx.close()
""").format(pkg=os.path.dirname(os.path.abspath(V.__file__)))


@pytest.mark.parametrize("nx,nz", [(2, 1), (5, 7), (16, 32), (19, 27)])
def test_forms_in_turn(nx, nz):
    print("[case] schedule check over forms", nx, nz, flush=True)
    r = subprocess.run([sys.executable, "-c", SCRIPT, str(nx), str(nz)], capture_output=True, text=True,
                       timeout=100, env=dict(os.environ, VX_CHECK_SCHEDULES="1"))
    assert r.returncode == 0, r.stdout[-500:] + r.stderr[-2000:]
