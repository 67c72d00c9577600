"""Staging a picture beside a running batch: h264g_picture_begin returns while the batch goes
on, whichever lane it runs on, and what was staged that way decodes to the same samples."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# A process of its own: which streams share a hardware queue depends on the streams that the
# process has created before.
PROGRAM = """
import sys
import numpy as np
from h264_video_decoder_demo_amd import Engine, Generator
with Engine(device=0, lane_split_mbs=int(sys.argv[1])) as eng:
    gens = [Generator(2, width_mbs=120, height_mbs=68, n_frames=1, seed=k + 1) for k in range(4)]
    sids = [eng.open_stream_for(g) for g in gens]
    pics = [eng.begin_raw(s, *g.picture_raw(0)) for s, g in zip(sids, gens)]
    batch = eng.batch_create(pics)
    small = Generator(2, width_mbs=22, height_mbs=18, n_frames=1, seed=9)
    sid = eng.open_stream_for(small)
    first = eng.begin_raw(sid, *small.picture_raw(0))
    eng.batch_run(batch)
    eng.submit(first)
    eng.sync()
    want = eng.readback(sid, first.desc.dst_slot)
    for rep in range(4):
        for _ in range(12):
            eng.batch_run(batch)
        half = eng.fence()
        for _ in range(12):
            eng.batch_run(batch)
        p = eng.begin_raw(sid, *small.picture_raw(0))
        running = not eng.done(half)
        print("batch still in its first half:", running, flush=True)
        eng.submit(p)
        eng.sync()
        eng.drop_fence(half)
        for g, w in zip(eng.readback(sid, p.desc.dst_slot), want):
            assert np.array_equal(g, w), rep
        eng.release(p)
        assert running, rep
    print("ok", flush=True)
"""


@pytest.mark.gpu
@pytest.mark.parametrize("split", [0, 100])
def test_begin_does_not_wait_for_a_running_batch(split):
    """The batch on lane 0 (no stream has 16384 MBs) and on lane 1 (all have 100)."""
    r = subprocess.run([sys.executable, "-u", "-c", PROGRAM, str(split)], cwd=ROOT, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and r.stdout.endswith("ok\n"), (r.stdout[-500:], r.stderr[-2000:])
