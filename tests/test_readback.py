"""Reading pictures back into the caller's memory: ordinary memory, memory pinned by the caller, and
planes of either kind in one call."""
import ctypes
import os
import statistics
import subprocess
import time

import numpy as np
import pytest

from h264_video_decoder_demo_amd import Engine, Generator
from h264_video_decoder_demo_amd import build as hbuild
from h264_video_decoder_demo_amd._lib import LIB_PATH, check, lib

from helpers import oracle_decode


class _Buffers:
    """Y, Cb, Cr of n MBs in memory of the process, or (where `pinned`) from hipHostMalloc."""

    def __init__(self, n, pinned):
        self.hip = ctypes.CDLL(LIB_PATH)  # (finds the symbols of the HIP runtime it is linked to)
        self.own, self.planes = [], []
        for k, p in zip((256, 64, 64), pinned):
            if p:
                ptr = ctypes.c_void_p()
                assert self.hip.hipHostMalloc(ctypes.byref(ptr), ctypes.c_size_t(k * n), ctypes.c_uint(0)) == 0
                self.own.append(ptr)
                self.planes.append(np.ctypeslib.as_array(ctypes.cast(ptr, ctypes.POINTER(ctypes.c_uint8)), (k * n,)))
            else:
                self.planes.append(np.empty(k * n, np.uint8))
            self.planes[-1][:] = 0x5A

    def __enter__(self):
        return self.planes

    def __exit__(self, *exc):
        for ptr in self.own:
            assert self.hip.hipHostFree(ptr) == 0


def _read(eng, sid, slot, bufs):
    check(lib().h264g_slot_readback(eng._h, sid, slot, *[ctypes.c_void_p(b.ctypes.data) for b in bufs]))


@pytest.mark.gpu
@pytest.mark.parametrize("pinned", [(0, 0, 0), (1, 1, 1), (1, 0, 0), (0, 1, 0), (0, 0, 1), (1, 0, 1)])
@pytest.mark.parametrize("size", [(1, 1), (22, 18), (120, 100), (161, 140)])
def test_readback_into_pinned_and_ordinary_memory(size, pinned):
    """Up to one half of the bounce buffer (4 MiB), more than one, more than two."""
    with Engine(device=0) as eng:
        gen = Generator(2, width_mbs=size[0], height_mbs=size[1], n_frames=1, seed=0x4EAD)
        sid = eng.open_stream_for(gen)
        (i, desc, want), = oracle_decode(gen)
        p = eng.begin(sid, *gen.picture(i))
        eng.submit(p)
        with _Buffers(size[0] * size[1], pinned) as bufs:
            _read(eng, sid, desc.dst_slot, bufs)
            for got, ref, plane in zip(bufs, want[2], "YUV"):
                assert np.array_equal(got, ref.reshape(-1)), plane
        eng.release(p)
        eng.close_stream(sid)


@pytest.mark.gpu
def test_pinned_memory_is_written_without_a_second_copy():
    """A 3840x2160 picture into pinned memory takes the transfer's time, about half of what it takes
    through the bounce buffer and a copy."""
    with Engine(device=0) as eng:
        sid = eng.open_stream(240, 135, 2)
        took = []
        for pinned in (0, 1):
            t = []
            with _Buffers(240 * 135, (pinned,) * 3) as bufs:
                for _ in range(20):
                    a = time.perf_counter()
                    _read(eng, sid, 0, bufs)
                    t.append(time.perf_counter() - a)
            took.append(statistics.median(t))
        print(f"ordinary {took[0] * 1e6:.0f} us, pinned {took[1] * 1e6:.0f} us", flush=True)
        assert took[1] < 0.75 * took[0]


def test_no_transfer_outlives_a_failed_readback(tmp_path):
    """Every split into planes and parts with every call failing in turn, and none: the bytes are
    right, and an error leaves no transfer into the buffer or the caller's memory under way."""
    exe = str(tmp_path / "readback_check")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-I", hbuild.CSRC, os.path.join(os.path.dirname(__file__), "readback_check.cpp"),
                    "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert (r.returncode, r.stdout) == (0, "ok\n"), r.stdout
