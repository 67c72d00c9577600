"""The band heights that are run: reported by the context, switched on open streams, and each
measured once by the autotuner, whatever is configured above them."""
import numpy as np
import pytest

from h264_video_decoder_demo_amd import Engine, Generator, _lib
from h264_video_decoder_demo_amd import autotune as at

from helpers import oracle_decode
from test_bands import _FakeEngine, _Gen


@pytest.mark.gpu
def test_run_heights_switch_on_open_streams():
    """Every change of the run heights, with batches of several streams in between: the oracle's
    bytes; a batch built for other heights is refused."""
    gens = [Generator(2, width_mbs=w, height_mbs=h, n_frames=6, seed=0x4E16 + h, intra_in_inter_permille=200, qp_lo=26, qp_hi=51)
            for w, h in [(9, 13), (22, 18), (5, 4), (3, 1)]]
    heights = [(1, 1), (2, 3), (3, 2), (4, 4), (1, 4), (24, 8)]
    with Engine(device=0, deblock_waves=1, intra_waves=1) as eng:
        sids = [eng.open_stream_for(g) for g in gens]
        stale = None
        for (d, i), wants in zip(heights, zip(*(oracle_decode(g) for g in gens))):
            assert eng.set_bands(d, i) == (min(d, 4), min(i, 4)) == eng.band_rows()
            if stale:
                with pytest.raises(_lib.H264GError) as e:
                    eng.batch_run(stale[0])
                assert e.value.code == _lib.H264G_E_STATE
                eng.batch_destroy(stale[0])
                for p in stale[1]:
                    eng.release(p)
            pics = [eng.begin(s, *g.picture(w[0])) for s, g, w in zip(sids, gens, wants)]
            batch = eng.batch_create(pics)
            eng.batch_run(batch)
            eng.sync()
            for s, (k, desc, want) in zip(sids, wants):
                for got, ref, plane in zip(eng.readback(s, desc.dst_slot), want[2], "YUV"):
                    assert np.array_equal(got, ref), (d, i, s, k, plane)
            stale = (batch, pics)


@pytest.mark.gpu
def test_heights_above_four_run_as_four():
    with Engine(device=0) as eng:
        assert eng.band_rows() == (4, 4)
    with Engine(device=0, deblock_waves=3, intra_waves=6) as eng:
        assert eng.band_rows() == (3, 4)
        assert eng.set_bands(16, 0) == (4, 4)


class _ClampingEngine(_FakeEngine):
    passes = 0

    def set_bands(self, d, i):
        super().set_bands(min(d, 4), min(i, 4))
        return self.cur

    def batch_create(self, pics):
        _ClampingEngine.passes += 1
        return self.cur


def test_autotuner_measures_each_run_height_once(monkeypatch, tmp_path):
    """Candidates that run alike share a measurement, and those below 4 rows are among them."""
    import h264_video_decoder_demo_amd.engine as engine_mod
    clock = _FakeEngine.clock = [0.0]
    _FakeEngine.cost = {(d, i): abs(d - 3) + abs(i - 2) * 0.5 + 1 for d in range(1, 5) for i in range(1, 5)}
    _ClampingEngine.passes = 0
    monkeypatch.setattr(engine_mod, "Engine", _ClampingEngine)
    monkeypatch.setattr(at, "_clock", lambda: clock[0])
    monkeypatch.setattr(at, "_device_id", lambda device: "gfx950|test device|256 CUs|2400000 kHz")
    monkeypatch.setenv("XDG_CACHE_HOME", str(tmp_path))
    r = at.autotune([_Gen(), _Gen()], n_frames=2, reps=2)
    assert (r["deblock_waves"], r["intra_waves"]) == (3, 2)
    run_d, run_i = {min(d, 4) for d in at.DEBLOCK_ROWS}, {min(i, 4) for i in at.INTRA_ROWS}
    assert len(run_d) > 1 and len(run_i) > 1
    assert _ClampingEngine.passes == 2 * (len(run_d) + len(run_i) - 1)  # (2 batches a pass)
