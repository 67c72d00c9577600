"""The DPB budget counts what a stream takes from the device: its slots and its progress sets, with
the strips of the band heights that are run (at most 4 rows, whatever is configured)."""
import re

import pytest

from h264_video_decoder_demo_amd import Engine, _lib

SETS = 4  # H264G_MAX_STREAM_PICS


def _up(n):
    return (n + 255) // 256 * 256


def _bytes(w, h, slots, mbaff, rows):
    """What h264g_stream_open requests for one stream."""
    slot = w * h * 384 + (_up(w * 8) if mbaff else 0)
    deblock, intra = (-(-h // min(r or 8, 4)) for r in rows)
    words = _up(_up(w * h * 4) + h * 8)  # per MB, per row
    return slots * slot + SETS * _up(words + deblock * w * 256 + intra * w * 64)


def _charged(eng, w, h, slots, mbaff):
    """(bytes used, bytes that one more stream counts) from the refusal, None if it was opened."""
    try:
        eng.open_stream(w, h, slots, mbaff)
    except _lib.H264GError as e:
        assert e.code == _lib.H264G_E_BUDGET
        return tuple(int(v) for v in re.search(r"DPB budget: (\d+) \+ (\d+) >", str(e)).groups())


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [(0, 0), (1, 1), (3, 2), (4, 4), (12, 6), (24, 8)])
@pytest.mark.parametrize("w,h,slots,mbaff", [(22, 18, 5, False), (120, 68, 5, False), (240, 135, 2, False), (45, 30, 3, True)])
def test_a_stream_counts_what_it_takes(w, h, slots, mbaff, rows):
    n = _bytes(w, h, slots, mbaff, rows)
    kw = dict(device=0, deblock_waves=rows[0], intra_waves=rows[1])
    with Engine(dpb_budget_bytes=n - 1, **kw) as eng:
        assert _charged(eng, w, h, slots, mbaff) == (0, n)
    with Engine(dpb_budget_bytes=2 * n, **kw) as eng:
        assert _charged(eng, w, h, slots, mbaff) is None
        assert _charged(eng, w, h, slots, mbaff) is None
        assert _charged(eng, w, h, slots, mbaff) == (2 * n, n)
        eng.close_stream(0)
        assert _charged(eng, w, h, slots, mbaff) is None
