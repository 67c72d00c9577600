"""The band schedules at the sizes where they can go wrong: pictures a few MBs wide or tall
(one MB, the register sets the deblocking rows are unrolled over, the strip rings' 8 slots
and one more, rows around the band heights, an odd second chroma row), every band height
that changes the cut, against the C oracle, byte for byte."""
import numpy as np
import pytest

from h264_video_decoder_demo_amd import Engine, Generator

from helpers import oracle_decode

SIZES = [(1, 1), (1, 9), (2, 4), (3, 5), (4, 8), (6, 3), (7, 7), (8, 2), (9, 6), (10, 13), (25, 5)]


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [(1, 1), (2, 3), (3, 8), (0, 0)])
def test_band_cuts_match_oracle(rows):
    """I, P and B pictures (4x4 and 8x8 transforms, strong and weak edges: QP 26..51)."""
    with Engine(device=0, deblock_waves=rows[0], intra_waves=rows[1]) as eng:
        for k, (w, h) in enumerate(SIZES):
            gen = Generator(2, width_mbs=w, height_mbs=h, n_frames=4, seed=0xBA9D00 + 16 * k, qp_lo=26, qp_hi=51,
                            intra_in_inter_permille=200, ipcm_permille=20)
            sid = eng.open_stream_for(gen)
            for i, desc, want in oracle_decode(gen):
                p = eng.begin(sid, *gen.picture(i))
                eng.submit(p)
                eng.sync()
                for got, ref, plane in zip(eng.readback(sid, desc.dst_slot), want[2], "YUV"):
                    assert np.array_equal(got, ref), (w, h, i, plane)
                eng.release(p)
            eng.close_stream(sid)


@pytest.mark.gpu
@pytest.mark.parametrize("permille", [4, 60, 700])
def test_sparse_and_dense_intra_rows_match_oracle(permille):
    """Intra MBs few and far between, and many, in P and B pictures wider than the intra rows'
    rings (64 columns): rows that wait far ahead of, or behind, the row above."""
    with Engine(device=0) as eng:
        for k, (w, h) in enumerate([(66, 9), (131, 6), (200, 3)]):
            gen = Generator(2, width_mbs=w, height_mbs=h, n_frames=3, b_frames=1, seed=0xBA9E00 + 16 * k,
                            intra_in_inter_permille=permille)
            sid = eng.open_stream_for(gen)
            for i, desc, want in oracle_decode(gen):
                p = eng.begin(sid, *gen.picture(i))
                eng.submit(p)
                eng.sync()
                for got, ref, plane in zip(eng.readback(sid, desc.dst_slot), want[2], "YUV"):
                    assert np.array_equal(got, ref), (w, h, i, plane)
                eng.release(p)
            eng.close_stream(sid)


@pytest.mark.gpu
def test_mbaff_and_frame_pictures_in_one_batch():
    """MBAFF frames of 1 to 20 pair rows (bands of 4 on workgroups of their own) beside
    frame pictures and a picture without deblocking in the same batches."""
    with Engine(device=0) as eng:
        gens = [Generator(3, width_mbs=w, height_mbs=h, n_frames=3, seed=0xBA9F00 + h, intra_in_inter_permille=200,
                          disable_deblocking_filter_idc=idc) for w, h, idc in [(1, 2, 0), (5, 34, 0), (9, 40, 0), (4, 6, 1)]]
        gens.append(Generator(2, width_mbs=9, height_mbs=5, n_frames=3, seed=0xBA9F99))
        sids = [eng.open_stream_for(g) for g in gens]
        for wants in zip(*(oracle_decode(g) for g in gens)):
            pics = [eng.begin(s, *g.picture(w[0])) for s, g, w in zip(sids, gens, wants)]
            b = eng.batch_create(pics)
            for _ in range(2):
                eng.batch_run(b)
            eng.sync()
            for k, (s, (i, desc, want)) in enumerate(zip(sids, wants)):
                for got, ref, plane in zip(eng.readback(s, desc.dst_slot), want[2], "YUV"):
                    assert np.array_equal(got, ref), (k, i, plane)
            eng.batch_destroy(b)
            for p in pics:
                eng.release(p)


@pytest.mark.gpu
@pytest.mark.parametrize("size", [(1, 8), (2, 10), (7, 16), (8, 18), (9, 24), (17, 26)])
def test_mbaff_band_cuts_match_oracle(size):
    """MBAFF frames of whole bands of 4 pair rows, one row more and one less, narrower and wider
    than what a row hands down at a time (8 pairs)."""
    w, h = size
    with Engine(device=0) as eng:
        gen = Generator(3, width_mbs=w, height_mbs=h, n_frames=4, seed=0xBAA000 + w, qp_lo=26, qp_hi=51, intra_in_inter_permille=200)
        assert gen.mbaff
        sid = eng.open_stream_for(gen)
        for i, desc, want in oracle_decode(gen):
            p = eng.begin(sid, *gen.picture(i))
            eng.submit(p)
            eng.sync()
            for got, ref, plane in zip(eng.readback(sid, desc.dst_slot), want[2], "YUV"):
                assert np.array_equal(got, ref), (size, i, plane)
            eng.release(p)
        eng.close_stream(sid)
