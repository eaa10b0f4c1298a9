"""GPU NCC matcher against the FP64 oracle: every winning score within 1e-5 relative
error, disparity maps agreeing except where FP32 rounding reorders a near tie
(reported and bounded)."""
import ctypes
import time

import numpy as np
import pytest

import clutec_stereo as cs
import orc

pytestmark = pytest.mark.gpu

SCORE_RTOL = 1e-5


def _check(ctx, W, H, D, win, seed, min_agree):
    L, R = cs.synth_pair(seed, W, H, 0, 8, D - 1, min(8, D - 1))
    m = cs.Matcher(ctx, W, H, algorithm=cs.ALGO_NCC, window=win, num_disp=D, tol=1)
    out, lr, rl, score = m.run(L, R, maps=True, scores=True)
    ref_out, ref_l, ref_r, ref_sc, vol = orc.ncc(L, R, D, window=win, tol=1, nthreads=8, with_volume=True)
    valid = ref_l >= 0
    assert np.array_equal(valid, lr >= 0)
    # score of the GPU's own winner against the FP64 score of the same candidate
    yy, xx = np.nonzero(valid)
    s64 = vol[yy, xx, lr[yy, xx]]
    s32 = score[yy, xx].astype(np.float64)
    zero = s64 == 0.0
    assert (s32[zero] == 0.0).all()
    rel = np.abs(s32[~zero] - s64[~zero]) / np.abs(s64[~zero])
    print(f"ncc {W}x{H} D={D} win={win}: max rel score error {rel.max():.3e}", flush=True)
    assert rel.max() <= SCORE_RTOL
    agree_l = (lr == ref_l).mean()
    agree_r = (rl == ref_r).mean()
    agree = (out == ref_out).mean()
    print(f"  agreement left {agree_l:.6f} right {agree_r:.6f} checked {agree:.6f}", flush=True)
    assert agree_l >= min_agree and agree_r >= min_agree and agree >= min_agree
    # where the maps differ the two candidates are tied to within FP32 rounding
    dif = np.nonzero((lr != ref_l) & valid)
    if dif[0].size:
        a = vol[dif[0], dif[1], lr[dif]]
        b = vol[dif[0], dif[1], ref_l[dif]]
        assert np.all(np.abs(a - b) <= 1e-6)


def _short(W, H, D, win):
    """The rule for the running sums."""
    return D <= (48 if win >= 9 else 32) and W * H * (2 if win >= 9 else 1) >= 55000 * D


@pytest.mark.parametrize("win", [(11, 11), (9, 9), (5, 5)])
def test_ncc_small(ctx, win):
    _check(ctx, 210, 96, 64, win, 31, 0.999)


def test_ncc_tall_segments(ctx):
    _check(ctx, 333, 130, 128, (7, 7), 32, 0.999)


@pytest.mark.parametrize("W,H,D,win", [
    (65, 33, 8, 11), (64, 32, 8, 5), (127, 35, 24, 7), (128, 37, 32, 9), (129, 34, 40, 11), (161, 33, 64, 11),
    (255, 34, 256, 5), (300, 35, 248, 11), (385, 33, 256, 9), (641, 40, 200, 7)])
def test_ncc_tiles(ctx, W, H, D, win):
    """Blocks of 32 x 32 candidates, tiles of 128 columns and 2 rows, segments of 32 or 64
    disparities: one column and row more and less, ranges that end inside a block, images narrower
    than their range."""
    assert not _short(W, H, D, win) and -(-W // 128) * -(-H // 4) < 1024  # the rule for 2 rows
    _check(ctx, W, H, D, (win, win), W + D, 0.99)


# Tiles of 4 rows, one segment: heights 1 and 2 past a tile, a column past and before one, ranges of 72
# (blocks up to 96) to 256.
@pytest.mark.parametrize("W,H,D,win", [(1023, 769, 192, 9), (1025, 770, 72, 11), (897, 514, 104, 7), (1153, 459, 256, 5)])
def test_ncc_tiles_of_four_rows(ctx, W, H, D, win):
    assert not _short(W, H, D, win) and -(-W // 128) * -(-H // 4) >= 1024 and H % 4  # the rule
    _check(ctx, W, H, D, (win, win), W + D, 0.99)


@pytest.mark.parametrize("W,H,D,win", [
    (1001, 449, 8, 5), (1283, 417, 8, 11), (1283, 701, 16, 7), (961, 701, 24, 9), (1153, 767, 32, 11),
    (2053, 873, 32, 5), (1291, 1030, 40, 11), (1291, 1030, 48, 9)])
def test_ncc_short_ranges(ctx, W, H, D, win):
    """Short ranges of large frames, which take the running sums: ragged tiles of 64 x 52, one group of 8
    disparities, whole and cut statistics tiles of 16, one to three segments."""
    assert _short(W, H, D, win)
    _check(ctx, W, H, D, (win, win), W + D, 0.99)


def test_ncc_short_range_costs_less(ctx):
    """A 1920 x 1080 frame of 8 disparities takes clearly less than one of 64 (0.41 of it; 0.91 where all ranges
    took the same kernel)."""
    W, H = 1920, 1080
    L, R = cs.synth_pair(3, W, H, 0, 8, 63, 8)
    l, r = (cs.DeviceImage.from_array(ctx, a, cs.PIXEL_LUM_U8) for a in (L, R))
    out = cs.DeviceImage(ctx, W, H, cs.PIXEL_LUM_I16)
    best = {}
    for D in (64, 8):
        m = cs.Matcher(ctx, W, H, algorithm=cs.ALGO_NCC, window=(11, 11), num_disp=D, tol=1)
        for _ in range(8):
            t = time.perf_counter()
            for _ in range(40):
                m.process(out, None, None, l, r)
            cs._check(cs.lib.stereo_synchronize(ctx.handle, None), ctx)
            best[D] = min(best.get(D, 1.0), time.perf_counter() - t)
    print({d: round(v / 40 * 1e6, 1) for d, v in best.items()}, "us", flush=True)
    assert best[8] < 0.7 * best[64]


@pytest.mark.parametrize("W,H,D,off,more", [(201, 37, 64, 0, 2), (201, 37, 64, 1, 3), (201, 37, 64, 3, 6),
                                            (1025, 431, 16, 1, 3)])
def test_ncc_any_alignment(ctx, W, H, D, off, more):
    """Images at any address and row pitch give the maps of the aligned ones."""
    pitch = W + more
    L, R = cs.synth_pair(5, W, H, 0, 8, D - 1, 8)
    m = cs.Matcher(ctx, W, H, algorithm=cs.ALGO_NCC, window=(11, 11), num_disp=D, tol=1)
    want = m.run(L, R, maps=True, scores=True)

    class View:
        def __init__(self, a):
            raw = np.zeros(off + H * pitch, np.uint8)
            for y in range(H):
                raw[off + y * pitch:off + y * pitch + W] = a[y]
            self.buf = cs.DeviceBuffer.from_array(ctx, raw)
            self.img = cs.Image(self.buf.ptr.value + off, pitch, cs.ImageFormat(W, H, cs.PIXEL_LUM_U8))
            self.ref = ctypes.byref(self.img)

    l, r = View(L), View(R)
    outs = [cs.DeviceImage(ctx, W, H, cs.PIXEL_LUM_I16) for _ in range(3)]
    m.process(*outs, l, r)
    score = cs.DeviceImage(ctx, W, H, cs.PIXEL_LUM_F32)
    cs._check(cs.lib.stereo_matcher_scores(m.handle, score.ref, l.ref, r.ref, None), ctx)
    for got, ref in zip([o.download() for o in outs] + [score.download()], want):
        assert np.array_equal(got, ref, equal_nan=got.dtype == np.float32)


def test_ncc_config1_rows(ctx):
    """1920-wide, D=256, 11x11: the headline NCC workload on a 160-row band."""
    W, H, D = 1920, 160, 256
    L, R = cs.synth_pair(1, 1920, 1080, 0, 24, 255, 8)
    L, R = np.ascontiguousarray(L[400:400 + H]), np.ascontiguousarray(R[400:400 + H])
    m = cs.Matcher(ctx, W, H, algorithm=cs.ALGO_NCC, window=(11, 11), num_disp=D, tol=1)
    out, lr, rl, score = m.run(L, R, maps=True, scores=True)
    ref_out, ref_l, ref_r, ref_sc = orc.ncc(L, R, D, window=(11, 11), tol=1, nthreads=8)
    same = (lr == ref_l) & (lr >= 0)
    rel = np.abs(score[same] - ref_sc[same]) / np.maximum(np.abs(ref_sc[same]), 1e-30)
    nz = ref_sc[same] != 0
    print(f"1080p band: agreement {(lr == ref_l).mean():.6f}, max rel score error {rel[nz].max():.3e}", flush=True)
    assert rel[nz].max() <= SCORE_RTOL
    assert (lr == ref_l).mean() >= 0.999 and (out == ref_out).mean() >= 0.998


def test_ncc_scores_need_ncc(ctx):
    m = cs.Matcher(ctx, 64, 32, algorithm=cs.ALGO_SAD, window=(5, 5), num_disp=16)
    with pytest.raises(cs.StereoError) as e:
        m.run(np.zeros((32, 64), np.uint8), np.zeros((32, 64), np.uint8), scores=True)
    assert e.value.status == cs.ERROR_INVALID_CONFIG
