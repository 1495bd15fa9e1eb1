"""The mean-squares column walk (every voxel of a grid, FP32) against the general
sample walk, which the same voxels given as an index list take: the same
samples valid, and the same per-sample FP32 arithmetic but for samples within
a rounding of the 1e-6 guard, where one of the two runs the exact chain (the
composed map is within 5e-13 voxel of it), so the sums agree to 1e-9 of their
norm. Sizes around the tiles (256 in-plane voxels, 64 planes) and around the rule
that sends thin and flat grids to the general walk (a quarter of the lanes idle,
fewer than eight planes), axes of one and two voxels, poses that put every sample on a voxel, on a
half voxel, across every face and fully outside, masks, two stages, and maps
of NaN and infinity, which no sample survives."""

import numpy as np
import pytest

from helpers import blob_volume

pytestmark = pytest.mark.gpu

SIZES = [(2, 2, 2), (1, 9, 8), (16, 16, 64), (17, 15, 65), (16, 17, 130), (64, 4, 3), (61, 67, 40),
         (16, 25, 130), (2, 128, 9), (128, 2, 8), (16, 12, 8)]


def _rot(a, b, c):
    ca, sa, cb, sb, cc, sc = np.cos(a), np.sin(a), np.cos(b), np.sin(b), np.cos(c), np.sin(c)
    return (np.array([[cc, -sc, 0], [sc, cc, 0], [0, 0, 1.0]]) @
            np.array([[1.0, 0, 0], [0, ca, -sa], [0, sa, ca]]) @
            np.array([[cb, 0, sb], [0, 1.0, 0], [-sb, 0, cb]]))


def _stage(m, centre, t):
    return np.concatenate([m.reshape(9), centre + t - m @ centre])


def _pair(hip, size, mask):
    sp, org = (1.0, 0.8, 1.3), (-4.0, 2.0, 1.0)
    f = blob_volume(size[::-1], 3, spacing=sp)
    m = blob_volume(size[::-1], 4, spacing=sp)
    geo = dict(spacing=sp, origin=org)
    df, dm = hip.DeviceImage.upload(f, **geo), hip.DeviceImage.upload(m, **geo)
    kw = {}
    if mask:
        mk = (np.random.default_rng(5).random(size[::-1]) > 0.3).astype(np.uint8)
        kw["moving_mask"] = hip.DeviceMask.upload(mk, **geo)
    idx = np.arange(f.size, dtype=np.int64)
    centre = np.array(org) + 0.5 * (np.array(size) - 1) * np.array(sp)
    return hip.ResidentMetric(df, dm, **kw), hip.ResidentMetric(df, dm, indices=idx, **kw), centre, sp


def _check(walk, general, stages):
    got, want = walk.evaluate(stages), general.evaluate(stages)
    assert got[13] == want[13]
    assert np.linalg.norm(got - want) <= 1e-9 * max(np.linalg.norm(want), 1e-300), (got, want)
    (sq, n), (sq_w, n_w) = walk.value(stages), general.value(stages)
    assert n == n_w == int(want[13]) and abs(sq - sq_w) <= 1e-9 * abs(sq_w)


@pytest.mark.parametrize("size", SIZES)
@pytest.mark.parametrize("mask", [False, True])
def test_columns_are_the_sample_walk(hip, size, mask):
    walk, general, c, sp = _pair(hip, size, mask)
    eye = np.eye(3)
    poses = [_stage(eye, c, np.zeros(3)),                      # every sample on a voxel
             _stage(eye, c, 0.5 * np.array(sp)),               # every sample on a half voxel
             _stage(_rot(0.1, -0.07, 0.2), c, np.array([0.7, -0.4, 0.9])),
             _stage(_rot(np.pi / 2, 0.0, 0.0), c, np.zeros(3)),
             _stage(1.3 * _rot(0.5, 0.4, -0.3), c, np.array([3.0, 2.0, -2.0])),
             _stage(eye, c, np.array([1e4, 0.0, 0.0]))]        # nothing inside
    for st in poses:
        _check(walk, general, st.reshape(1, 12))
    _check(walk, general, np.stack([poses[2], poses[4]]))      # two stages


@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf, 1e300])
def test_samples_without_a_finite_point_are_dropped(hip, bad):
    """(1e300 as a scale leaves the plane it maps to a finite point: the sums
    are then those of that plane, within the bound above.)"""
    walk, general, c, _ = _pair(hip, (17, 15, 9), False)
    for k in (0, 10):
        st = _stage(np.eye(3), c, np.zeros(3))
        st[k] = bad
        _check(walk, general, st.reshape(1, 12))
        if not np.isfinite(bad):
            assert walk.evaluate(st.reshape(1, 12))[13] == 0


def test_one_batch_of_both_walks(hip):
    """A batch's tiles of the column walk: the single evaluation's sums."""
    metrics, stages, singles = [], [], []
    for i, size in enumerate(SIZES):
        walk, _, c, _ = _pair(hip, size, bool(i % 2))
        st = _stage(_rot(0.05 * i, -0.03, 0.02), c, np.array([0.4, 0.3 * i, -0.2]))
        metrics.append(walk)
        stages.append(st)
        singles.append(walk.evaluate(st.reshape(1, 12)))
    b = hip.Batch(metrics)
    for tile in (256, 1024, 4096, 1 << 20):
        b.set_tiling(tile)
        vals, mom, valid = b.evaluate(np.stack(stages))
        for i, w in enumerate(singles):
            assert valid[i] == int(w[13])
            assert np.linalg.norm(mom[i] - w) <= 1e-12 * max(np.linalg.norm(w), 1e-300)


@pytest.mark.parametrize("size,columns", [((16, 12, 8), True), ((16, 12, 7), False), ((17, 11, 64), False),
                                          ((8, 8, 300), False), ((16, 17, 40), False),
                                          ((16, 24, 40), True), ((2, 96, 8), True), ((1, 256, 64), False)])
def test_thin_and_flat_grids_take_the_general_walk(hip, size, columns):
    """A column walk leaves the lanes without an in-plane voxel idle: 8 x 8 x
    40,000 voxels took it twice as long as the general walk."""
    walk, _, c, _ = _pair(hip, size, False)
    st = _stage(np.eye(3), c, np.array([0.3, 0.2, -0.1])).reshape(1, 12)
    hip.profile_enable(True)
    try:
        hip.profile_reset()
        walk.evaluate(st)
        walk.value(st)
        seen = [hip.profile_query(n)[0] for n in ("ms_moments", "ms_moments_columns", "ms_value",
                                                  "ms_value_columns")]
    finally:
        hip.profile_enable(False)
    assert seen == [1, int(columns), 1, int(columns)]
