"""The linear resample against the oracle, bit for bit, where its paired corner
loads have edges: volumes of one, two and three voxels along x, points on and
past both faces, exact voxel hits next to infinite and NaN voxels (a corner of
zero weight contributes nothing, whatever it holds)."""

import numpy as np
import pytest

import oracle as O
from helpers import stages_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size", [(1, 5, 4), (2, 3, 7), (3, 1, 2), (5, 4, 1), (17, 9, 6)])
@pytest.mark.parametrize("special", [False, True])
def test_resample_is_the_oracles(hip, size, special):
    rng = np.random.default_rng(sum(size))
    v = rng.normal(100.0, 30.0, size[::-1]).astype(np.float32)
    if special:
        flat = v.reshape(-1)
        flat[0], flat[-1] = np.inf, np.nan
    sp, org = (1.0, 0.8, 1.25), (-2.0, 1.0, 3.0)
    img = hip.DeviceImage.upload(v, spacing=sp, origin=org)
    out_size = (11, 9, 8)
    osp = tuple(1.3 * s * n / o for s, n, o in zip(sp, size, out_size))
    oorg = tuple(o - 0.7 * s for o, s in zip(org, sp))
    grids = [(size, sp, org), (out_size, osp, oorg)]  # every voxel hit exactly; past every face
    for params in ([0.0] * 6, [0.3, -0.2, 0.1, 0.4, 0.0, -0.3]):
        t = O.make_transform(O.EULER3D, params, center=[0.0, 2.0, 4.0])
        for gsize, gsp, gorg in grids:
            want = O.resample_linear(v, sp, org, gsize, gsp, gorg, t, default=-7.0)
            got = hip.resample_linear(img, hip.Geometry.make(gsize, gsp, gorg), stages_of(t),
                                      default_value=-7.0).to_host()
            assert np.array_equal(got, want, equal_nan=True), (params, gsize)


@pytest.mark.parametrize("fine", [(a, b, c) for a in (0, 1) for b in (0, 1) for c in (0, 1)])
def test_axes_that_fall_on_voxels(hip, fine):
    """Grids whose voxels fall on voxels along some axes and between them along
    the others, for whole waves (140 voxels to a row) and for parts of one: the
    corners that a wave leaves out are those whose weight is zero in every lane.
    Infinite and NaN voxels lie where a corner that should not count would read
    them: one beyond the exact axes, and past the last voxel."""
    size, sp, org = (70, 6, 5), (1.0, 1.0, 1.0), (0.0, 0.0, 0.0)
    rng = np.random.default_rng(8)
    v = rng.normal(100.0, 30.0, size[::-1]).astype(np.float32)
    v[3, 4, 40:] = np.nan
    v[2, 1, :20] = np.inf
    img = hip.DeviceImage.upload(v)
    for step in (0.5, 0.75):
        gsp = [step if f else 1.0 for f in fine]
        gsize = [2 * n if f else n for n, f in zip(size, fine)]
        t = O.make_transform(O.TRANSLATION, [0.0, 0.0, 0.0])
        want = O.resample_linear(v, sp, org, tuple(gsize), tuple(gsp), org, t, default=-7.0)
        got = hip.resample_linear(img, hip.Geometry.make(gsize, gsp, org), default_value=-7.0).to_host()
        assert np.array_equal(got, want, equal_nan=True), step
