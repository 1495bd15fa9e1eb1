"""The recursive Gaussian's two-lane kernel over the line lengths where it changes
shape, bit for bit against the oracle: no register block pairs up to all five
(one more every 32 voxels from 40 to 168), whole and partial blocks before and
after the middle, odd lengths, lines whose parked values stay within 64 KB of LDS
(to 417), need more (to 801, 160 KB), or do not fit at all (the one-lane kernel, from
802), along each axis, alone (float to float) and with the others (through
FP64), with a last workgroup that is not full."""

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

LENGTHS = [8, 9, 10, 13, 15, 16, 17, 23, 24, 39, 40, 41, 42, 55, 56, 71, 72, 73, 88, 89, 103, 104,
           135, 136, 137, 150, 161, 167, 168, 169, 199, 200, 201, 256, 385, 416, 417, 418, 641, 767, 780, 800,
           801, 802, 1001]


@pytest.mark.parametrize("n", LENGTHS)
def test_lines_of(hip, n):
    for axis in range(3):
        size = [37, 9, 10]
        size[axis] = n
        v = O.synth(77 + n + axis, size[0] * size[1] * size[2]).reshape(size[::-1])
        img = hip.DeviceImage.upload(v)
        alone = [0.0, 0.0, 0.0]
        alone[axis] = 1.7
        for sigma in (alone, [1.1, 2.3, 0.9]):
            want = O.smoothing_recursive_gaussian(v, tuple(size), (1, 1, 1), sigma)
            got = hip.recursive_gaussian(img, sigma).to_host().reshape(-1)
            assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), (axis, sigma)


def test_a_batch_of_ragged_volumes_is_its_volumes(hip):
    rng = np.random.default_rng(3)
    sizes = [tuple(int(x) for x in rng.integers(8, 140, 3)) for _ in range(7)]
    sizes += [(300, 9, 8), (8, 8, 8), (7, 20, 20), (9, 1001, 8), (801, 8, 9)]
    imgs = [hip.DeviceImage.upload(O.synth(i, s[0] * s[1] * s[2]).reshape(s[::-1]))
            for i, s in enumerate(sizes)]
    sigma = [[1.0 + 0.1 * i, 0.8, 2.0] for i in range(len(sizes))]
    for i, (img, s, out) in enumerate(zip(imgs, sigma, hip.recursive_gaussian_batch(imgs, sigma))):
        got = out.to_host()
        want = hip.recursive_gaussian(img, s).to_host()
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
        if max(sizes[i]) > 780:  # the one-lane kernel's volume, and the longest of the other's
            ref = O.smoothing_recursive_gaussian(img.to_host(), sizes[i], (1, 1, 1), s)
            assert np.array_equal(got.reshape(-1).view(np.uint32), ref.view(np.uint32))
