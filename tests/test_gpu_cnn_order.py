"""The order of the training step's sums. Training amplifies rounding (Adam
divides each gradient by its own size: two orders of one FP32 sum, 3e-7 apart in
the first step's gradients, are 3e-2 apart in the fourth's), so the order is
kept for good, and a training run gives the same bits as it always has: the
digests below are those of the first kernels, which added each split of the
positions, and then the splits, one after another. The batch sizes are those
where the splits change: one position split per layer and several, splits that
are (26) and are not (3) cut inside a chunk of staged positions or differ from
the bias gradient's, and the first layer's 256 splits (from 4 on)."""

import hashlib

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

DIGESTS = {1: "a03b209fb863b9c3", 3: "472b1a90b32a6997", 5: "a5c128cc587415d1",
           24: "1d0b3cae3733ed27", 26: "005c0e9852ee68a8"}


def training_digest(hip, n):
    net = hip.CNN(max_batch=n, seed=11)
    for b in range(n):
        vols = [O.synth(100 * n + 2 * b + k, 64 ** 3).reshape(64, 64, 64) for k in range(2)]
        net.set_input_raw(b, *vols)
    targets = np.sin(np.arange(12.0 * n)).astype(np.float32).reshape(n, 12)
    h = hashlib.sha256()
    for _ in range(3):
        loss = net.train_step(n, targets, lr=1e-3)
        h.update(np.float64(loss).tobytes())
        h.update(net.grads().tobytes())
    h.update(net.params().tobytes())
    h.update(net.forward(n).tobytes())
    return h.hexdigest()[:16]


@pytest.mark.parametrize("n", sorted(DIGESTS))
def test_training_keeps_its_bits(hip, n):
    assert training_digest(hip, n) == DIGESTS[n]
