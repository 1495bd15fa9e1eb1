"""The learned initializer's convolutions over the batch sizes where their tiling
changes: one sample (fewer chunks of positions than workgroups), two (every
workgroup one chunk of the first layer) and odd larger ones (workgroups walk
several chunks, unevenly). A sample's activations and input gradients do not
depend on the batch it is in, bit for bit; the batch's weight gradients are the
sum of its samples', which FP32 sums of the same products in another order
reach to 2^-24 per addition: 1e-5 of the gradient's norm bounds it with room.
(Each layer of one batch size is checked against the FP64 oracle in
test_gpu_cnn.py.)
"""

import numpy as np
import pytest

from oracle import cnn as N

pytestmark = pytest.mark.gpu

N_MAX = 7


@pytest.fixture(scope="module")
def samples(hip):
    rng = np.random.default_rng(21)
    z, y, x = np.meshgrid(*(np.arange(64, dtype=np.float32),) * 3, indexing="ij")
    vols = []
    for _ in range(2 * N_MAX):
        c, s = rng.uniform(16, 48, 3), rng.uniform(5, 12)
        v = 100.0 * np.exp(-((x - c[0]) ** 2 + (y - c[1]) ** 2 + (z - c[2]) ** 2) / (2 * s * s))
        vols.append(v + rng.normal(0, 3, v.shape).astype(np.float32))
    dout = rng.normal(0, 0.1, (N_MAX, 12)).astype(np.float32)
    net = hip.CNN(max_batch=1, seed=5)
    p = net.params()
    p += rng.normal(0, 1e-3, p.size).astype(np.float32) * (p != 0)
    net.set_params(p)
    alone = []
    for b in range(N_MAX):
        net.set_input_raw(0, vols[2 * b], vols[2 * b + 1])
        out = net.forward(1)
        net.backward(1, dout[b:b + 1])
        alone.append(dict(out=out[0], acts=[net.activation(i, 1)[0] for i in range(1, 6)],
                          dacts=[net.activation(i, 1, gradient=True)[0] for i in range(1, 6)],
                          grads=net.grads().astype(np.float64)))
    return dict(vols=vols, dout=dout, params=p, alone=alone)


@pytest.mark.parametrize("n", [1, 2, 3, N_MAX])
def test_a_batch_is_its_samples(hip, samples, n):
    net = hip.CNN(max_batch=n, seed=1)
    net.set_params(samples["params"])
    for b in range(n):
        net.set_input_raw(b, samples["vols"][2 * b], samples["vols"][2 * b + 1])
    out = net.forward(n)
    net.backward(n, samples["dout"][:n])
    acts = [net.activation(i, n) for i in range(1, 6)]
    dacts = [net.activation(i, n, gradient=True) for i in range(1, 6)]
    for b in range(n):
        one = samples["alone"][b]
        assert np.array_equal(out[b], one["out"])
        for layer in range(5):
            assert np.array_equal(acts[layer][b], one["acts"][layer]), (b, layer)
            assert np.array_equal(dacts[layer][b], one["dacts"][layer]), (b, layer)
    offs, _ = N.layout()
    got = N.unflatten(net.grads().astype(np.float64), offs)
    want = N.unflatten(sum(s["grads"] for s in samples["alone"][:n]), offs)
    for name, w in want.items():
        assert np.linalg.norm(got[name] - w) <= 1e-5 * max(np.linalg.norm(w), 1e-30), name
