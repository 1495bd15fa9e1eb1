"""The work that programs built on this library have it do, as timed cases.

Each case goes through the public entry points of ``sitk_hip`` (the binding of
the C ABI): one Mattes or mean-squares evaluation, the recursive Gaussian of the
pyramid, a batched evaluation of many pairs, a B-spline evaluation, the learned
initializer's forward and training step, and whole batched registrations. The
sizes are those of the repository's own workloads (``workload.py``, ``bench.py``,
the tests) and ragged ones around them. Volumes are sums of Gaussian blobs with
voxel noise, as the repository's generators make them; a pair's moving volume
is the rigidly moved scene with noise of its own.

``exact`` restates every path in 64 bits with plain torch, without this
library's code.
"""

import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "sitk-rs_amd"))
import sitk_hip as S  # noqa: E402

DEV = "cuda:0"


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # The coarsest level of a three-level registration of one large pair:
        # the launches and the host round trip are most of the time.
        dict(name="mattes_coarse", op="mattes", nx=64, ny=64, nz=40, sx=3.6, sy=3.6, sz=6.0,
             bins=50, percent=20.0, f64=False, masks=False),
        # Its finest level: the evaluation an optimizer makes hundreds of times.
        dict(name="mattes_full", op="mattes", nx=256, ny=256, nz=160, sx=0.9, sy=0.9, sz=1.5,
             bins=50, percent=20.0, f64=False, masks=False),
        # Parity checks: the FP64 path, an odd grid, a fixed and a moving mask.
        dict(name="mattes_f64_masked", op="mattes", nx=129, ny=117, nz=65, sx=1.0, sy=1.0, sz=2.0,
             bins=32, percent=25.0, f64=True, masks=True),
        # Mean squares of a same-modality pair over every voxel.
        dict(name="ms_full", op="ms", nx=256, ny=256, nz=256, sx=1.0, sy=1.0, sz=1.0, percent=100.0,
             f64=False, masks=False),
        # Pyramid smoothing of one large volume, and of a batch's ragged volumes.
        dict(name="smooth_full", op="smooth", n=1, lo=256, hi=256, nz=160, sigma=2.0),
        dict(name="smooth_batch", op="smooth", n=48, lo=32, hi=128, nz=0, sigma=1.0),
        # One optimizer iteration of many rigid pairs of uneven sizes (even
        # pairs mean squares on every voxel, odd pairs Mattes at 25%).
        dict(name="batch_pairs", op="batch", n=96, lo=32, hi=128, bins=32, percent=25.0),
        # A deformable registration's evaluation: one start, and many at once.
        dict(name="bspline_one", op="bspline", edge=192, mesh=7, starts=1, bins=32, percent=10.0),
        dict(name="bspline_starts", op="bspline", edge=192, mesh=7, starts=64, bins=32,
             percent=10.0),
        # The learned initializer: prediction of a batch, one training step.
        dict(name="cnn_predict", op="cnn", train=False, n=32, lo=128, hi=128),
        dict(name="cnn_train", op="cnn", train=True, n=24, lo=128, hi=128),
        # Whole registrations of many small pairs together, pyramid included.
        dict(name="register_pairs", op="register", n=32, lo=40, hi=96, bins=32, percent=25.0,
             iterations=25),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["mattes", "mattes", "ms", "smooth", "smooth", "batch", "bspline", "cnn", "cnn",
                     "register"])
    if op in ("mattes", "ms"):
        # an axis of up to 256 voxels, in-plane axes near one another
        e = _log_int(rng, 24, 256)
        size = [max(16, min(256, int(e * rng.uniform(0.75, 1.25)))) for _ in range(2)]
        nz = max(12, min(256 if op == "ms" else 160, int(e * rng.uniform(0.4, 1.0))))
        c = dict(op=op, nx=size[0], ny=size[1], nz=nz, sx=round(rng.uniform(0.7, 1.3), 2),
                 sy=round(rng.uniform(0.7, 1.3), 2), sz=round(rng.uniform(0.8, 3.0), 2),
                 f64=rng.random() < 0.25, masks=rng.random() < 0.25)
        if op == "mattes":
            c.update(bins=rng.choice([16, 24, 32, 50, 64]), percent=rng.choice([5.0, 10.0, 20.0]))
        else:
            c.update(percent=rng.choice([25.0, 100.0, 100.0]))
        return c
    if op == "smooth":
        if rng.random() < 0.5:
            e = _log_int(rng, 24, 240)
            return dict(op=op, n=1, lo=e, hi=int(e * 1.05) + 1, nz=max(16, min(160, int(e * 0.6))),
                        sigma=round(rng.uniform(0.8, 4.0), 2))
        lo = rng.randint(24, 48)
        return dict(op=op, n=rng.randint(3, 48), lo=lo, hi=rng.randint(lo + 8, 112), nz=0,
                    sigma=round(rng.uniform(0.8, 2.5), 2))
    if op == "batch":
        lo = rng.randint(24, 48)
        return dict(op=op, n=_log_int(rng, 4, 96), lo=lo, hi=rng.randint(lo + 8, 112),
                    bins=rng.choice([16, 32, 50]), percent=rng.choice([10.0, 25.0]))
    if op == "bspline":
        return dict(op=op, edge=rng.randint(72, 176), mesh=rng.randint(3, 9),
                    starts=_log_int(rng, 1, 48), bins=rng.choice([24, 32, 50]),
                    percent=rng.choice([5.0, 10.0]))
    if op == "cnn":
        lo = rng.randint(64, 128)
        return dict(op=op, train=rng.random() < 0.5, n=_log_int(rng, 1, 24), lo=lo,
                    hi=rng.randint(lo, 136))
    lo = rng.randint(32, 56)
    return dict(op=op, n=_log_int(rng, 1, 24), lo=lo, hi=rng.randint(lo + 8, 88),
                bins=rng.choice([24, 32]), percent=25.0, iterations=rng.randint(10, 25))


# ------------------------------------------------------------- synthetic input
class Pair:
    """A fixed and a moving volume of one scene (float32, device), identity
    direction, and a point-map stage near the map that aligns them."""

    def __init__(self, gen, size, spacing, nblobs=40, mm=4.0, deg=5.0, miss=1.0):
        self.size, self.spacing = tuple(size), tuple(spacing)
        ext = torch.tensor([n * s for n, s in zip(size, spacing)], dtype=torch.float64)
        self.origin = (-3.0, 2.0, 1.0)
        org = torch.tensor(self.origin, dtype=torch.float64)
        u = torch.rand(nblobs, 5, generator=gen, dtype=torch.float64)
        centres = org + u[:, :3] * ext
        amps, sigmas = 50.0 + 150.0 * u[:, 3], 2.0 + 6.0 * u[:, 4]
        mid = org + 0.5 * ext
        ang, t = self._uniform(gen, math.radians(deg)), self._uniform(gen, mm)
        rot = _rotation(ang)
        self.fixed = self._volume(gen, centres, amps, sigmas)
        self.moving = self._volume(gen, (centres - mid) @ rot.T + mid + t, amps, sigmas)
        # the evaluated pose misses the aligning one a little
        rot = _rotation(ang + miss * self._uniform(gen, math.radians(1.0)))
        t = t + miss * self._uniform(gen, 1.0)
        self.centre = mid
        self.stage = torch.cat([rot.reshape(9), mid + t - rot @ mid]).numpy()

    @staticmethod
    def _uniform(gen, a):
        return (2.0 * torch.rand(3, generator=gen, dtype=torch.float64) - 1.0) * a

    def _volume(self, gen, centres, amps, sigmas):
        g = []
        for d in range(3):
            x = self.origin[d] + self.spacing[d] * torch.arange(self.size[d], dtype=torch.float64)
            g.append(torch.exp(-((x[None] - centres[:, d:d + 1]) ** 2) / (2 * sigmas[:, None] ** 2)))
        g = [v.float().to(DEV) for v in g]
        plane = (g[1][:, :, None] * g[0][:, None, :]).reshape(len(amps), -1)
        v = ((g[2] * amps.float().to(DEV)[:, None]).T.contiguous() @ plane)
        noise = torch.Generator(DEV)
        noise.manual_seed(int(torch.randint(1 << 40, (1,), generator=gen)))
        v = v.reshape(self.size[::-1])
        return v + 5.0 * torch.randn(v.shape, generator=noise, device=DEV)

    def images(self):
        geo = dict(spacing=self.spacing, origin=self.origin)
        return (S.DeviceImage.upload(self.fixed.cpu().numpy(), **geo),
                S.DeviceImage.upload(self.moving.cpu().numpy(), **geo))


def _rotation(a):
    c, s = torch.cos(a).tolist(), torch.sin(a).tolist()
    rx = torch.tensor([[1, 0, 0], [0, c[0], -s[0]], [0, s[0], c[0]]], dtype=torch.float64)
    ry = torch.tensor([[c[1], 0, s[1]], [0, 1, 0], [-s[1], 0, c[1]]], dtype=torch.float64)
    rz = torch.tensor([[c[2], -s[2], 0], [s[2], c[2], 0], [0, 0, 1]], dtype=torch.float64)
    return rz @ rx @ ry


def _samples(gen, voxels, percent):
    """Random draws with replacement; None for every voxel in order."""
    if percent >= 100.0:
        return None
    return torch.randint(voxels, (int(voxels * percent / 100.0),), generator=gen)


def _ellipsoid(size, radius):
    ax = [(torch.arange(n, dtype=torch.float32) - 0.5 * (n - 1)) / (0.5 * n * radius) for n in size]
    return (ax[2][:, None, None] ** 2 + ax[1][None, :, None] ** 2 + ax[0][None, None, :] ** 2) <= 1.0


class _View:
    """A device image's voxels as a torch tensor sees them (no copy)."""

    def __init__(self, img):
        g = img.geometry()
        self.img = img
        self.__cuda_array_interface__ = {
            "shape": (g.size[2], g.size[1], g.size[0]), "typestr": "<f4", "version": 2,
            "data": (img.device_ptr(), False), "strides": None}


def _tensor(img):
    return torch.as_tensor(_View(img), device=DEV)


# The sizes of a ragged set depend on the case alone, so that `work` knows them.
def _ragged(case, n):
    r = torch.Generator()
    r.manual_seed(1000 * case["lo"] + case["hi"] + n)
    return torch.randint(case["lo"], case["hi"] + 1, (n, 3), generator=r).tolist()


def _smooth_sizes(case):
    if case["n"] == 1:
        return [[case["lo"], case["hi"], case["nz"]]]
    return _ragged(case, case["n"])


# Everything random of a case, from its seed (used by prepare and by exact).
def _inputs(case, seed):
    gen = torch.Generator()
    gen.manual_seed(seed)
    op = case["op"]
    if op in ("mattes", "ms"):
        size = (case["nx"], case["ny"], case["nz"])
        p = Pair(gen, size, (case["sx"], case["sy"], case["sz"]))
        idx = _samples(gen, math.prod(size), case["percent"])
        masks = (_ellipsoid(size, 0.95), _ellipsoid(size, 0.9)) if case["masks"] else None
        return dict(pair=p, idx=idx, masks=masks)
    if op == "smooth":
        sp = (0.9, 0.9, 1.5) if case["n"] == 1 else (1.0, 1.0, 1.0)
        return dict(pairs=[Pair(gen, s, sp) for s in _smooth_sizes(case)], spacing=sp)
    if op in ("batch", "register"):
        pairs = [Pair(gen, s, (1.0, 1.0, 1.0)) for s in _ragged(case, case["n"])]
        idx = [_samples(gen, math.prod(p.size), case["percent"] if i % 2 else 100.0)
               for i, p in enumerate(pairs)]
        return dict(pairs=pairs, idx=idx)
    if op == "bspline":
        e = case["edge"]
        p = Pair(gen, (e, e, e), (1.0, 1.0, 1.0), nblobs=135, miss=0.0)
        idx = _samples(gen, e ** 3, case["percent"])
        ncp = (case["mesh"] + 3) ** 3
        coef = torch.randn(case["starts"], 3 * ncp, generator=gen, dtype=torch.float64)
        stages = []
        for _ in range(case["starts"]):  # perturbed starts, as a multi-start run makes them
            rot = _rotation(Pair._uniform(gen, math.radians(2.0)))
            t = Pair._uniform(gen, 2.0)
            m = torch.from_numpy(p.stage)
            a = rot @ m[:9].reshape(3, 3)
            stages.append(torch.cat([a.reshape(9), rot @ (m[9:] - p.centre) + p.centre + t]))
        return dict(pair=p, idx=idx, coef=coef, stages=torch.stack(stages))
    pairs = [Pair(gen, s, (1.0, 1.0, 1.0), mm=10.0, deg=20.0) for s in _ragged(case, case["n"])]
    return dict(pairs=pairs, params=_cnn_params(gen),
                targets=0.2 * torch.randn(case["n"], 12, generator=gen))


# --------------------------------------------------------------- prepare / run
def _resident(pair, idx, masks=None, bins=None, f64=False):
    fixed, moving = pair.images()
    kw = dict(indices=None if idx is None else idx.numpy(),
              precision=S.PRECISION_F64 if f64 else S.PRECISION_F32)
    if masks is not None:
        geo = dict(spacing=pair.spacing, origin=pair.origin)
        kw["fixed_mask"] = S.DeviceMask.upload(masks[0].numpy().astype(np.uint8), **geo)
        kw["moving_mask"] = S.DeviceMask.upload(masks[1].numpy().astype(np.uint8), **geo)
    if bins is None:
        return S.ResidentMetric(fixed, moving, **kw)
    return S.ResidentMattes(fixed, moving, bins=bins, **kw)


def prepare(case, seed):
    S.backend_init(0)
    x = _inputs(case, seed)
    op = case["op"]
    st = dict(case=case)
    if op in ("mattes", "ms"):
        st["metric"] = _resident(x["pair"], x["idx"], x["masks"], case.get("bins"), case["f64"])
        st["stage"] = x["pair"].stage.reshape(1, 12)
    elif op == "smooth":
        st["images"] = [p.images()[0] for p in x["pairs"]]
        st["sigma"] = [[case["sigma"]] * 3] * len(x["pairs"])
    elif op == "batch":
        st["batch"] = S.Batch([_resident(p, i, bins=None if i is None else case["bins"])
                               for p, i in zip(x["pairs"], x["idx"])])
        st["stages"] = np.stack([p.stage for p in x["pairs"]])
    elif op == "bspline":
        p = x["pair"]
        m = _resident(p, x["idx"], bins=case["bins"])
        gsp = case["edge"] / case["mesh"]
        b = S.BSplineMattes(m, [case["mesh"] + 3] * 3, [o - gsp for o in p.origin], [gsp] * 3)
        st["coef"] = x["coef"].numpy()
        if case["starts"] == 1:
            b.set_moving_initial(x["stages"][0].numpy())
            st["one"] = b
        else:
            st["many"] = S.BSplineMulti(b, case["starts"], stages=x["stages"].numpy())
    elif op == "cnn":
        st["net"] = S.CNN(max_batch=case["n"])
        st["net"].set_params(x["params"].numpy())
        imgs = [p.images() for p in x["pairs"]]
        st["fixed"], st["moving"] = [f for f, _ in imgs], [m for _, m in imgs]
        st["targets"] = x["targets"].numpy()
    else:
        imgs = [p.images() for p in x["pairs"]]
        st["fixed"], st["moving"] = [f for f, _ in imgs], [m for _, m in imgs]
        st["centres"] = [p.centre.tolist() for p in x["pairs"]]
        st["configs"] = [
            S.registration_config(
                metric=S.MATTES if i % 2 else S.MEAN_SQUARES, bins=case["bins"],
                sampling=S.SAMPLING_RANDOM if i % 2 else S.SAMPLING_NONE,
                sampling_percentage=case["percent"] / 100.0, seed=17 + i, minimum_step=1e-3,
                iterations=case["iterations"], gradient_tolerance=1e-8,
                learning_rate_mode=S.LR_ONCE, shrink_factors=((2, 2, 2), (1, 1, 1)),
                sigmas=(1.0, 0.0)) for i in range(case["n"])]
    return st


def run(st):
    case = st["case"]
    op = case["op"]
    if op == "mattes":
        value, moments, valid = st["metric"].value_and_moments(st["stage"])
        return dict(value=np.float64(value), moments=moments, valid=valid)
    if op == "ms":
        return dict(moments=st["metric"].evaluate(st["stage"]))
    if op == "smooth":
        if case["n"] == 1:
            st["out"] = [S.recursive_gaussian(st["images"][0], st["sigma"][0])]
        else:
            st["out"] = S.recursive_gaussian_batch(st["images"], st["sigma"])
        return [_tensor(o) for o in st["out"]]
    if op == "batch":
        values, moments, valid = st["batch"].evaluate(st["stages"])
        return dict(ms_value=values[0::2], ms_moments=moments[0::2], mattes_value=values[1::2],
                    mattes_moments=moments[1::2], valid=valid.astype(np.int64))
    if op == "bspline":
        if case["starts"] == 1:
            value, deriv, valid = st["one"].value_and_derivative(st["coef"][0])
            return dict(value=np.float64(value), deriv=deriv, valid=valid)
        values, derivs, valid = st["many"].value_and_derivative(st["coef"])
        return dict(value=values, deriv=derivs, valid=valid.astype(np.int64))
    if op == "cnn":
        net = st["net"]
        net.set_inputs(0, st["fixed"], st["moving"])
        if not case["train"]:
            return dict(out=net.forward(case["n"]))
        loss = net.train_step(case["n"], st["targets"], lr=1e-3)
        return dict(loss=loss, grads=net.grads())
    n = case["n"]
    if n == 1:
        params, res = S.register(st["fixed"][0], st["moving"][0], st["configs"][0], S.EULER3D,
                                 [0.0] * 6, center=st["centres"][0])
        return dict(params=params, value=np.float64(res.value))
    params, res = S.register_batch(st["fixed"], st["moving"], st["configs"], [S.EULER3D] * n,
                                   [[0.0] * 6] * n, st["centres"])
    return dict(params=np.stack(params), ms_value=np.array([r.value for r in res[0::2]]),
                mattes_value=np.array([r.value for r in res[1::2]]))


# ------------------------------------------------------------- work, tolerance
def _evaluation_work(samples, voxels):
    # a sample's stored index and bin or value; the moving voxels that the
    # samples reach, each once (eight corners of four bytes at most)
    return dict(bytes=5 * samples + min(4 * voxels, 32 * samples), flops=150 * samples)


def _cnn_work(case):
    # multiply-adds of the five convolutions (output positions x 27 x in x out)
    macs = 27 * (64 ** 3 * 2 * 16 + 32 ** 3 * 16 * 32 + 16 ** 3 * 32 * 64 + 8 ** 3 * 64 * 64 +
                 4 ** 3 * 64 * 128)
    pixels = sum(math.prod(s) for s in _ragged(case, case["n"]))
    flops = 2 * macs * case["n"]
    return dict(bytes=8 * pixels + 4 * 390_000, flops=3 * flops if case["train"] else flops)


def work(case):
    op = case["op"]
    if op in ("mattes", "ms"):
        v = case["nx"] * case["ny"] * case["nz"]
        return _evaluation_work(int(v * case["percent"] / 100.0), v)
    if op == "smooth":
        v = sum(math.prod(s) for s in _smooth_sizes(case))
        return dict(bytes=8 * v, flops=96 * v)
    if op == "bspline":
        v = case["edge"] ** 3
        n = int(v * case["percent"] / 100.0)
        return dict(bytes=5 * n + min(4 * v, 32 * n) + 48 * case["starts"] * (case["mesh"] + 3) ** 3,
                    flops=900 * n * case["starts"])
    if op == "cnn":
        return _cnn_work(case)
    b = f = 0
    for i, s in enumerate(_ragged(case, case["n"])):
        v = math.prod(s)
        e = _evaluation_work(int(v * (case["percent"] / 100.0 if i % 2 else 1.0)), v)
        # a registration: both volumes smoothed once, then its evaluations, on
        # the fine level and on an eighth of its samples
        reps = 1 if op == "batch" else case["iterations"] * 1.125
        b += e["bytes"] * reps + (0 if op == "batch" else 16 * v)
        f += e["flops"] * reps + (0 if op == "batch" else 192 * v)
    return dict(bytes=int(b), flops=int(f))


def tolerance(case):
    """About four times the largest error against `exact` that draws of each path show."""
    op = case["op"]
    if op == "smooth":
        return "exact"  # the recursion's 64-bit operation order is part of the interface
    if op in ("mattes", "ms"):
        # FP64: the histogram's 2^-32 units; FP32: weights and gradients rounded to float
        return {"rel": 8e-10, "max": 1e-9} if case["f64"] else {"rel": 8e-7, "max": 2e-6}
    if op == "batch":
        return {"rel": 2e-7, "max": 5e-7}
    if op == "bspline":
        return {"rel": 2.5e-7, "max": 4e-6}
    if op == "register":
        # FP32 against FP64 arithmetic along the whole path moves parameters by 1e-4
        return {"rel": 4e-4, "max": 4e-3}
    # bf16 activations; gradients cross ReLUs whose sign a rounding decides
    return {"rel": 3e-2, "max": 9e-1} if case["train"] else {"rel": 1e-2, "max": 3e-2}


# ----------------------------------------------- the same in 64 bits, plain torch
def _b3(u):
    a = u.abs()
    return torch.where(a < 1, (4 - 6 * a * a + 3 * a ** 3) / 6,
                       torch.where(a < 2, (2 - a) ** 3 / 6, torch.zeros_like(a)))


def _b3_deriv(u):
    a = u.abs()
    d = torch.where(a < 1, -2 * a + 1.5 * a * a,
                    torch.where(a < 2, -0.5 * (2 - a) ** 2, torch.zeros_like(a)))
    return torch.sign(u) * d


class _Exact:
    """The sampled metric of a pair in 64 bits."""

    def __init__(self, pair, idx, masks=None):
        nx, ny, nz = pair.size
        flat = torch.arange(nx * ny * nz, device=DEV) if idx is None else idx.to(DEV)
        if masks is not None:
            flat = flat[masks[0].to(DEV).reshape(-1)[flat]]
        self.pair, self.flat = pair, flat
        self.f = pair.fixed.reshape(-1)[flat].double()
        self.sp = torch.tensor(pair.spacing, device=DEV, dtype=torch.float64)
        self.org = torch.tensor(pair.origin, device=DEV, dtype=torch.float64)
        ijk = torch.stack([flat % nx, flat // nx % ny, flat // (nx * ny)], 1)
        self.x = self.org + ijk.double() * self.sp
        self.mmask = None if masks is None else masks[1].to(DEV).reshape(-1)

    def sample(self, y):
        """(valid, value, physical gradient) of the moving volume at y."""
        p = self.pair
        c = (y - self.org) / self.sp
        n = torch.tensor(p.size, device=DEV)
        ok = ((c >= -0.5) & (c < n - 0.5)).all(1)
        if self.mmask is not None:
            r = torch.floor(c + 0.5).long()
            r = torch.minimum(r.clamp(min=0), n - 1)
            ok &= self.mmask[r[:, 0] + p.size[0] * (r[:, 1] + p.size[1] * r[:, 2])]
        base = torch.floor(c)
        fr = c - base
        lo = torch.minimum(base.long().clamp(min=0), n - 1)
        hi = torch.minimum((base.long() + 1).clamp(min=0), n - 1)
        vol = p.moving.reshape(-1)
        value = torch.zeros(len(c), device=DEV, dtype=torch.float64)
        grad = torch.zeros(len(c), 3, device=DEV, dtype=torch.float64)
        for k in range(8):
            i = [hi[:, d] if k >> d & 1 else lo[:, d] for d in range(3)]
            w = [fr[:, d] if k >> d & 1 else 1 - fr[:, d] for d in range(3)]
            v = vol[i[0] + p.size[0] * (i[1] + p.size[1] * i[2])].double()
            value += w[0] * w[1] * w[2] * v
            for d in range(3):
                a, b = (w[e] for e in range(3) if e != d)
                grad[:, d] += (1.0 if k >> d & 1 else -1.0) * a * b * v
        return ok, value, grad / self.sp

    def map(self, stage, x=None):
        m = torch.as_tensor(stage, device=DEV, dtype=torch.float64)
        return (self.x if x is None else x) @ m[:9].reshape(3, 3).T + m[9:]

    def mean_squares(self, stage):
        ok, v, g = self.sample(self.map(stage))
        d = (v - self.f) * ok
        dg = d[:, None] * g
        return torch.cat([(d * d).sum()[None], dg.sum(0), (dg.T @ self.x).reshape(9),
                          ok.sum().double()[None]])

    def mattes(self, y, bins):
        """(-MI, the per-sample weight of the moving gradient, that gradient)."""
        m = self.pair.moving.reshape(-1)
        if self.mmask is not None:
            m = m[self.mmask]
        lo, hi = m.min().double(), m.max().double()
        step = (hi - lo) / (bins - 4)
        flo, fstep = self.f.min(), (self.f.max() - self.f.min()) / (bins - 4)
        fb = ((self.f - flo) / fstep + 2).long().clamp(2, bins - 3)
        ok, v, g = self.sample(y)
        ok &= (v >= lo) & (v <= hi)
        term = (v - lo) / step + 2
        first = term.long().clamp(2, bins - 3) - 1
        arg = [(first + k).double() - term for k in range(4)]
        joint = torch.zeros(bins * bins, device=DEV, dtype=torch.float64)
        for k in range(4):
            joint += torch.bincount(fb * bins + first + k, weights=_b3(arg[k]) * ok,
                                    minlength=bins * bins)
        joint = joint.reshape(bins, bins)
        count = torch.bincount(fb, weights=ok.double(), minlength=bins)
        total = joint.sum()
        p, pf = joint / total, count / total
        pm = p.sum(0)
        eps = np.finfo(np.float64).eps
        use = (p > eps) & (pf > eps)[:, None] & (pm > eps)[None]
        one = torch.ones_like(p)
        ratio = torch.log(torch.where(use, p / pm.clamp(min=eps), one))
        logf = torch.where(pf > eps, pf, torch.ones_like(pf)).log()
        value = -(torch.where(use, p, 0 * p) * (ratio - logf[:, None])).sum()
        ratio = (torch.where(use, ratio, 0 * p) / (step * ok.sum())).reshape(-1)
        w = sum(ratio[fb * bins + first + k] * _b3_deriv(arg[k]) for k in range(4)) * ok
        return float(value), w, g, int(ok.sum())

    def mattes_moments(self, stage, bins):
        value, w, g, valid = self.mattes(self.map(stage), bins)
        wg = w[:, None] * g
        return value, torch.cat([wg.sum(0), (wg.T @ self.x).reshape(9)]), valid


def _exact_bspline(case, x):
    e = _Exact(x["pair"], x["idx"])
    mesh, gsp = case["mesh"], case["edge"] / case["mesh"]
    gs = mesh + 3
    # a fixed point's support does not depend on the start: group the samples
    # by support cell once
    c = (e.x - (e.org - gsp)) / gsp
    inside = ((c >= 1) & (c < gs - 2)).all(1)
    first = torch.floor(c - 1).clamp(0, mesh - 1)
    cell = (first[:, 0] + mesh * (first[:, 1] + mesh * first[:, 2])).long()
    order = torch.argsort(torch.where(inside, cell, mesh ** 3))
    e.x, e.f, e.flat = e.x[order], e.f[order], e.flat[order]
    c, first, inside, cell = c[order], first[order], inside[order], cell[order]
    u = c - first
    w = [torch.stack([_b3(u[:, d] - k) for k in range(4)], 1) for d in range(3)]
    w = (w[2][:, :, None, None] * w[1][:, None, :, None] * w[0][:, None, None, :]).reshape(-1, 64)
    w = w * inside[:, None]
    i = torch.arange(4, device=DEV)
    tap = (i[None, None, :] + gs * (i[None, :, None] + gs * i[:, None, None])).reshape(1, 64)
    start = (first[:, 0] + gs * (first[:, 1] + gs * first[:, 2])).long()
    bounds = torch.searchsorted(torch.where(inside, cell, mesh ** 3),
                                torch.arange(mesh ** 3 + 1, device=DEV)).tolist()
    out = dict(value=[], deriv=[], valid=None)
    for coef, stage in zip(x["coef"].to(DEV), x["stages"]):
        coef = coef.reshape(3, -1)
        disp = torch.stack([(w * coef[d][start[:, None] + tap]).sum(1) for d in range(3)], 1)
        value, a, g, _ = e.mattes(e.map(stage, e.x + disp), case["bins"])
        g = a[:, None] * (g @ stage[:9].reshape(3, 3).to(DEV))
        deriv = torch.zeros(3, gs ** 3, device=DEV, dtype=torch.float64)
        for lo, hi in zip(bounds[:-1], bounds[1:]):
            if hi > lo:
                deriv.index_add_(1, start[lo] + tap[0], g[lo:hi].T.contiguous() @ w[lo:hi])
        out["value"].append(value)
        out["deriv"].append(deriv.reshape(-1).cpu().numpy())
    if case["starts"] == 1:
        return dict(value=np.float64(out["value"][0]), deriv=out["deriv"][0], valid=None)
    return dict(value=np.array(out["value"]), deriv=np.stack(out["deriv"]), valid=None)


def _deriche(sigma):
    """Farneback & Westin's fourth-order recursive approximation of the Gaussian
    with unit gain: numerators n, m and denominator d of the two passes."""
    a1, a2, b1, b2 = 1.3530, -0.3531, 1.8151, 0.0902
    w1, l1, w2, l2 = 0.6681 / sigma, -1.3932 / sigma, 2.0787 / sigma, -1.3732 / sigma
    c1, s1, c2, s2 = math.cos(w1), math.sin(w1), math.cos(w2), math.sin(w2)
    e1, e2 = math.exp(l1), math.exp(l2)
    d = [-2 * (e2 * c2 + e1 * c1), 4 * c2 * c1 * e1 * e2 + e1 * e1 + e2 * e2,
         -2 * c1 * e1 * e2 * e2 - 2 * c2 * e2 * e1 * e1, e1 * e1 * e2 * e2]
    n = [a1 + a2,
         e2 * (b2 * s2 - (a2 + 2 * a1) * c2) + e1 * (b1 * s1 - (a1 + 2 * a2) * c1),
         2 * e1 * e2 * ((a1 + a2) * c2 * c1 - b1 * c2 * s1 - b2 * c1 * s2) + a2 * e1 * e1 +
         a1 * e2 * e2,
         e2 * e1 * e1 * (b2 * s2 - a2 * c2) + e1 * e2 * e2 * (b1 * s1 - a1 * c1)]
    alpha = 2 * sum(n) / (1 + sum(d)) - n[0]
    n = [v / alpha for v in n]
    m = [n[1] - d[0] * n[0], n[2] - d[1] * n[0], n[3] - d[2] * n[0], -d[3] * n[0]]
    return n, m, d


def _exact_smooth(v, sigmas):
    v = v.double()
    for axis, sigma in zip((2, 1, 0), sigmas):
        n, m, d = _deriche(sigma)
        x = v.movedim(axis, 0).contiguous()
        total = torch.zeros_like(x)
        gain = 1 + sum(d)
        for coef, rows, lag in ((n, range(len(x)), 0), (m, range(len(x) - 1, -1, -1), 1)):
            # before the line begins it is taken to be constant
            edge = x[rows[0]]
            past = [edge] * 4
            old = [edge * (sum(coef) / gain)] * 4
            for k in rows:
                taps = [x[k]] + past[:3] if lag == 0 else past
                y = sum(c * t for c, t in zip(coef, taps)) - sum(c * t for c, t in zip(d, old))
                total[k] += y
                past, old = [x[k]] + past[:3], [y] + old[:3]
        v = total.movedim(0, axis)
    return v.contiguous()


_CHANNELS = (8, 16, 32, 64, 64, 128)


def _cnn_params(gen):
    """He-initialised weights in the network's flat layout (conv W[co][27][ci]
    and bias per layer, the two head layers); 2 of the 8 input channels used."""
    out = []
    for ci, co in zip(_CHANNELS[:-1], _CHANNELS[1:]):
        used = 2 if ci == 8 else ci
        w = torch.zeros(co, 27, ci)
        w[:, :, :used] = torch.randn(co, 27, used, generator=gen) * math.sqrt(2 / (27 * used))
        out += [w.reshape(-1), 0.05 * torch.randn(co, generator=gen)]
    out += [torch.randn(128 * 128, generator=gen) * math.sqrt(2 / 128), torch.zeros(128),
            torch.randn(12 * 128, generator=gen) * 0.1 * math.sqrt(1 / 128), torch.zeros(12)]
    return torch.cat(out)


def _to_64(v):
    """Linear resampling of a volume onto 64 blocks per axis, then z-scored."""
    v = v.double()
    for axis in range(3):
        n = v.shape[axis]
        c = ((torch.arange(64, device=DEV, dtype=torch.float64) + 0.5) * n / 64 - 0.5).clamp(0, n - 1)
        lo = torch.floor(c).long()
        hi = (lo + 1).clamp(max=n - 1)
        f = (c - lo).reshape([-1 if d == axis else 1 for d in range(3)])
        v = v.index_select(axis, lo) * (1 - f) + v.index_select(axis, hi) * f
    return (v - v.mean()) / v.std(unbiased=False)


def _exact_cnn(case, x):
    p = x["params"].double().to(DEV).requires_grad_(case["train"])
    a = torch.stack([torch.stack([_to_64(q.fixed), _to_64(q.moving)], -1) for q in x["pairs"]])
    at = 0

    def take(*shape):
        nonlocal at
        v = p[at:at + math.prod(shape)].reshape(shape)
        at += math.prod(shape)
        return v

    for layer, (ci, co) in enumerate(zip(_CHANNELS[:-1], _CHANNELS[1:])):
        w, b = take(co, 27, ci), take(co)
        if layer == 0:
            w = w[:, :, :2]
        step = 1 if layer == 0 else 2
        edge = a.shape[1] // step
        padded = torch.nn.functional.pad(a, (0, 0, 1, 1, 1, 1, 1, 1))
        y = b.expand(case["n"], edge, edge, edge, co)
        for tap in range(27):
            k = (tap // 9, tap // 3 % 3, tap % 3)
            s = [slice(q, q + step * (edge - 1) + 1, step) for q in k]
            part = padded[:, s[0], s[1], s[2]].reshape(-1, w.shape[2])
            y = y + (part @ w[:, tap].T.contiguous()).reshape(y.shape)
        a = torch.relu(y)
    feat = a.mean((1, 2, 3))
    w, b = take(128, 128), take(128)
    hidden = torch.relu(feat @ w.T.contiguous() + b)
    w, b = take(12, 128), take(12)
    out = hidden @ w.T.contiguous() + b
    if not case["train"]:
        return dict(out=out.cpu().numpy())
    loss = ((out - x["targets"].double().to(DEV)) ** 2).mean()
    loss.backward()
    return dict(loss=float(loss.detach()), grads=p.grad.cpu().numpy())


def exact(case, seed):
    op = case["op"]
    if op == "register":
        return None  # an optimizer's whole path has no closed form to state it by
    x = _inputs(case, seed)
    if op == "mattes":
        e = _Exact(x["pair"], x["idx"], x["masks"])
        value, moments, _ = e.mattes_moments(x["pair"].stage, case["bins"])
        return dict(value=np.float64(value), moments=moments.cpu().numpy(), valid=None)
    if op == "ms":
        e = _Exact(x["pair"], x["idx"], x["masks"])
        return dict(moments=e.mean_squares(x["pair"].stage).cpu().numpy())
    if op == "smooth":
        return [_exact_smooth(p.fixed, [case["sigma"] / s for s in x["spacing"]])
                for p in x["pairs"]]
    if op == "batch":
        ms, mv, mm = [], [], []
        for i, (p, idx) in enumerate(zip(x["pairs"], x["idx"])):
            e = _Exact(p, idx)
            if i % 2 == 0:
                ms.append(e.mean_squares(p.stage).cpu().numpy())
            else:
                value, moments, _ = e.mattes_moments(p.stage, case["bins"])
                mv.append(value)
                mm.append(np.concatenate([moments.cpu().numpy(), np.zeros(2)]))
        ms = np.stack(ms)
        return dict(ms_value=ms[:, 0] / ms[:, 13], ms_moments=ms, mattes_value=np.array(mv),
                    mattes_moments=np.stack(mm), valid=None)
    if op == "bspline":
        return _exact_bspline(case, x)
    return _exact_cnn(case, x)
