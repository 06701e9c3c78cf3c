"""Forward-only compositing against a float64 evaluation of the reference's
loop: rays of none, one, and a block of 16 samples and its neighbours, long
rays, opaque ones that stop early, network outputs and plain sigmas, fp16,
fp32 and float64 sums, more rays than one pass of the grid takes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_rays", [1, 3, 700, 70_001])
@pytest.mark.parametrize("dtype,fp64,raw", [("float16", False, True), ("float32", False, True),
                                            ("float32", False, False), ("float32", True, True)])
def test_composite_forward(cuda, n_rays, dtype, fp64, raw):
    import torch

    from turbonerf_amd import ops

    print(f"[composite forward] rays {n_rays} {dtype} fp64 {fp64} raw {raw}", flush=True)
    rng = np.random.default_rng(n_rays)
    lengths = np.array([0, 1, 15, 16, 17, 31, 33, 64, 65, 500])
    steps = rng.choice(lengths, n_rays, p=[0.3] + [0.085] * 8 + [0.02]) if n_rays > 3 else lengths[[9, 0, 4]][:n_rays]
    offs = np.concatenate([[0], np.cumsum(steps)[:-1]])
    n = int(steps.sum())
    ray = np.repeat(np.arange(n_rays), steps)
    opaque = rng.random(n_rays) < 0.3
    level = np.where(opaque, 5.0, -1.0)[ray]
    s = (level + rng.normal(0, 1.5, n)).astype(dtype)
    if not raw:
        s = np.exp(np.minimum(s, 5)).astype(dtype)
    c = rng.random((3, n)).astype(dtype)
    dt = rng.uniform(1e-3, 8e-3, n).astype(np.float32)
    T = lambda a: torch.from_numpy(np.ascontiguousarray(a).ravel()).cuda()
    info = torch.tensor([n_rays, n, 0, 0], dtype=torch.int32, device="cuda")
    got = ops.composite_forward(info, n, n, n_rays, T(steps.astype(np.int32)), T(offs.astype(np.int32)), T(s), T(c), T(dt),
                                raw_density=raw, min_T=1e-4, fp64_accumulate=fp64).cpu().numpy().reshape(4, n_rays)
    # float64: the prefix of sigma dt per ray, weights up to the early stop
    sigma = np.exp(np.minimum(s.astype(np.float64), 12.0) - 1.0) if raw else s.astype(np.float64)
    tau = sigma * dt.astype(np.float64)
    P = np.cumsum(tau)
    start = np.concatenate([[0.0], P])[offs]
    Te = np.exp(-(P - tau - start[ray]))
    alpha = -np.expm1(-tau)
    w = np.where(Te >= 1e-4, Te * alpha, 0.0)
    wc = np.where(alpha > 1e-4, w, 0.0)
    ref = np.stack([np.bincount(ray, wc * c[k].astype(np.float64), n_rays) for k in range(3)] +
                   [np.bincount(ray, w, n_rays)])
    # sigma and T each carry a relative error of at most |x| 2^-23 in the
    # exponential's argument x (|x| <= 11 and 9.3), which tau adds up to
    # max x e^-x over a ray: under 2e-6; a sample within that of a threshold
    # may count or not and is worth at most 1e-4
    near = (np.abs(Te / 1e-4 - 1) < 1e-4) | (np.abs(alpha / 1e-4 - 1) < 1e-4)
    tol = 4e-6 + 1e-4 * np.bincount(ray, near, n_rays)
    err = np.abs(got - ref)
    print(f"  samples {n}, largest error {err.max():.2e}, near a threshold {int(near.sum())}", flush=True)
    assert (err <= tol[None]).all()
    assert (got[:, steps == 0] == 0).all()
