"""The marching kernels over their group sizes (16 lanes per ray up to 24,576
rays, 8 above) bit for bit against the oracle: part-filled waves, rays along
axes, on cell faces and with zero and negative-zero components, sparse, full
and empty grids, one and several cascades, a resolution that is no power of
two and a box larger than the grid's cascades."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DT_MIN = math.sqrt(3.0) / 1024.0
CONE = 1.0 / 256.0


def _rays(rng, n, aabb):
    """Rays from inside and around the box: random ones, then rays along the
    axes (the other components +0 or -0), starting on cell faces."""
    d = rng.normal(size=(3, n))
    o = rng.uniform(-0.6, 0.6, (3, n)) * aabb
    special = np.arange(n) % 4 == 1
    axis = rng.integers(0, 3, n)
    for a in range(3):
        zero = np.where(rng.random(n) < 0.5, 0.0, -0.0)
        d[a] = np.where(special, np.where(axis == a, rng.choice([-1.0, 1.0], n), zero), d[a])
        o[a] = np.where(special, np.round(o[a] * 64) / 64, o[a])
    d /= np.linalg.norm(d, axis=0)
    return o.astype(np.float32), d.astype(np.float32)


@pytest.mark.parametrize("n_rays", [1, 3, 4, 61, 24576, 24577])
@pytest.mark.parametrize("aabb,levels,res,fill", [(1.0, 1, 128, 0.05), (1.0, 1, 128, 1.0), (1.0, 1, 100, 0.3),
                                                  (4.0, 3, 128, 0.02), (3.0, 2, 64, 0.2), (16.0, 5, 32, 0.0)])
def test_march_groups_match_oracle(cuda, n_rays, aabb, levels, res, fill):
    import torch

    import oracle
    from turbonerf_amd import ops, scenes

    if n_rays > 1000 and (fill == 1.0 or res == 32):
        n_rays //= 8  # enough for the groups of 16; the large counts are covered by the other grids
    print(f"[march groups] rays {n_rays} aabb {aabb} levels {levels} res {res} fill {fill}", flush=True)
    rng = np.random.default_rng(n_rays + levels)
    vol = res ** 3 if res & (res - 1) == 0 else 128 ** 3  # Morton codes of a resolution that is no power of two
    bits = np.zeros(vol, np.uint8)
    for l in range(levels):
        bits |= ((rng.random(vol) < fill).astype(np.uint8) << l).astype(np.uint8)
    o, d = _rays(rng, n_rays, aabb)
    t = rng.uniform(0.0, 0.1, n_rays).astype(np.float32)
    tmax = rng.uniform(0.0, 2.0 * aabb, n_rays).astype(np.float32)
    alive = (rng.random(n_rays) < 0.9).astype(np.uint8)
    rays = ops.Rays.empty(n_rays)
    T = lambda a: torch.from_numpy(np.ascontiguousarray(a).ravel()).cuda()
    rays.ori, rays.dir, rays.t, rays.tmax, rays.alive = T(o), T(d), T(t), T(tmax), T(alive)
    rr = dict(ori=o.ravel(), dir=d.ravel(), t=t, tmax=tmax, alive=alive.copy(),
              img_id=np.arange(n_rays, dtype=np.uint32))
    rays.img_id = T(rr["img_id"].view(np.int32))
    bits_d = T(bits)
    grid = ops.grid_struct(bits_d, None, levels, res)
    box = scenes.bbox(aabb)
    dt_max = aabb * DT_MIN
    for max_steps in (0xFFFFFFFF, 37):
        rays.alive = T(alive)
        ops.march_count(rays, n_rays, box, grid, CONE, DT_MIN, dt_max, max_steps)
        rr["alive"] = alive.copy()
        n_ref, alive_ref = oracle.march_count(n_rays, n_rays, box, bits, levels, res, CONE, DT_MIN, dt_max, rr,
                                              max_steps)
        n_gpu = rays.n_steps.cpu().numpy().view(np.uint32)
        assert np.array_equal(n_gpu, n_ref)
        assert np.array_equal(rays.alive.cpu().numpy(), alive_ref)
        ns = int(n_ref.sum())
        if ns == 0:
            continue
        cap = ns + 7
        info = torch.zeros(4, dtype=torch.int32, device="cuda")
        ops.scan_select(rays, n_rays, cap, info, mode=1)
        smp = ops.Samples.empty(cap)
        ops.march_generate(rays, smp, n_rays, info, box, 1.0 / aabb, grid, DT_MIN, dt_max, CONE)
        excl = np.concatenate([[0], np.cumsum(n_ref)[:-1]]).astype(np.uint32)
        so = oracle.march_generate(n_rays, n_rays, cap, box, 1.0 / aabb, bits, levels, res, DT_MIN, dt_max, CONE, rr,
                                   excl, alive_ref, n_ref)
        assert np.array_equal(smp.t[:ns].cpu().numpy().view(np.uint32), so["t"][:ns].view(np.uint32))
        assert np.array_equal(smp.img_id[:ns].cpu().numpy().view(np.uint32), so["img_id"][:ns])
        g = smp.pos.cpu().numpy().reshape(3, cap)[:, :ns]
        assert np.array_equal(g.view(np.uint32), so["pos"].reshape(3, cap)[:, :ns].view(np.uint32))


@pytest.mark.parametrize("n_rays", [61, 24577])
@pytest.mark.parametrize("levels,fill", [(1, 1.0), (1, 0.3), (3, 0.2)])
def test_generate_with_dt_max_below_dt_min(cuda, n_rays, levels, fill):
    """tn_march_generate takes steps whose upper bound lies below the lower
    one (tn_march_count refuses them): every step is then the upper bound, in t
    and in dt, wherever t times the cone angle lies. Bit for bit against the
    oracle, the counts from the oracle as well."""
    import torch

    import oracle
    from turbonerf_amd import ops, scenes

    print(f"[march dt_max < dt_min] rays {n_rays} levels {levels} fill {fill}", flush=True)
    rng = np.random.default_rng(n_rays + levels)
    aabb, res, dt_min, dt_max, cone = float(1 << (levels - 1)), 64, 0.02, 0.01, 0.05
    bits = np.zeros(res ** 3, np.uint8)
    for l in range(levels):
        bits |= ((rng.random(res ** 3) < fill).astype(np.uint8) << l).astype(np.uint8)
    o, d = _rays(rng, n_rays, aabb)
    t = rng.uniform(0.0, 0.1, n_rays).astype(np.float32)
    tmax = rng.uniform(0.0, 2.0 * aabb, n_rays).astype(np.float32)
    box = scenes.bbox(aabb)
    rr = dict(ori=o.ravel(), dir=d.ravel(), t=t, tmax=tmax, alive=np.ones(n_rays, np.uint8),
              img_id=np.arange(n_rays, dtype=np.uint32))
    n_ref, alive_ref = oracle.march_count(n_rays, n_rays, box, bits, levels, res, cone, dt_min, dt_max, rr, 0xFFFFFFFF)
    excl = np.concatenate([[0], np.cumsum(n_ref)[:-1]]).astype(np.uint32)
    ns = int(n_ref.sum())
    assert ns > n_rays
    so = oracle.march_generate(n_rays, n_rays, ns, box, 1.0 / aabb, bits, levels, res, dt_min, dt_max, cone, rr, excl,
                               alive_ref, n_ref)
    T = lambda a: torch.from_numpy(np.ascontiguousarray(a).ravel()).cuda()
    rays = ops.Rays.empty(n_rays)
    rays.ori, rays.dir, rays.t, rays.tmax, rays.alive = T(o), T(d), T(t), T(tmax), T(alive_ref)
    rays.img_id, rays.n_steps, rays.offset = (T(a.view(np.int32)) for a in (rr["img_id"], n_ref, excl))
    smp = ops.Samples.empty(ns)
    ops.march_generate(rays, smp, n_rays, ops.batch_info(n_rays, ns), box, 1.0 / aabb,
                       ops.grid_struct(T(bits), None, levels, res), dt_min, dt_max, cone)
    words = lambda x: np.asarray(x).view(np.uint32)
    assert np.array_equal(words(smp.t.cpu().numpy()), words(so["t"]))
    assert np.array_equal(words(smp.dt.cpu().numpy()), words(so["dt"]))
    assert np.array_equal(words(smp.pos.cpu().numpy()), words(so["pos"]))
