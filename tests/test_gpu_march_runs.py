"""tn_march_count_runs and tn_march_generate_runs equal tn_march_count and
tn_march_generate bit for bit: rays of none, one, up to 15 (the records that a
ray has) and more runs of samples, runs of more than 16 samples, capped rays,
a sample budget that drops rays, constant and growing steps, and the outputs
that a render leaves out."""
import pytest

from test_gpu_march_groups import CONE, DT_MIN, _rays

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_rays", [1, 61, 5000, 24577])
@pytest.mark.parametrize("aabb,levels,res,fill", [(1.0, 1, 128, 0.05), (1.0, 1, 128, 0.5), (1.0, 1, 64, 1.0),
                                                  (4.0, 3, 128, 0.02), (3.0, 2, 64, 0.2), (2.0, 2, 32, 0.0)])
def test_march_runs(cuda, n_rays, aabb, levels, res, fill):
    import numpy as np
    import torch

    from turbonerf_amd import ops, scenes
    from turbonerf_amd._capi import call, ptr, query, stream_ptr

    print(f"[march runs] rays {n_rays} aabb {aabb} levels {levels} res {res} fill {fill}", flush=True)
    rng = np.random.default_rng(n_rays + levels)
    bits = np.zeros(res ** 3, np.uint8)
    for l in range(levels):
        bits |= ((rng.random(res ** 3) < fill).astype(np.uint8) << l).astype(np.uint8)
    o, d = _rays(rng, n_rays, aabb)
    T = lambda a: torch.from_numpy(np.ascontiguousarray(a).ravel()).cuda()
    bits_d = T(bits)
    grid, box = ops.grid_struct(bits_d, None, levels, res), scenes.bbox(aabb)
    rays = ops.Rays.empty(n_rays)
    rays.ori, rays.dir = T(o), T(d)
    rays.t, rays.tmax = T(rng.uniform(0.0, 0.1, n_rays).astype(np.float32)), T(
        rng.uniform(0.0, 2.0 * aabb, n_rays).astype(np.float32))
    rays.img_id = torch.arange(n_rays, dtype=torch.int32, device="cuda") + 3
    alive = T((rng.random(n_rays) < 0.9).astype(np.uint8))
    nb = query("tn_march_runs_bytes", n_rays)
    assert nb == 128 * n_rays
    for max_steps, dt_max, budget in ((0xFFFFFFFF, aabb * DT_MIN, 1.0), (37, aabb * DT_MIN, 0.6),
                                      (0xFFFFFFFF, DT_MIN, 1.0)):
        rays.alive = alive.clone()
        ops.march_count(rays, n_rays, box, grid, CONE, DT_MIN, dt_max, max_steps)
        n_ref, alive_ref = rays.n_steps.clone(), rays.alive.clone()
        rays.alive = alive.clone()
        rays.n_steps = torch.full_like(n_ref, -1)
        runs = torch.full((nb,), 0xA5, dtype=torch.uint8, device="cuda")
        call("tn_march_count_runs", n_rays, None, n_rays, box, grid, CONE, DT_MIN, dt_max, max_steps, ptr(rays.dir),
             ptr(rays.tmax), ptr(rays.alive), ptr(rays.ori), ptr(rays.t), ptr(rays.n_steps), ptr(runs), nb,
             stream_ptr())
        assert torch.equal(rays.n_steps, n_ref) and torch.equal(rays.alive, alive_ref)
        cap = max(1, int(int(n_ref.sum().item()) * budget))
        info = torch.zeros(4, dtype=torch.int32, device="cuda")
        ops.scan_select(rays, n_rays, cap, info, mode=0 if budget < 1.0 else 1)
        ref, out, few = (ops.Samples.empty(cap) for _ in range(3))
        ops.march_generate(rays, ref, n_rays, info, box, 1.0 / aabb, grid, DT_MIN, dt_max, CONE)
        for s, opt in ((out, True), (few, False)):
            call("tn_march_generate_runs", n_rays, ptr(info), n_rays, cap, box, 1.0 / aabb, grid, DT_MIN, dt_max, CONE,
                 ptr(rays.img_id) if opt else None, ptr(rays.ori), ptr(rays.dir), ptr(rays.t), ptr(rays.offset),
                 ptr(rays.alive), ptr(rays.n_steps), ptr(runs), nb, ptr(s.img_id) if opt else None,
                 ptr(s.t) if opt else None, ptr(s.pos), ptr(s.dir), ptr(s.dt), ptr(s.m_norm) if opt else None,
                 ptr(s.dt_norm) if opt else None, stream_ptr())
        n = int(info[1].item())
        most = int(runs.view(torch.int32).view(n_rays, 32)[:, 0][alive_ref != 0].max().item()) if n else 0
        print(f"  samples {n}, most runs {most}", flush=True)
        if fill == 0.5 and n_rays > 1 and budget == 1.0:
            assert most > 15  # rays of more runs than records
        words = lambda x: x.view(torch.int32).view(-1, cap)[:, :n]
        for k in ("img_id", "t", "pos", "dir", "dt", "m_norm", "dt_norm"):
            assert torch.equal(words(getattr(ref, k)), words(getattr(out, k))), k
        for k in ("pos", "dir", "dt"):
            assert torch.equal(words(getattr(ref, k)), words(getattr(few, k))), k
