"""tn_training_rays and tn_batch_select, a training batch's rays and selection
in one launch each, equal the separate entry points bit for bit: stream
offsets of every alignment, the alpha rule on and off, ray counts below and
above one round of the selecting workgroup (16,384 rays), budgets that keep
all, some or none of the rays."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,capacity,offset,alpha", [(1, 64, 0, 1.0), (777, 1000, 5, 0.6), (20000, 20000, 1 << 33, 1.0)])
def test_training_rays(cuda, n, capacity, offset, alpha):
    import torch

    from turbonerf_amd import ops, scenes
    from turbonerf_amd._capi import call, ptr, stream_ptr

    print(f"[training rays] {n} of {capacity}, offset {offset}, alpha {alpha}", flush=True)
    seed, n_img, W = 91, 5, 24
    cams = torch.from_numpy(scenes.cameras_bytes(scenes.sphere_cameras(3, n_img, 2.0, W, W, 50.0))).cuda()
    images = torch.randint(0, 256, (n_img * W * W * 4,), dtype=torch.uint8, device="cuda",
                           generator=torch.Generator("cuda").manual_seed(1))
    box = ops.upload_struct(scenes.bbox(1.0))
    count = torch.tensor([n], dtype=torch.int32, device="cuda")
    off = torch.tensor([offset], dtype=torch.int64, device="cuda")
    a, b = ops.Rays.empty(capacity), ops.Rays.empty(capacity)
    rnd = ops.fill_uniform(4 * capacity, seed, offset)
    ops.init_training_rays(a, capacity, n_img, W, W, -1.0, box, cams, images, rnd, d_n_rays=count)
    prob = 0.5 if alpha < 1.0 else 1.0
    if alpha < 1.0:
        call("tn_deactivate_rays", capacity, ptr(count), capacity, alpha, prob, ptr(a.pix_rgba),
             ptr(rnd) + 4 * capacity, ptr(a.alive), stream_ptr())
    out = torch.zeros(4 * capacity, device="cuda")
    call("tn_training_rays", capacity, ptr(count), capacity, n_img, W * W, W, W, ptr(box), ptr(cams), ptr(images), seed,
         ptr(off), alpha, prob, ptr(out), ptr(b.pix_rgba), ptr(b.img_id), ptr(b.ori), ptr(b.dir), ptr(b.t),
         ptr(b.tmax), ptr(b.alive), stream_ptr())
    for k in ("pix_rgba", "img_id", "ori", "dir", "t", "tmax", "alive"):
        assert torch.equal(getattr(a, k), getattr(b, k)), k
    assert torch.equal(out.view(4, -1)[:, :n], rnd.view(4, -1)[:, :n])
    assert int(off.item()) == offset


@pytest.mark.parametrize("n", [1, 63, 1000, 16384, 16385, 50001])
@pytest.mark.parametrize("mean,budget", [(60, 1 << 18), (0.3, 1 << 12), (200, 100)])
def test_batch_select(cuda, n, mean, budget):
    import torch

    from turbonerf_amd import ops
    from turbonerf_amd._capi import call, ptr, stream_ptr

    rng = np.random.default_rng(n)
    cap = n + 37
    steps = np.zeros(cap, np.int32)
    steps[:n] = rng.poisson(mean, n)
    count = torch.tensor([n], dtype=torch.int32, device="cuda")
    a, b = ops.Rays.empty(cap), ops.Rays.empty(cap)
    a.n_steps = b.n_steps = torch.from_numpy(steps).cuda()
    ia, ib = (torch.zeros(4, dtype=torch.int32, device="cuda") for _ in range(2))
    ops.scan_select(a, cap, budget, ia, mode=0, d_n_rays=count)
    nxt = torch.zeros(1, dtype=torch.int32, device="cuda")
    call("tn_estimate_rays", ptr(ia), budget, cap, 64, ptr(nxt), stream_ptr())
    off = torch.tensor([7], dtype=torch.int64, device="cuda")
    call("tn_batch_select", cap, ptr(count), ptr(b.n_steps), budget, ptr(b.offset), ptr(ib), cap, 64, ptr(count),
         ptr(off), 4 * cap, stream_ptr())
    print(f"[batch select] rays {n} kept {ia.tolist()}", flush=True)
    assert ia.tolist() == ib.tolist()
    assert torch.equal(a.offset, b.offset)
    assert int(count.item()) == int(nxt.item()) and int(off.item()) == 7 + 4 * cap


@pytest.mark.parametrize("n,offset", [(1, 0), (5, 3), (4096, 1 << 33), (100_003, 6)])
def test_fill_uniform_dev(cuda, n, offset):
    """tn_fill_uniform_dev is tn_fill_uniform at the position kept on the
    device, which advances, call after call."""
    import torch

    from turbonerf_amd import ops
    from turbonerf_amd._capi import call, ptr, stream_ptr

    print(f"[fill uniform dev] n {n} offset {offset}", flush=True)
    off = torch.tensor([offset], dtype=torch.int64, device="cuda")
    for k in range(3):
        out = torch.full((n + 9,), -1.0, device="cuda")
        call("tn_fill_uniform_dev", n, 17, ptr(off), ptr(out), stream_ptr())
        assert torch.equal(out[:n], ops.fill_uniform(n, 17, offset + k * n)) and bool((out[n:] == -1.0).all())
        assert int(off.item()) == offset + (k + 1) * n
