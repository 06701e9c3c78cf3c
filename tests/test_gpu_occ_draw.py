"""tn_occ_draw_points and tn_occ_draw_update equal a uniform fill with
tn_occ_sample_points and tn_occ_update_density bit for bit: stream offsets,
strides, cell counts and starts that are and are not multiples of four, the
warm-up and the subset rule, both network precisions."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,stride,start", [(4096, 4096, 0), (4095, 4097, 1), (1, 1, 5), (1030, 2046, 4), (262144, 262144, 0)])
@pytest.mark.parametrize("offset", [0, 3, (1 << 34) + 2])
def test_occ_draw(cuda, n, stride, start, offset):
    import torch

    from turbonerf_amd import ops
    from turbonerf_amd._capi import call, ptr, stream_ptr

    print(f"[occ draw] cells {n} stride {stride} start {start} offset {offset}", flush=True)
    res, levels, level, seed = 64, 3, 2, (77 << 32) + 5
    vol = res ** 3
    gen = torch.Generator("cuda").manual_seed(n)
    bits = torch.randint(0, 8, (vol,), dtype=torch.uint8, device="cuda", generator=gen)
    before = torch.rand(levels * vol, device="cuda", generator=gen)
    rnd = ops.fill_uniform(4 * stride, seed, offset)
    a, b = torch.zeros(3 * stride, device="cuda"), torch.zeros(3 * stride, device="cuda")
    grid = ops.grid_struct(bits, before, levels, res)
    call("tn_occ_sample_points", n, stride, start, grid, level, 0.25, ptr(rnd), ptr(a), stream_ptr())
    call("tn_occ_draw_points", n, stride, start, grid, level, 0.25, seed, offset, ptr(b), stream_ptr())
    assert torch.equal(a, b)
    for code, dtype in ((0, torch.float32), (1, torch.float16)):
        raw = torch.randn(stride, device="cuda", generator=gen).to(dtype)
        for warm in (0, 1):
            da, db = before.clone(), before.clone()
            call("tn_occ_update_density", code, n, start, ops.grid_struct(bits, da, levels, res), level, warm,
                 ptr(rnd) + 12 * stride, ptr(raw), stream_ptr())
            call("tn_occ_draw_update", code, n, stride, start, ops.grid_struct(bits, db, levels, res), level, warm, seed,
                 offset, ptr(raw), stream_ptr())
            assert torch.equal(da, db)
