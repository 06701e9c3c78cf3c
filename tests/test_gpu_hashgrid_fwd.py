"""The hash-grid forward over its launch rules against a float64 restatement:
level counts that do not pair up evenly, small tables (every level hashed or
dense), sizes on both sides of the rule that gives each XCD its levels, part-filled
workgroups, and positions on and beyond the box's faces, whose dense cells wrap
around the level. The bar per feature is 4e-7 of the sum of |weight * entry|
(products of four and sums of eight fp32 numbers, 2^-24 each), 1e-3 of it for
fp16 features (2^-11 for the feature itself), and half of fp16's smallest
step."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _reference(g, pos, table):
    """(features, sum of |weight * entry|) [2L][n] in float64 from the fp32 positions."""
    out, bar = [], []
    t = table.astype(np.float64).reshape(-1, 2)
    for l in range(g.n_levels):
        s, r, size, off = np.float32(g.scale[l]), g.resolution[l], g.level_size[l], g.level_offset[l]
        x = (pos * s + np.float32(0.5)).astype(np.float32)
        c = np.floor(x)
        f = (x - c).astype(np.float64)
        c = c.astype(np.int64)
        acc, mag = np.zeros((2, pos.shape[1])), np.zeros((2, pos.shape[1]))
        for k in range(8):
            q = [(c[a] + ((k >> a) & 1)) & 0xFFFFFFFF for a in range(3)]
            if g.level_dense[l]:
                idx = ((q[0] + q[1] * r + q[2] * r * r) & 0xFFFFFFFF) % size
            else:
                idx = (q[0] ^ ((q[1] * 2654435761) & 0xFFFFFFFF) ^ ((q[2] * 805459861) & 0xFFFFFFFF)) & (size - 1)
            w = np.prod([f[a] if (k >> a) & 1 else 1 - f[a] for a in range(3)], axis=0)
            v = w * t[off + idx].T
            acc += v
            mag += np.abs(v)
        out.append(acc)
        bar.append(mag)
    return np.concatenate(out), np.concatenate(bar)


@pytest.mark.parametrize("n", [1, 63, 257, 131072, 131073])
@pytest.mark.parametrize("levels,log2_T", [(16, 19), (16, 12), (1, 14), (7, 16)])
def test_forward_launch_rules(cuda, n, levels, log2_T):
    import torch

    from turbonerf_amd import ops

    g = ops.hashgrid_layout(n_levels=levels, log2_T=log2_T, per_level_scale=1.38)
    rng = np.random.default_rng(n + levels)
    pos = rng.uniform(0, 1, (3, n)).astype(np.float32)
    edge = rng.random((3, n))
    pos[edge < 0.05] = 0.0
    pos[edge > 0.95] = 1.0
    pos[(edge > 0.47) & (edge < 0.48)] = 1.3
    pos[(edge > 0.48) & (edge < 0.49)] = -0.2
    table = rng.uniform(-1, 1, g.n_params).astype(np.float16)
    print(f"[hashgrid fwd] n {n} levels {levels} log2_T {log2_T}", flush=True)
    p = torch.from_numpy(pos.ravel()).cuda()
    ref, mag = _reference(g, pos, table)
    for tdt, fdt, rel in ((np.float32, torch.float32, 4e-7), (np.float16, torch.float32, 4e-7),
                          (np.float16, torch.float16, 1e-3)):
        t = torch.from_numpy(table.astype(tdt)).cuda()
        out = ops.hashgrid_forward(g, n, p, n, t, feat_dtype=fdt).float().cpu().numpy().reshape(2 * levels, n)
        assert np.all(np.abs(out - ref) <= rel * mag + 6e-8), np.abs(out - ref).max()
