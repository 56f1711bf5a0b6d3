"""Kernels at the sizes where their tiling can go wrong: one workgroup's edge,
a remainder, the first size of another variant, the smallest and a large input.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def spot_reference(x, y, f, G):
    """n, centroid, variance and RMS radius per group, two passes in numpy"""
    out = np.zeros((G, 6))
    for g in range(G):
        m = f[g::G] == 1
        xs, ys = x[g::G][m], y[g::G][m]
        if xs.size:
            vx, vy = xs.var(), ys.var()
            out[g] = [xs.size, xs.mean(), ys.mean(), vx, vy, np.sqrt(vx + vy)]
    return out


# a workgroup covers 256 // G strides of the groups 8 times (2048 rays in one
# group); 257 groups take a second block of groups; above 2^21 rays a workgroup
# walks its chunk in two passes
@pytest.mark.parametrize("n,G", [(1, 1), (2047, 1), (2048, 1), (2049, 1), (2040, 5), (2041, 5), (7, 255), (4097, 256),
                                 (257 * 8 + 1, 257), (3000, 1000), ((1 << 21) - 1, 3), ((1 << 21) + 4095, 1)])
def test_group_spots_at_chunk_edges(hip, n, G):
    print(f"[group spots] n={n} groups={G}", flush=True)
    g = torch.Generator().manual_seed(n + G)
    rays = torch.zeros((7, n), dtype=torch.float64)
    rays[0] = torch.randn(n, generator=g, dtype=torch.float64) * 0.01 + 12.5
    rays[1] = torch.randn(n, generator=g, dtype=torch.float64) * 0.3 - 2.0
    flag = (torch.rand(n, generator=g) < 0.9).to(torch.int8)
    dev, fd = rays.cuda(), flag.cuda()
    out = torch.full((G, hip.SPOT_STRIDE), float("nan"), dtype=torch.float64, device="cuda")
    got = hip.group_spots(dev, fd, G, out=out).cpu().numpy()
    want = spot_reference(rays[0].numpy(), rays[1].numpy(), flag.numpy(), G)
    assert np.array_equal(got[:, 0], want[:, 0])
    # centroids: a few roundings of values near 12.5; variances: squares of
    # differences that carry 12.5 * 2^-53 each, against a variance of 1e-4
    assert np.all(np.abs(got[:, 1:3] - want[:, 1:3]) <= 1e-13)
    assert np.all(np.abs(got[:, 3:6] - want[:, 3:6]) <= 1e-10 * np.abs(want[:, 3:6]) + 1e-28)
