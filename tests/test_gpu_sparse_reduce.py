"""The gradient reduction's two ways of finding claimed slots: a cloud one short
of the count at which a wave looks through 16 Gaussians' claim bits, and the same
cloud with splats off the screen added past it.  Every sum is taken in the same
order, so the gradients are equal bit for bit, and the added splats' are zero."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from gaussian_splatting import synthetic
from helpers import assert_bitwise

pytestmark = pytest.mark.gpu

LINE = 1 << 19
NAMES = ("d_mean2d", "d_cov2d", "d_colors", "d_alpha")


@pytest.mark.parametrize("sigma,added", [(26.0, 1), (26.0, 18), (26.0, 77), (75.0, 18)])
def test_sparse_reduce_equals_rows(crc, device, sigma, added):
    print(f"[gpu] sparse reduce sigma {sigma} added {added}", flush=True)
    H, W = 400, 520
    n = LINE - 1
    rng = np.random.default_rng(7)
    f32 = np.float32
    mean = rng.uniform([0.0, 0.0], [W, H], (n + added, 2))
    mean[n:] = -1.0e5
    sig = sigma * rng.uniform(0.8, 1.3, (n + added, 2))
    sig[n:] = 1.0
    cov = np.stack([sig[:, 0] ** 2, 0.1 * sig[:, 0] * sig[:, 1], sig[:, 1] ** 2], 1)
    s = dict(depth=rng.uniform(0.5, 9.0, n + added), mean2d=mean, cov2d=cov,
             colors=rng.uniform(0.0, 1.0, (n + added, 3)),
             alpha=rng.uniform(0.02, 0.6, (n + added, 1)))
    t = {k: torch.from_numpy(v.astype(f32)).to(device) for k, v in s.items()}
    G = synthetic.grad_image(H, W, seed=3).to(device)

    def grads(count):
        a = {k: v[:count].contiguous() for k, v in t.items()}
        _, ids, ranges, fT, nc = crc.rasterize(count, a["depth"], a["mean2d"], a["cov2d"],
                                               a["colors"], a["alpha"], H, W)
        assert ids.numel() > (256 if sigma > 50 else 64) * count
        out = crc.backwards_rasterization(G, a["mean2d"], a["cov2d"], a["colors"], a["alpha"],
                                          ids, ranges, fT, nc, count, H, W)
        return [x.cpu().numpy() for x in out]

    rows, sparse = grads(n), grads(n + added)
    for want, got, nm in zip(rows, sparse, NAMES):
        assert np.abs(want).max() > 0.0
        assert_bitwise(got[:n], want, nm)
        assert not got[n:].any(), nm
