"""The block lists at large counts (one work-group per 512 depth ranks from 2^19
Gaussians on): counts around that line and around a work-group's ranks, screens
of up to 64 x 64 blocks of 8 x 8 tiles, one column or row more, and more blocks
than the scatter takes at a time.  Tile lists equal to the oracle's."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from helpers import assert_bitwise
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

LINE = 1 << 19


def _scene(n, H, W):
    """Mostly small splats (some off the screen, without tiles), a few over
    hundreds of blocks, depths with ties."""
    rng = np.random.default_rng(n + W)
    f32 = np.float32
    mean = rng.uniform([-0.1 * W, -0.1 * H], [1.1 * W, 1.1 * H], (n, 2))
    sig = rng.uniform(0.3, 3.0, (n, 2))
    sig[rng.choice(n, 12, replace=False)] = [W / 8.0, H / 8.0]
    sig[rng.choice(n, 300, replace=False)] = [90.0, 4.0]
    cov = np.stack([sig[:, 0] ** 2 + 0.3, 0.2 * sig[:, 0] * sig[:, 1], sig[:, 1] ** 2 + 0.3], 1)
    depth = np.round(rng.uniform(0.5, 9.0, n), 3)
    return dict(depth=depth.astype(f32), mean2d=mean.astype(f32), cov2d=cov.astype(f32),
                colors=rng.uniform(0.0, 1.0, (n, 3)).astype(f32),
                alpha=rng.uniform(0.02, 0.4, (n, 1)).astype(f32))


@pytest.mark.parametrize("n,H,W", [
    (LINE - 1, 144, 8192), (LINE, 144, 8192), (LINE + 1, 144, 8192), (LINE + 513, 8192, 144),
    (LINE + 65, 144, 8200), (LINE + 65, 8200, 144),  # 65 blocks a side
    (LINE + 511, 2080, 4112),                        # 33 x 17 blocks
])
def test_block_lists_at_large_counts(crc, device, n, H, W):
    print(f"[gpu] block lists n {n} {H}x{W}", flush=True)
    s = _scene(n, H, W)
    t = {k: torch.from_numpy(v).to(device) for k, v in s.items()}
    img, ids, ranges, fT, nc = crc.rasterize(n, t["depth"], t["mean2d"], t["cov2d"], t["colors"],
                                             t["alpha"], H, W)
    w_img, w_ids, w_rng, w_fT, w_nc, _ = orc.rasterize(s["depth"], s["mean2d"], s["cov2d"],
                                                       s["colors"], s["alpha"], H, W)
    for got, want, nm in ((ids, w_ids, "ids"), (ranges, w_rng, "ranges"), (nc, w_nc, "n_contrib"),
                          (img, w_img, "img"), (fT, w_fT, "final_T")):
        assert_bitwise(got.cpu().numpy(), want, nm)
