"""The blends' entry groups (four list entries at a time): lists whose lengths
leave every remainder of a group, a wave's 64 entries and a batch, of plain
entries only, of none, and mixed within a group, on a screen of partial tiles."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from gaussian_splatting import synthetic
from helpers import assert_bitwise, assert_grad_close
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

NAMES = ("d_mean2d", "d_cov2d", "d_colors", "d_alpha")


def _scene(n, kind, H=21, W=37):
    """n splats over the screen's six tiles.  Not plain: an opacity at or above
    the clamp, a negative colour, a mean a hair from 0, a needle whose conic is
    near singular."""
    rng = np.random.default_rng(n)
    mean = rng.uniform([0.0, 0.0], [W, H], (n, 2))
    sig = rng.uniform(2.0, 9.0, (n, 2))
    rho = rng.uniform(-0.7, 0.7, n)
    cov = np.stack([sig[:, 0] ** 2 + 0.3, rho * sig[:, 0] * sig[:, 1], sig[:, 1] ** 2 + 0.3], 1)
    alpha = rng.uniform(0.02, 0.4, n)
    colors = rng.uniform(0.0, 1.0, (n, 3))
    odd = np.zeros(n, bool) if kind == "plain" else np.ones(n, bool)
    if kind == "mixed":
        odd = rng.random(n) < 0.3
    how = rng.integers(0, 4, n)
    alpha = np.where(odd & (how == 0), rng.choice([0.99, 0.999, 1.5], n), alpha)
    colors[odd & (how == 1), 0] *= -1.0
    mean[odd & (how == 2), 1] = 1e-20
    needle = odd & (how == 3)
    cov[needle] = np.array([3000.3, 2999.99, 3000.3])
    f32 = np.float32
    return dict(mean2d=mean.astype(f32), cov2d=cov.astype(f32), colors=colors.astype(f32),
                alpha=alpha.astype(f32).reshape(-1, 1),
                depth=rng.uniform(0.5, 9.0, n).astype(f32)), H, W


@pytest.mark.parametrize("kind", ["plain", "mixed", "odd"])
@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 63, 64, 65, 66, 127, 129, 200])
def test_groups_of_entries(crc, device, n, kind):
    print(f"[gpu] groups n {n} {kind}", flush=True)
    s, H, W = _scene(n, kind)
    t = {k: torch.from_numpy(np.ascontiguousarray(v)).to(device) for k, v in s.items()}
    img, ids, ranges, fT, nc = crc.rasterize(n, t["depth"], t["mean2d"], t["cov2d"], t["colors"],
                                             t["alpha"], H, W)
    w_img, w_ids, w_rng, w_fT, w_nc, _ = orc.rasterize(s["depth"], s["mean2d"], s["cov2d"],
                                                       s["colors"], s["alpha"], H, W)
    for got, want, nm in ((ids, w_ids, "ids"), (nc, w_nc, "n_contrib"), (img, w_img, "img"),
                          (fT, w_fT, "final_T")):
        assert_bitwise(got.cpu().numpy(), want, nm)
    G = synthetic.grad_image(H, W, seed=n).numpy()
    got = crc.backwards_rasterization(torch.from_numpy(G).to(device), t["mean2d"], t["cov2d"],
                                      t["colors"], t["alpha"], ids, ranges, fT, nc, n, H, W)
    torch.cuda.synchronize()
    args = (G, s["mean2d"], s["cov2d"], s["colors"], s["alpha"], w_ids, w_rng, w_fT, w_nc, H, W)
    ref, ref64 = orc.blend_bwd(*args, with_abs=True), orc.blend_bwd(*args, dtype=np.float64)
    for x, r, ab, r64, nm in zip(got, ref[:4], ref[4:], ref64, NAMES):
        # the needles' terms cancel to a few 1e-6 of their sum in any fp32
        # evaluation: an element also passes within twice the fp32 oracle's own
        # error against float64
        assert_grad_close(x.cpu().numpy().reshape(r.shape), r, ab, nm, want64=r64)
