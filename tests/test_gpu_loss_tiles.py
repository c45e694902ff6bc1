"""The loss kernels at the edges of their 32x16 tiles: images of one window, of
one tile, one row or column more and less, and tiles whose halo leaves the image
on every side, against the float64 oracle (bars: tests/test_gpu_loss.py)."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from helpers import assert_grad_close
from oracle import loss_oracle as lo

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,W", [(11, 12), (15, 31), (16, 32), (17, 33), (21, 37), (26, 42),
                                 (32, 64), (33, 65), (47, 11), (11, 97)])
def test_loss_at_tile_edges(crc, device, H, W):
    print(f"[gpu] loss tiles {H}x{W}", flush=True)
    rng = np.random.default_rng(H * 101 + W)
    r = rng.normal(0.5, 0.35, (H, W, 3)).astype(np.float32)
    g = rng.uniform(0.0, 1.0, (H, W, 3)).astype(np.float32)
    rt, gt = torch.from_numpy(r).to(device), torch.from_numpy(g).to(device)
    out, ws = crc.l1_dssim(rt, gt, 0.2)
    d = crc.l1_dssim_backward(rt, gt, 0.2, ws, torch.tensor([2.0], device=device))
    got, want = out.cpu().numpy(), lo.l1_dssim(r, g, 0.2)
    assert np.abs(got - np.asarray(want)).max() <= 1e-5
    wg, ab = lo.l1_dssim_grad(r, g, 0.2, grad_loss=2.0, with_abs=True)
    assert_grad_close(d.cpu().numpy(), wg, ab, f"dL/drendered {H}x{W}")


def test_loss_keeps_nan(crc, device):
    """A NaN pixel reaches the loss (the clamp keeps it), as torch's does."""
    r = torch.full((40, 40, 3), 0.5, device=device)
    r[20, 20, 1] = float("nan")
    out, _ = crc.l1_dssim(r, torch.full_like(r, 0.25), 0.2)
    assert torch.isnan(out).all()
