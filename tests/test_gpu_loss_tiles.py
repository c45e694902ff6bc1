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


def test_loss_gradient_is_as_near_to_64_bits_as_fp32_sums_allow(crc, device):
    """The SSIM gradient's distance from float64 on white noise (no cancellation
    in the variances, so the window sums' own rounding is what is left), mean of
    eight images.  A window sum of 22 products adds them two passes of 11, and
    its rounding grows with its partial sums: 1.69e-7 measured with the
    horizontal pass taken from the window's ends inwards, 2.18e-7 to 2.20e-7 with
    both in the order of the taps (+- 0.02e-7 per image)."""
    err = []
    for seed in range(8):
        rng = np.random.default_rng(seed)
        r, g = (rng.uniform(0.0, 1.0, (64, 96, 3)).astype(np.float32) for _ in range(2))
        rt, gt = torch.from_numpy(r).to(device), torch.from_numpy(g).to(device)
        out, ws = crc.l1_dssim(rt, gt, 1.0)
        d = crc.l1_dssim_backward(rt, gt, 1.0, ws).cpu().numpy().astype(np.float64)
        want = lo.l1_dssim_grad(r, g, 1.0)
        err.append(np.linalg.norm(d - want) / np.linalg.norm(want))
    print(f"[gpu] loss gradient from float64: {np.mean(err):.3e}", flush=True)
    assert np.mean(err) <= 1.9e-7
