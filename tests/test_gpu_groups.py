"""The blends' entry groups (four list entries at a time): lists whose lengths
leave every remainder of a group, of 64 and of 128 entries, of plain entries
only, of none, and mixed within a group.  On a small screen of partial tiles,
whose grid is resident on the device at once (one pixel per lane forward,
128-entry batches and split tiles backward), and in a corner of one of 7,708
tiles, which is not (two pixels per lane, 64-entry batches)."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from gaussian_splatting import synthetic
from helpers import assert_bitwise, assert_grad_close
from oracle import oracle as orc
from test_gpu_parity import _threshold_scene

pytestmark = pytest.mark.gpu

NAMES = ("d_mean2d", "d_cov2d", "d_colors", "d_alpha")
SMALL, LARGE = (21, 37), (1301, 1493)
# at the trainer's bound on the logit, log(0.99 / 0.01), the fp32 sigmoid is
# just above the blends' clamp at 0.99
BOUND = np.float32(0.99000007)


def _scene(n, kind, screen=SMALL):
    """n splats over six tiles in the screen's upper right corner.  Not plain: an
    opacity at or above the clamp, a negative or infinite colour, a mean a hair
    from 0, a needle whose conic is near singular."""
    H, W = screen
    rng = np.random.default_rng(n)
    mean = rng.uniform([W - 37.0, 0.0], [W, 21.0], (n, 2))
    sig = rng.uniform(2.0, 9.0, (n, 2))
    rho = rng.uniform(-0.7, 0.7, n)
    cov = np.stack([sig[:, 0] ** 2 + 0.3, rho * sig[:, 0] * sig[:, 1], sig[:, 1] ** 2 + 0.3], 1)
    alpha = rng.uniform(0.02, 0.4, n)
    colors = rng.uniform(0.0, 1.0, (n, 3))
    if kind == "bound":  # a trained cloud: a third at the bound
        alpha = np.where(rng.random(n) < 0.3, BOUND, alpha)
    odd = np.zeros(n, bool) if kind in ("plain", "bound") else np.ones(n, bool)
    if kind == "mixed":
        odd = rng.random(n) < 0.3
    how = rng.integers(0, 5, n)
    alpha = np.where(odd & (how == 0), rng.choice([0.99, BOUND, 1.0, 1.5, 6.0, -0.2], n), alpha)
    colors[odd & (how == 1), 0] *= -1.0
    mean[odd & (how == 2), 1] = 1e-20
    cov[odd & (how == 3)] = np.array([30000.3, 29999.99, 30000.3])
    cov[odd & (how == 4)] = np.array([3000.3, 2999.99, 3000.3])
    f32 = np.float32
    return dict(mean2d=mean.astype(f32), cov2d=cov.astype(f32), colors=colors.astype(f32),
                alpha=alpha.astype(f32).reshape(-1, 1),
                depth=rng.uniform(0.5, 9.0, n).astype(f32)), H, W


def _forward(crc, device, s, H, W):
    """The forward on the GPU and by the oracle, equal bit for bit."""
    t = {k: torch.from_numpy(np.ascontiguousarray(s[k])).to(device)
         for k in ("depth", "mean2d", "cov2d", "colors", "alpha")}
    n = s["alpha"].shape[0]
    img, ids, ranges, fT, nc = crc.rasterize(n, t["depth"], t["mean2d"], t["cov2d"], t["colors"],
                                             t["alpha"], H, W)
    w_img, w_ids, w_rng, w_fT, w_nc, _ = orc.rasterize(s["depth"], s["mean2d"], s["cov2d"],
                                                       s["colors"], s["alpha"], H, W)
    for got, want, nm in ((ids, w_ids, "ids"), (nc, w_nc, "n_contrib"), (img, w_img, "img"),
                          (fT, w_fT, "final_T")):
        assert_bitwise(got.cpu().numpy(), want, nm)
    args = (t["mean2d"], t["cov2d"], t["colors"], t["alpha"], ids, ranges, fT, nc, n, H, W)
    return args, (w_ids, w_rng, w_fT, w_nc)


def _backward(crc, device, s, H, W, seed):
    args, (w_ids, w_rng, w_fT, w_nc) = _forward(crc, device, s, H, W)
    G = synthetic.grad_image(H, W, seed=seed)
    Gt = G.to(device)
    got = crc.backwards_rasterization(Gt, *args)
    torch.cuda.synchronize()
    oargs = (G.numpy(), s["mean2d"], s["cov2d"], s["colors"], s["alpha"], w_ids, w_rng, w_fT, w_nc,
             H, W)
    ref, ref64 = orc.blend_bwd(*oargs, with_abs=True), orc.blend_bwd(*oargs, dtype=np.float64)
    for x, r, ab, r64, nm in zip(got, ref[:4], ref[4:], ref64, NAMES):
        # the needles' terms cancel to a few 1e-6 of their sum in any fp32
        # evaluation: an element also passes within twice the fp32 oracle's own
        # error against float64.  A near singular needle's determinant is 2e-5
        # of a c, which leaves 3e-3 (6e-8 over 2e-5) in any fp32 conversion of
        # its terms, and a list of such alone is all that its tensor holds: the
        # tensor is held to 1.5 times the fp32 oracle's own error there.
        assert_grad_close(x.cpu().numpy().reshape(r.shape), r, ab, nm, want64=r64,
                          tensor_vs64=True)
    return (Gt, *args), got


@pytest.mark.parametrize("screen", [SMALL, LARGE], ids=["small", "large"])
@pytest.mark.parametrize("kind", ["plain", "bound", "mixed", "odd"])
@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 63, 64, 65, 66, 127, 129, 200])
def test_groups_of_entries(crc, device, n, kind, screen):
    print(f"[gpu] groups n {n} {kind} {screen}", flush=True)
    s, H, W = _scene(n, kind, screen)
    _backward(crc, device, s, H, W, seed=n)


@pytest.mark.parametrize("kind", ["plain", "bound", "mixed"])
def test_groups_in_split_tiles(crc, device, kind, monkeypatch):
    """Lists long enough for the split of the longest tiles: an entry's sums do
    not depend on the group that it is walked in, so the gradients are those of
    whole tiles (GSR_BWD_SPLIT=0) bit for bit."""
    print(f"[gpu] groups in split tiles {kind}", flush=True)
    s, H, W = _scene(900, kind)
    s["alpha"] = np.where(s["alpha"] < 0.5, s["alpha"] * np.float32(0.1), s["alpha"])
    if kind == "bound":  # behind most of the others, whose lists stay long
        at = s["alpha"][:, 0] > 0.5
        s["depth"] = np.where(at, s["depth"] + np.float32(7.0), s["depth"])
    args, split = _backward(crc, device, s, H, W, seed=9)
    assert int(args[8].max()) >= 256  # n_contrib
    monkeypatch.setenv("GSR_BWD_SPLIT", "0")
    whole = crc.backwards_rasterization(*args)
    for x, y, nm in zip(split, whole, NAMES):
        assert_bitwise(x.cpu().numpy(), y.cpu().numpy(), nm)


def test_thresholds_on_a_large_screen(crc, device):
    """Alphas within a few ulp of 1/255 and opacities about the clamp
    (test_gpu_parity's scene) on the large screen."""
    print("[gpu] thresholds on a large screen", flush=True)
    s = _threshold_scene()
    _backward(crc, device, s, *LARGE, seed=4)


def test_infinite_colours_on_a_large_screen(crc, device):
    print("[gpu] infinite colours on a large screen", flush=True)
    s = _threshold_scene(seed=23)
    rng = np.random.default_rng(5)
    pick = rng.choice(np.arange(600, s["alpha"].shape[0]), 12, replace=False)
    s["colors"][pick, rng.integers(0, 3, 12)] = np.float32(np.inf)
    _forward(crc, device, s, *LARGE)
