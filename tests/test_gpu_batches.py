"""The backward's batches: of a tile's list only the entries that one of its
strips meets are staged, 128 list entries looked at together, until a batch is
half full; what does not fit waits for the next.  Lists of needle-shaped splats
(few entries meet a strip), of wide ones (all do), and of runs of both, whose
windows overflow a batch at any fill; opaque enough that pixels stop at
different entries, and long enough for split tiles."""

from __future__ import annotations

import numpy as np
import pytest

from helpers import assert_bitwise
from test_gpu_groups import LARGE, NAMES, SMALL, _backward

pytestmark = pytest.mark.gpu


def _scene(kind, n, screen):
    H, W = screen
    rng = np.random.default_rng(len(kind) * 1000 + n)
    if kind == "needles":
        needle = np.ones(n, bool)
    elif kind == "wide":
        needle = np.zeros(n, bool)
    else:  # runs of 1 to 200 of either, in depth order
        needle = np.zeros(0, bool)
        while needle.size < n:
            run = int(rng.integers(1, 200))
            needle = np.concatenate([needle, np.full(run, rng.random() < 0.6)])
        needle = needle[:n]
    mean = rng.uniform([W - 77.0, -40.0], [W + 40.0, 61.0], (n, 2))
    long_, short = np.where(needle, 45.0, 14.0), np.where(needle, 0.4, 9.0)
    angle = rng.uniform(0.0, np.pi, n)
    c, s = np.cos(angle), np.sin(angle)
    a, b = long_ ** 2, short ** 2
    cov = np.stack([a * c * c + b * s * s + 0.3, (a - b) * c * s, a * s * s + b * c * c + 0.3], 1)
    f32 = np.float32
    return dict(mean2d=mean.astype(f32), cov2d=cov.astype(f32),
                colors=rng.uniform(0.0, 1.0, (n, 3)).astype(f32),
                alpha=np.where(needle, rng.uniform(0.1, 0.9, n),
                               rng.uniform(0.004, 0.02, n)).astype(f32).reshape(-1, 1),
                depth=np.linspace(0.5, 9.0, n).astype(f32)), H, W


@pytest.mark.parametrize("screen", [SMALL, LARGE], ids=["small", "large"])
@pytest.mark.parametrize("kind,n", [("needles", 130), ("needles", 900), ("wide", 129),
                                    ("wide", 700), ("runs", 257), ("runs", 1500), ("runs", 1501)])
def test_batches(crc, device, kind, n, screen, monkeypatch):
    print(f"[gpu] batches {kind} {n} {screen}", flush=True)
    s, H, W = _scene(kind, n, screen)
    args, split = _backward(crc, device, s, H, W, seed=n)
    monkeypatch.setenv("GSR_BWD_SPLIT", "0")
    whole = crc.backwards_rasterization(*args)
    for x, y, nm in zip(split, whole, NAMES):
        assert_bitwise(x.cpu().numpy(), y.cpu().numpy(), nm)
