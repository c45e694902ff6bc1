"""The densification gather at the edges of its 256-source blocks and of the
scan's 1024 runs: one block less and more by one, and a last block of one
source, against the oracle (the comparison of tests/test_gpu_adc.py)."""

from __future__ import annotations

import pytest

from test_gpu_adc import test_adc_matches_the_oracle as _matches_the_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 63, 65, 255, 256, 257, 513, 262_145])
@pytest.mark.parametrize("reset", [False, True])
def test_adc_block_edges(device, n, reset):
    print(f"[gpu] adc blocks {n} {reset}", flush=True)
    _matches_the_oracle(device, n, seed=n + 11, reset=reset, screen=40.0)
