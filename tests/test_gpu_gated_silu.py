"""GPU test of gated_silu_half over every fp16 gate: SiLU and product keep fp32's precision before
their one rounding to fp16."""

import numpy as np
import pytest
import torch

from animaxs_amd import BlockOps
from tests.helpers import dev

pytestmark = pytest.mark.gpu


def _run(ctx, gate, up):
    out = torch.empty(gate.size, dtype=torch.float16, device="cuda")
    BlockOps(ctx).gated_silu_half(dev(gate), dev(up), out, gate.size)
    torch.cuda.synchronize()
    return out.cpu().numpy()


@pytest.mark.parametrize("seed", range(8))
def test_every_gate_rounds_as_fp32_allows(ctx, seed):
    """The result is the fp16 neighbour of a value within 3 ulp of fp32 of silu(gate) * up: 2 ulp
    for the SiLU (expf 1, the sum and the quotient 0.5 each) and 0.5 for the product, whose ulp
    may be half as large."""
    gate = np.arange(65536, dtype=np.uint32).astype(np.uint16).view(np.float16)
    gate = gate[np.isfinite(gate)]
    up = np.ones_like(gate)
    if seed:
        up = np.random.default_rng(seed).uniform(0.25, 4.0, gate.size).astype(np.float16)
    x = gate.astype(np.float64)
    with np.errstate(over="ignore"):
        exact = x / (1.0 + np.exp(-x)) * up.astype(np.float64)
    print(f"SILU seed={seed}", flush=True)
    y = _run(ctx, gate, up)
    slack = 3.0 * 2.0 ** -23 * np.abs(exact)
    with np.errstate(over="ignore"):
        lo, hi = (exact - slack).astype(np.float16), (exact + slack).astype(np.float16)
    bad = ~((y >= lo) & (y <= hi))
    assert not bad.any(), (int(bad.sum()), gate[bad][:4], up[bad][:4], y[bad][:4])
    if not seed:
        with np.errstate(over="ignore"):
            assert int((y != exact.astype(np.float16)).sum()) <= 1


def test_special_gates(ctx):
    inf, nan = np.float16(np.inf), np.float16(np.nan)
    gate = np.array([inf, -inf, nan, 0.0, -0.0, 65504, -65504, 128, 130, -88.6875, -88.75, -90, -inf, inf], np.float16)
    up = np.array([1, 1, 1, 1, 1, 1, 1, 1, 1, inf, inf, 1, 0, 0], np.float16)
    want = np.array([inf, nan, nan, 0.0, -0.0, 65504, -0.0, 128, 130, -inf, nan, -0.0, nan, nan], np.float16)
    y = _run(ctx, gate, up)
    assert np.array_equal(y, want, equal_nan=True)
    assert np.array_equal(np.signbit(y[~np.isnan(want)]), np.signbit(want[~np.isnan(want)]))
