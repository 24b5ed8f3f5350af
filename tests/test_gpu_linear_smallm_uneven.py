"""GPU tests of the small-M linear where K is not a whole number of 128-wide chunks or of K
slices: every row-block count and slice length, padded weight rows whose padding must not be
read into the sum, and a last group that dequantises to infinity."""

import numpy as np
import pytest
import torch

import animaxs_amd
from animaxs_amd import LinearExecutor
from oracle import inputs, quant
from tests.helpers import dev

pytestmark = pytest.mark.gpu


def _case(storage, M, N, K, pad, infinite=False):
    g = torch.Generator().manual_seed(M + N + K)
    w = (inputs.symmetric_w4 if storage == 0 else inputs.symmetric_w8)(g, N, K)
    stride, groups = w["row_stride"] + pad, (K + 63) // 64
    rows = np.full((N, stride), 0xFF, np.uint8)
    rows[:, :w["row_stride"]] = np.asarray(w["packed"], np.uint8).reshape(N, -1)
    s, z = (np.asarray(w[n], np.uint16).reshape(N, groups).copy() for n in ("scale_bits", "zero_bits"))
    x = torch.randn(M, K, generator=g).half()
    if infinite:   # row 0: codes of the last group times 65504
        s[0, -1], z[0, -1] = 0x7BFF, 0
        rows[0, w["row_stride"] - (32 if storage == 0 else 64):w["row_stride"]] = 0x77
        x = x.abs() + 0.25
    with np.errstate(over="ignore"):
        dense = quant.dequant_to_half(storage, rows, s, z, N, K, stride)
    buffers = [dev(rows.reshape(-1))] + [dev(a.reshape(-1).view(np.int16)) for a in (s, z)]
    q = animaxs_amd.QuantizedLinearWeightBuffers(storage, *buffers, N, K, stride)
    return q, torch.from_numpy(dense.view(np.float16).astype(np.float64)), x


# Weight streaming: one half chunk, waves with a half chunk or none of their own, one to four
# row blocks of X.  Split K: slices of 1, 2, 4 and 8 chunks whose last one ends short, by
# whole chunks and by half a chunk, down to a slice of one half chunk.
SHAPES = [(1, 17, 64, 0), (1, 64, 192, 16), (16, 100, 320, 16), (17, 513, 448, 0), (33, 8200, 320, 0), (64, 8192, 64, 16),
          (1, 520, 7616, 0), (9, 1000, 1088, 16), (40, 520, 64, 0), (40, 130, 704, 16), (64, 2048, 1920, 0),
          (20, 5000, 6720, 0), (64, 4096, 1088, 16), (50, 7000, 2112, 0), (59, 6032, 2560, 0), (13, 300, 16448, 0)]


@pytest.mark.parametrize("storage", [0, 1])
@pytest.mark.parametrize("M,N,K,pad", SHAPES)
def test_uneven_k(ctx, storage, M, N, K, pad):
    """Within the fp16 store's half ulp and K rounding steps of the fp32 sum on sum |x w|."""
    q, dense, x = _case(storage, M, N, K, pad)
    print(f"UNEVEN storage={storage} M={M} N={N} K={K} pad={pad}", flush=True)
    y = torch.full((M + 1, N), float("nan"), dtype=torch.float16, device="cuda")
    LinearExecutor(ctx).encode(dev(x), q, y, M)
    torch.cuda.synchronize()
    assert bool(torch.isnan(y[M]).all())
    ref, mag = x.double() @ dense.T, x.double().abs() @ dense.abs().T
    err = (y[:M].cpu().double() - ref).abs()
    bound = ref.abs() * 2.0 ** -11 + (K + 1) * 2.0 ** -24 * mag * (1 + 2.0 ** -10) + 2.0 ** -25
    assert bool((err <= bound).all()), float((err / bound).max())


@pytest.mark.parametrize("storage", [0, 1])
@pytest.mark.parametrize("M,N,K", [(1, 64, 192), (20, 130, 1088), (64, 512, 1984), (20, 512, 6720)])
def test_infinite_last_group(ctx, storage, M, N, K):
    """The repeated end of a row counts for nothing, infinities included."""
    q, dense, x = _case(storage, M, N, K, 0, infinite=True)
    y = torch.full((M, N), float("nan"), dtype=torch.float16, device="cuda")
    LinearExecutor(ctx).encode(dev(x), q, y, M)
    torch.cuda.synchronize()
    assert bool(torch.isposinf(y[:, 0]).all()) and bool(torch.isinf(dense[0, -64:]).all())
    assert bool(torch.isfinite(y[:, 1:]).all())


# More than 32 rows on either side of the X that streams (96 KB) at K = 64 (mod 128).
@pytest.mark.parametrize("storage", [0, 1])
@pytest.mark.parametrize("M,N,K", [(33, 77, 1472), (33, 77, 1600), (48, 130, 960), (48, 130, 1088), (64, 300, 704),
                                   (64, 300, 832), (64, 6000, 320)])
def test_streamed_rows_limit(ctx, storage, M, N, K):
    test_uneven_k(ctx, storage, M, N, K, 0)
