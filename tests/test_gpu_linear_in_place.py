"""GPU test of a linear whose output lies over its input: right where the ping-pong kernel covers
it with one tile (64 < rows <= 128, or K = 64 (mod 128), and up to 256 columns)."""

import pytest
import torch

from animaxs_amd import LinearExecutor
from tests.helpers import dev
from tests.test_gpu_linear_tile import _weight

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("storage", [0, 1])
@pytest.mark.parametrize("M,N,K,rows", [(100, 256, 256, 0), (128, 192, 192, 0), (65, 130, 1024, 0), (40, 192, 192, 0),
                                        (128, 256, 256, 3)])
def test_output_over_the_input(ctx, storage, M, N, K, rows):
    """rows: input rows that the output starts behind."""
    qw, dense = _weight(storage, N, K, M + N, False)
    x = torch.randn(M, K, generator=torch.Generator().manual_seed(M)).half()
    buf = torch.zeros(max(M * K, M * N + rows * K), dtype=torch.float16)
    buf[:M * K] = x.reshape(-1)
    buf = dev(buf)
    print(f"IN PLACE storage={storage} M={M} N={N} K={K} rows={rows}", flush=True)
    LinearExecutor(ctx).encode(buf, qw, buf, M, output_offset=2 * rows * K)
    torch.cuda.synchronize()
    y = buf[rows * K:rows * K + M * N].reshape(M, N).cpu().double()
    ref, mag = x.double() @ dense.T, x.double().abs() @ dense.abs().T
    err = (y - ref).abs()
    bound = ref.abs() * 2.0 ** -11 + (K + 1) * 2.0 ** -24 * mag * (1 + 2.0 ** -10) + 2.0 ** -25
    assert bool((err <= bound).all()), float((err / bound).max())
