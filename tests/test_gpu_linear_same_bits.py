"""GPU tests that a linear sums over K the same way alone, in a group and with a fused output
stage, where it runs split over K or in a small-M form that a fused launch does not have."""

import pytest
import torch

from animaxs_amd import LinearExecutor
from tests.helpers import dev
from tests.test_gpu_linear_tile import _weight

pytestmark = pytest.mark.gpu


def _bits(t):
    return t.view(torch.int16 if t.dtype == torch.float16 else torch.int32)


# Small tiles of 64 x 128 that split K in two, in two uneven splits, and 32 x 64 ones.
@pytest.mark.parametrize("storage,M,N,K", [(1, 512, 2048, 4096), (0, 512, 2048, 4096), (1, 500, 1920, 4672),
                                           (1, 77, 2048, 8192)])
def test_head_rmsnorm_keeps_the_split(ctx, storage, M, N, K):
    """An output eight halfs into its buffer takes the linear, then the norm in place; one at the
    start of its buffer may take the fused stage, with the same sums."""
    qw, _ = _weight(storage, N, K, M + N, False)
    g = torch.Generator().manual_seed(M)
    x, nw = dev(torch.randn(M, K, generator=g).half()), dev((0.8 + 0.4 * torch.rand(128, generator=g)).half())
    lin = LinearExecutor(ctx)
    outs = [torch.full((M * N + 8,), float("nan"), dtype=torch.float16, device="cuda") for _ in range(2)]
    print(f"HEADNORM SPLIT storage={storage} M={M} N={N} K={K}", flush=True)
    lin.encode_head_rmsnorm(x, qw, outs[0], M, nw)
    lin.encode_head_rmsnorm(x, qw, outs[1], M, nw, output_offset=16)
    torch.cuda.synchronize()
    assert torch.equal(_bits(outs[0][:M * N]), _bits(outs[1][8:]))
