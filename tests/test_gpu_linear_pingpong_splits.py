"""GPU tests of problems that need a second round of small tiles: on either side of the K that the
small tiles keep, and the ping-pong kernel's K splits (two and three, aligned scale windows and
not, odd element counts) with their output stages, in a group and under the Q/K norm."""

import pytest
import torch

from animaxs_amd import LinearExecutor
from tests.helpers import dev
from tests.test_gpu_linear_tile import _weight
from tests.test_gpu_linear_tile import test_small_tile_gemm_and_its_output_stages as check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("storage,misalign", [(0, False), (1, False), (0, True), (1, True)])
@pytest.mark.parametrize("M,N,K", [(1100, 2048, 512), (1100, 2048, 576), (1100, 2048, 1024), (1100, 2048, 1280),
                                   (1100, 2048, 2048), (1100, 2048, 2304), (1100, 2048, 4096), (2200, 1001, 4224),
                                   (2200, 1001, 3136)])
def test_second_round(ctx, storage, misalign, M, N, K):
    check(ctx, storage, misalign, M, N, K)


@pytest.mark.parametrize("storage", [0, 1])
def test_split_members_and_norm_keep_their_bits(ctx, storage):
    M, N, K = 1100, 2048, 4096
    qw, _ = _weight(storage, N, K, 5, False)
    g = torch.Generator().manual_seed(storage)
    x, nw = dev(torch.randn(M, K, generator=g).half()), dev((0.8 + 0.4 * torch.rand(128, generator=g)).half())
    lin = LinearExecutor(ctx)
    print(f"PINGPONG SPLIT storage={storage}", flush=True)
    y = torch.empty(M, N, dtype=torch.float16, device="cuda")
    lin.encode(x, qw, y, M)
    group = [torch.full_like(y, float("nan")) for _ in range(2)]
    lin.encode_group(x, [qw, qw], group, M)
    norms = [torch.full((M * N + 8,), float("nan"), dtype=torch.float16, device="cuda") for _ in range(2)]
    lin.encode_head_rmsnorm(x, qw, norms[0], M, nw)
    lin.encode_head_rmsnorm(x, qw, norms[1], M, nw, output_offset=16)
    torch.cuda.synchronize()
    for o in group:
        assert torch.equal(o.view(torch.int16), y.view(torch.int16))
    assert torch.equal(norms[0][:M * N].view(torch.int16), norms[1][8:].view(torch.int16))
