"""GPU tests that a linear sums over K the same way alone, in a group and with a fused output
stage, where it runs split over K or in a small-M form that a fused launch does not have."""

import pytest
import torch

from animaxs_amd import BlockOps, LinearExecutor
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


# 17 to 64 rows past the K of the weight-streaming kernel: the plain linear runs split over K.
@pytest.mark.parametrize("storage,M,N,K", [(1, 40, 2048, 8256), (0, 40, 2048, 9216), (1, 64, 512, 16448),
                                           (0, 33, 130, 8256)])
def test_small_m_past_the_streaming_limit(ctx, storage, M, N, K):
    qw, _ = _weight(storage, N, K, M + N, False)
    g = torch.Generator().manual_seed(M)
    x, res, gate = dev(torch.randn(M, K, generator=g).half()), dev(torch.randn(M, N, generator=g)), dev(torch.randn(N, generator=g))
    lin, ops = LinearExecutor(ctx), BlockOps(ctx)
    print(f"SMALL M storage={storage} M={M} N={N} K={K}", flush=True)
    branch = torch.empty(M, N, dtype=torch.float16, device="cuda")
    lin.encode(x, qw, branch, M)
    gelu, want = torch.full_like(branch, float("nan")), branch.clone()
    lin.encode_epilogue(x, qw, gelu, M, "gelu")
    ops.gelu_half_inplace(want, M * N)
    r = [res.clone() for _ in range(4)]
    lin.encode_epilogue(x, qw, torch.empty_like(branch), M, "gate_add", residual=r[0], gate=gate)
    ops.gate_add_half_f32(r[1], branch, gate, N, M * N)
    lin.encode_epilogue(x, qw, torch.empty_like(branch), M, "residual_add", residual=r[2])
    ops.add_half_into_float(r[3], branch, M * N)
    group = [torch.full_like(branch, float("nan")) for _ in range(2)]
    lin.encode_group(x, [qw, qw], group, M)
    torch.cuda.synchronize()
    for a, b in ((gelu, want), (r[0], r[1]), (r[2], r[3]), (group[0], branch), (group[1], branch)):
        assert torch.equal(_bits(a), _bits(b))
