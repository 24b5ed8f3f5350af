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


# Members of the ping-pong kernel and of small tiles, of both tile shapes, one that splits K
# between two that do not, two storages, two rounds of tiles and the K that leaves them, and rows that fill the ping-pong kernel together.
@pytest.mark.parametrize("M,members,K", [(2000, ((1, 2048), (1, 1024), (1, 1024)), 512),
                                         (300, ((0, 2048), (0, 1024), (0, 1024)), 1024),
                                         (77, ((1, 4096), (1, 256), (1, 4096)), 4096),
                                         (512, ((0, 1024), (1, 1024), (0, 1024)), 512),
                                         (2100, ((0, 1024), (0, 1024)), 512), (2100, ((0, 1024), (1, 1024)), 1024), (77, ((1, 192), (1, 64)), 192)])
def test_groups_of_several_kernels(ctx, M, members, K):
    qws = [_weight(st, N, K, i + N, False)[0] for i, (st, N) in enumerate(members)]
    x = dev(torch.randn(M, K, generator=torch.Generator().manual_seed(M)).half())
    lin = LinearExecutor(ctx)
    refs, outs = ([torch.full((M, N), float("nan"), dtype=torch.float16, device="cuda") for _, N in members]
                  for _ in range(2))
    print(f"GROUP KERNELS M={M} members={members} K={K}", flush=True)
    for qw, r in zip(qws, refs):
        lin.encode(x, qw, r, M)
    lin.encode_group(x, qws, outs, M)
    torch.cuda.synchronize()
    for r, o in zip(refs, outs):
        assert bool(torch.isfinite(r).all()) and torch.equal(_bits(r), _bits(o))


# Encoder layers whose Q, K and V are one launch: of small tiles of one shape where the linears
# alone would take two, of the narrow ones, and of the ping-pong kernel in place of small tiles.
@pytest.mark.parametrize("S", [20, 150, 300, 700])
def test_encoder_projections_in_one_launch(ctx, S):
    from animaxs_amd import QwenLayerExecutor
    from oracle import blocks, inputs
    from tests.helpers import device_weight, mean_rel
    d = inputs.qwen_layer(B=1, S=S, hidden=256, heads=16, kv_heads=8, intermediate=192)
    print(f"ENCODER S={S}", flush=True)
    weights, keep = {}, []
    for n, w in d["w"].items():
        weights[n], k = device_weight(w)
        keep.append(k)
    norms = {n: dev(d[n]) for n in ("input_norm", "post_attention_norm", "q_norm", "k_norm")}
    residual = dev(d["x"].clone())
    QwenLayerExecutor(ctx).encode(weights, norms, residual, dev(d["rope"]), batch=1, tokens=S,
                                  key_lengths=d["key_lengths"].numpy(), hidden=256, heads=16, kv_heads=8, intermediate=192)
    torch.cuda.synchronize()
    ref = blocks.qwen_layer(d, boundary="fp16") - d["x"]
    assert mean_rel(residual.cpu() - d["x"], ref) <= 2e-3
