"""GPU tests of executors under graph capture: a first call may be a captured one (no workspace
can be allocated then), and a captured call's workspace outlives larger eager calls."""

import pytest
import torch

from animaxs_amd import AttentionExecutor, Context, LinearExecutor
from tests.helpers import dev
from tests.test_gpu_linear_tile import _weight

pytestmark = pytest.mark.gpu


@pytest.fixture
def stream():
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        yield s
    torch.cuda.synchronize()


def _captured(stream, call):
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=stream):
        call()
    return graph


def _close(y, ref, label):
    """Sums over K or the keys in another order, then one fp16 rounding."""
    err = float((y.double() - ref.double()).norm() / ref.double().norm())
    print(f"CAPTURE {label}: rel {err:.2e}", flush=True)
    assert err <= 1e-3


# Small tiles and the small-M kernel where an eager call splits K, whole and uneven.
@pytest.mark.parametrize("storage,M,N,K", [(1, 109, 128, 5696), (0, 191, 752, 6016), (1, 40, 130, 704), (0, 20, 464, 1216)])
def test_first_linear_call_under_capture(stream, storage, M, N, K):
    qw, _ = _weight(storage, N, K, M + N, False)
    x = dev(torch.randn(M, K, generator=torch.Generator().manual_seed(M)).half())
    eager, y = (torch.empty(M, N, dtype=torch.float16, device="cuda") for _ in range(2))
    ctx = Context(0, stream)
    LinearExecutor(ctx).encode(x, qw, eager, M)
    cold = LinearExecutor(ctx)
    graph = _captured(stream, lambda: cold.encode(x, qw, y, M))
    for _ in range(3):
        y.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        _close(y, eager, f"storage={storage} M={M} N={N} K={K}")


@pytest.mark.parametrize("S", [200, 900])
def test_first_wide_attention_call_under_capture(stream, S):
    q, k, v = (dev(torch.randn(S, 384, generator=torch.Generator().manual_seed(i)).half()) for i in range(3))
    eager, y = (torch.empty_like(q) for _ in range(2))
    ctx = Context(0, stream)
    args = dict(query=q, key=k, value=v, heads=1, query_count=S, key_count=S, head_dim=384)
    AttentionExecutor(ctx, layout="headMajor").encode(output=eager, **args)
    cold = AttentionExecutor(ctx, layout="headMajor")
    graph = _captured(stream, lambda: cold.encode(output=y, **args))
    for _ in range(3):
        y.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        _close(y, eager, f"head_dim 384 S={S}")
