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


def test_captured_workspace_outlives_a_larger_call(stream):
    """A graph of a split linear, then an eager call whose partial rows need more: the graph's rows
    stay its own on later replays, also once the memory that a freed one would return is taken."""
    M, N, K = 109, 128, 5696
    qw, _ = _weight(1, N, K, 1, False)
    big, _ = _weight(1, 752, 6016, 2, False)
    x = dev(torch.randn(M, K, generator=torch.Generator().manual_seed(3)).half())
    xb = dev(torch.randn(191, 6016, generator=torch.Generator().manual_seed(4)).half())
    eager, y = (torch.empty(M, N, dtype=torch.float16, device="cuda") for _ in range(2))
    yb = torch.empty(191, 752, dtype=torch.float16, device="cuda")
    lin = LinearExecutor(Context(0, stream))
    lin.encode(x, qw, eager, M)
    graph = _captured(stream, lambda: lin.encode(x, qw, y, M))
    lin.encode(xb, big, yb, 191)
    torch.cuda.synchronize()
    taken = torch.full((1 << 22,), 7.0, device="cuda")
    for _ in range(3):
        y.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y.view(torch.int16), eager.view(torch.int16))
    assert bool((taken == 7.0).all())


def test_workspace_bytes_count_what_a_graph_keeps(stream):
    q, k, v = (dev(torch.randn(4000, 384, generator=torch.Generator().manual_seed(i)).half()) for i in range(3))
    o = torch.empty_like(q)
    ex = AttentionExecutor(Context(0, stream), layout="headMajor")

    def call(S):
        ex.encode(query=q[:S], key=k[:S], value=v[:S], output=o[:S], heads=1, query_count=S, key_count=S, head_dim=384)

    call(500)
    small = ex.workspace_bytes()
    graph = _captured(stream, lambda: call(500))
    call(4000)
    held = ex.workspace_bytes()
    other = AttentionExecutor(Context(0, stream), layout="headMajor")
    other.encode(query=q, key=k, value=v, output=o, heads=1, query_count=4000, key_count=4000, head_dim=384)
    torch.cuda.synchronize()
    assert small > 0 and held == small + other.workspace_bytes()
    del graph
