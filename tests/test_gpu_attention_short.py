"""GPU parity of the short-sequence attention kernel: tile and chunk edges (32 query rows,
128 keys), every prologue form, masks, layouts and strides, against the CPU oracle and
against the 256-row kernel, which takes the same calls with flash_rows = 256."""

import numpy as np
import pytest
import torch

from animaxs_amd import AttentionExecutor, QKPrologue
from oracle import attention as oatt
from tests.helpers import assert_attention_close, dev, mean_rel

pytestmark = pytest.mark.gpu


def _table(g, n, D, rotation=True):
    a = torch.rand(n, D // 2, generator=g) * 6.28
    lower = a.sin() if rotation else 0.5 * a.sin()   # the lower row is read on its own for K
    return torch.stack([a.cos(), -a.sin(), lower, a.cos()], dim=-1).reshape(n, D // 2, 2, 2).contiguous()


def _case(ctx, B, H, Hkv, Sq, Sk, D, pro, *, causal=False, lengths=None, head_major=False, device_lengths=False):
    g = torch.Generator().manual_seed(7 * Sq + 3 * Sk + D + B)
    q = torch.randn(B, Sq, H, D, generator=g).half()
    k, v = (torch.randn(B, Sk, Hkv, D, generator=g).half() for _ in range(2))
    qw, kw = ((0.8 + 0.4 * torch.rand(D, generator=g)).half() for _ in range(2))
    if "norm" not in pro:
        qw = kw = None
    rq = _table(g, Sq, D) if "rope" in pro else None
    rk = _table(g, Sk, D) if "rope" in pro else None
    args = None
    if pro:
        args = QKPrologue(qw if qw is None else dev(qw), kw if kw is None else dev(kw), 1e-6,
                          rq if rq is None else dev(rq), Sq if rq is not None else 0, rq is not None, rk is not None,
                          k_rope=rk if rk is None else dev(rk), k_rope_tokens=Sk if rk is not None else 0)
    perm = (lambda t: t.permute(0, 2, 1, 3).contiguous()) if head_major else (lambda t: t)
    kwargs = dict(heads=H, key_value_heads=Hkv, query_count=Sq, key_count=Sk, head_dim=D, batch=B, causal=causal,
                  prologue=args)
    if not head_major and Hkv != H:
        kwargs["kv_token_stride"] = Hkv * D
    if lengths is not None:
        kwargs["key_lengths"] = dev(torch.tensor(lengths, dtype=torch.int32)) if device_lengths else np.asarray(lengths, np.int32)
        kwargs["key_lengths_on_device"] = device_lengths
    outs = []
    for rows in (0, 256):
        o = torch.full(perm(q).shape, float("nan"), dtype=torch.float16, device="cuda")
        ex = AttentionExecutor(ctx, layout="headMajor" if head_major else ("tokenMajor", H * D), flash_rows=rows)
        ex.execute(query=dev(perm(q)), key=dev(perm(k)), value=dev(perm(v)), output=o, **kwargs)
        if rows == 0:
            assert ex.workspace_bytes() == 0, "the short kernel needs no workspace"
        outs.append(o.permute(0, 2, 1, 3).float().cpu() if head_major else o.float().cpu())
    ref = oatt.sdpa(oatt.qk_prologue(q, qw, 1e-6, rq), oatt.qk_prologue(k, kw, 1e-6, rk), v, causal=causal,
                    key_lengths=lengths)
    assert_attention_close(outs[0], ref)
    # Both kernels round Q, K, P and O to fp16 once: neither may be further from the oracle
    # than the other by more than the spread of such roundings over few rows.
    assert mean_rel(outs[0], ref) <= 1.2 * mean_rel(outs[1], ref) + 1e-5


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("Sq,Sk", [(1, 1), (31, 15), (32, 16), (33, 17), (77, 64), (5, 127), (64, 128), (40, 129),
                                   (32, 257), (96, 512)])
def test_tile_and_chunk_edges(ctx, D, Sq, Sk):
    _case(ctx, 1, 4, 4, Sq, Sk, D, "norm rope")


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("pro", ["", "norm", "rope", "norm rope"])
@pytest.mark.parametrize("head_major", [False, True])
def test_prologue_forms_and_layouts(ctx, D, pro, head_major):
    _case(ctx, 2, 4, 2, 50, 150, D, pro, head_major=head_major)


@pytest.mark.parametrize("S,lengths,device_lengths", [(1, None, False), (32, [32, 1], False), (77, [77, 20], True),
                                                      (130, [129, 64], False), (300, [7, 300], True)])
def test_causal_and_lengths(ctx, S, lengths, device_lengths):
    _case(ctx, 1 if lengths is None else 2, 4, 2, S, S, 128, "norm rope", causal=True, lengths=lengths,
          device_lengths=device_lengths)


def test_two_rounds_of_one_chunk(ctx):
    _case(ctx, 2, 16, 16, 512, 100, 64, "norm", lengths=[100, 31])


def test_general_table_is_read_as_the_prologue_reads_it(ctx):
    """A table whose lower row is no rotation's: K follows its own entries on both paths."""
    g = torch.Generator().manual_seed(5)
    q, k, v = (dev(torch.randn(40, 4, 128, generator=g).half()) for _ in range(3))
    pro = QKPrologue(None, None, 1e-6, dev(_table(g, 40, 128, rotation=False)), 40, True, True)
    outs = []
    for rows in (0, 256):
        o = torch.empty_like(q)
        AttentionExecutor(ctx, layout=("tokenMajor", 512), flash_rows=rows).execute(
            query=q, key=k, value=v, output=o, heads=4, query_count=40, key_count=40, head_dim=128, prologue=pro)
        outs.append(o.float().cpu())
    assert mean_rel(outs[0], outs[1]) <= 1e-3


def test_output_over_the_keys(ctx):
    """Behind a K prologue the output may take the key rows' place."""
    g = torch.Generator().manual_seed(6)
    q, k, v = (torch.randn(1, 70, 4, 128, generator=g).half() for _ in range(3))
    kw = torch.ones(128, dtype=torch.float16)
    kd = dev(k)
    AttentionExecutor(ctx, layout=("tokenMajor", 512)).execute(
        query=dev(q), key=kd, value=dev(v), output=kd, heads=4, query_count=70, key_count=70, head_dim=128,
        prologue=QKPrologue(None, dev(kw), 1e-6, None, 0, False, False))
    ref = oatt.sdpa(q, oatt.qk_prologue(k, kw, 1e-6, None), v)
    assert_attention_close(kd.float().cpu(), ref)


@pytest.mark.parametrize("where", ["key", "value", "query", "query shifted"])
@pytest.mark.parametrize("S,D", [(40, 64), (70, 128), (256, 128)])
def test_output_over_an_input(ctx, where, S, D):
    """Up to 256 queries the output may take an input's place, whatever kernel runs: the bits of
    the 256-row kernel where it does, and the query's own rows in the short kernel too."""
    g = torch.Generator().manual_seed(S)
    x = {n: torch.randn(S, 1, D, generator=g).half() for n in ("query", "key", "value")}
    kw = dict(heads=1, query_count=S, key_count=S, head_dim=D)
    want = torch.empty(S, 1, D, dtype=torch.float16, device="cuda")
    print(f"OVER {where} S={S} D={D}", flush=True)
    rows = 0 if where == "query" else 256
    AttentionExecutor(ctx, layout=("tokenMajor", D), flash_rows=rows).execute(
        **{n: dev(t) for n, t in x.items()}, output=want, **kw)
    d = {n: dev(t) for n, t in x.items()}
    if where == "query shifted":   # eight rows into the buffer that holds the query rows
        d["query"] = dev(torch.cat([x["query"], torch.zeros(8, 1, D, dtype=torch.float16)]))
        AttentionExecutor(ctx, layout=("tokenMajor", D)).execute(**d, output=d["query"], output_offset=16 * D, **kw)
        got = d["query"][8:]
    else:
        AttentionExecutor(ctx, layout=("tokenMajor", D)).execute(**d, output=d[where], **kw)
        got = d[where]
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
