"""GPU parity of the head-dim-384 attention's key splits: counts from one to sixteen, chunks
that end short, fp32 partial rows (fewer than 1024 keys) and fp16 ones, several heads and
batch entries, and the allocation-free entry point on both sides of its scratch limit."""

import pytest
import torch

from animaxs_amd import AttentionExecutor, QKPrologue
from oracle import attention as oatt
from tests.helpers import assert_attention_close, dev

pytestmark = pytest.mark.gpu
D = 384


def _run(ctx, B, H, Sq, Sk, noalloc=False):
    g = torch.Generator().manual_seed(Sq + 7 * Sk + B)
    q = torch.randn(B, Sq, H, D, generator=g).half()
    k, v = (torch.randn(B, Sk, H, D, generator=g).half() for _ in range(2))
    o = torch.full((B, H, Sq, D), float("nan"), dtype=torch.float16, device="cuda")
    hm = [dev(t.permute(0, 2, 1, 3)) for t in (q, k, v)]
    ex = AttentionExecutor(ctx, layout="headMajor")
    call = ex.encode_noalloc if noalloc else ex.encode
    print(f"WIDE B={B} H={H} Sq={Sq} Sk={Sk} noalloc={noalloc}", flush=True)
    call(query=hm[0], key=hm[1], value=hm[2], output=o, heads=H, query_count=Sq, key_count=Sk, head_dim=D, batch=B)
    torch.cuda.synchronize()
    return o.permute(0, 2, 1, 3).float().cpu(), oatt.sdpa(q, k, v)


# Key counts: one split, one key more, a short last chunk, the most splits of one chunk each,
# the last with fp32 rows, the first with fp16 rows, chunks of several tiles.
@pytest.mark.parametrize("B,H,Sq,Sk", [(1, 1, 1, 64), (1, 1, 128, 65), (1, 1, 129, 200), (1, 1, 300, 1000),
                                       (1, 1, 257, 1023), (1, 1, 257, 1024), (1, 1, 100, 2100), (2, 3, 130, 700),
                                       (1, 15, 1024, 130), (1, 17, 1024, 130), (3, 2, 500, 1500)])
def test_wide_key_splits(ctx, B, H, Sq, Sk):
    out, ref = _run(ctx, B, H, Sq, Sk)
    assert_attention_close(out, ref, label=f"wide B={B} H={H} Sq={Sq} Sk={Sk}")


def test_wide_noalloc_equals_encode(ctx):
    a, ref = _run(ctx, 1, 1, 257, 1000)
    b, _ = _run(ctx, 1, 1, 257, 1000, noalloc=True)
    assert_attention_close(a, ref)
    assert torch.equal(a, b)


def test_wide_noalloc_beyond_its_scratch_takes_fewer_splits(ctx):
    """47 MB of normalised key rows and 50 MB of fp32 partial rows exceed the 64 MiB scratch;
    without the fine splits the call fits and runs."""
    B, Sq, Sk = 64, 128, 1000
    g = torch.Generator().manual_seed(5)
    q = torch.randn(B, 1, Sq, D, generator=g).half()
    k, v = (torch.randn(B, 1, Sk, D, generator=g).half() for _ in range(2))
    kw = (0.8 + 0.4 * torch.rand(D, generator=g)).half()
    ex = AttentionExecutor(ctx, layout="headMajor")
    args = dict(query=dev(q), key=dev(k), value=dev(v), heads=1, query_count=Sq, key_count=Sk, head_dim=D, batch=B,
                prologue=QKPrologue(None, dev(kw), 1e-6, None, 0, False, False))
    outs = [torch.full((B, 1, Sq, D), float("nan"), dtype=torch.float16, device="cuda") for _ in range(2)]
    ex.encode(output=outs[0], **args)
    ex.encode_noalloc(output=outs[1], **args)
    torch.cuda.synchronize()
    tm = [t.permute(0, 2, 1, 3) for t in (q, k, v)]
    ref = oatt.sdpa(tm[0], oatt.qk_prologue(tm[1], kw, 1e-6, None), tm[2])
    for o in outs:
        assert_attention_close(o.permute(0, 2, 1, 3), ref)


def test_wide_noalloc_equals_encode_beyond_its_scratch(ctx):
    """The same plan, and so the same bits, also where fine splits would exceed the scratch."""
    B, Sq, Sk = 64, 128, 1000
    g = torch.Generator().manual_seed(6)
    q, k, v = (dev(torch.randn(B, 1, n, D, generator=g).half()) for n in (Sq, Sk, Sk))
    kw = dev((0.8 + 0.4 * torch.rand(D, generator=g)).half())
    ex = AttentionExecutor(ctx, layout="headMajor")
    args = dict(query=q, key=k, value=v, heads=1, query_count=Sq, key_count=Sk, head_dim=D, batch=B,
                prologue=QKPrologue(None, kw, 1e-6, None, 0, False, False))
    outs = [torch.full((B, 1, Sq, D), float("nan"), dtype=torch.float16, device="cuda") for _ in range(2)]
    print("WIDE scratch limit", flush=True)
    ex.encode(output=outs[0], **args)
    ex.encode_noalloc(output=outs[1], **args)
    torch.cuda.synchronize()
    assert torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16))


# Calls whose fp32 partial rows cost more than the key tiles they would save, and one that splits.
@pytest.mark.parametrize("H,Sq,Sk,splits", [(1, 4096, 100, 1), (1, 2048, 256, 1), (8, 1024, 192, 1), (1, 128, 128, 1),
                                            (1, 4096, 500, 4), (2, 100, 1000, 16)])
def test_wide_split_count(ctx, H, Sq, Sk, splits):
    q, k, v = (torch.randn(H, n, D, device="cuda").half() for n in (Sq, Sk, Sk))
    ex = AttentionExecutor(ctx, layout="headMajor")
    print(f"WIDE COUNT H={H} Sq={Sq} Sk={Sk}", flush=True)
    ex.execute(query=q, key=k, value=v, output=torch.empty_like(q), heads=H, query_count=Sq, key_count=Sk, head_dim=D)
    rows = splits * H * Sq
    need = (rows * D * 4 + 255) // 256 * 256 + rows * 8 if splits > 1 else 0
    assert need <= ex.workspace_bytes() <= need + need // 8 + 8192
