"""GPU: calls whose work follows lengths on the device, captured once and replayed with other lengths: chunked
prefill whose key tiles are split over as many workgroups as the contexts need (none, a few, the grid's
room), paged decode in two launches, and the MoE layers of a few rows per expert.  Replays are interleaved
with eager work and synchronisations and compared with the eager call bit for bit."""
import pytest
import torch

from oracle import attention as oatt
from oracle import fp8 as ofp8

pytestmark = pytest.mark.gpu


def _capture(fn):
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        fn()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = fn()
    return graph, out


@pytest.mark.parametrize("decode", [False, True])
def test_contexts_change_between_replays(dev, decode):
    from dlcompiler_amd.kernels.paged_attention import paged_attention_fwd

    Hq, Hkv, D, page, width, B = 8, 2, 64, 64, 128, 3
    new = 1 if decode else 20
    gen = torch.Generator().manual_seed(2)
    kc, vc = (torch.randn((B * width, page, Hkv, D), generator=gen).bfloat16().to(dev) for _ in range(2))
    table = torch.randperm(B * width, generator=gen).to(torch.int32).view(B, width).to(dev)
    q = torch.empty((B * new, Hq, D), dtype=torch.bfloat16, device=dev)
    o = torch.empty_like(q)
    start = torch.arange(B, dtype=torch.int32, device=dev) * new
    lens = torch.full((B,), new, dtype=torch.int32, device=dev)
    ctx = torch.empty((B,), dtype=torch.int32, device=dev)

    def call():
        paged_attention_fwd(q, kc, vc, o, table, start, lens, ctx, new)
        return o

    def fill(contexts, seed):
        ctx.copy_(torch.tensor(contexts, dtype=torch.int32))
        q.copy_(torch.randn(q.shape, generator=torch.Generator().manual_seed(seed)).bfloat16())

    fill([8000, 20, 3000], 0)
    graph, _ = _capture(call)
    for rep, contexts in enumerate([[20, 21, 500], [8192, 8192, 8192], [900, 5000, 20], [20, 20, 20], [8000, 20, 3000]]):
        fill(contexts, 10 + rep)
        eager = call().clone()
        o.fill_(7.0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(o, eager), contexts
    ref = (oatt.paged_decode(q.cpu(), kc.cpu(), vc.cpu(), table.cpu(), ctx.cpu()) if decode else
           oatt.paged_prefill(q.cpu(), kc.cpu(), vc.cpu(), table.cpu(), start.cpu(), lens.cpu(), ctx.cpu()))
    torch.testing.assert_close(o.cpu().float(), ref.float(), rtol=2e-2, atol=2e-2)


@pytest.mark.parametrize("fp8", [False, True])
def test_moe_of_a_few_rows_per_expert(dev, fp8):
    from dlcompiler_amd.kernels.fused_moe import ALIGN_BLOCK, fused_moe, fused_moe_fp8
    from dlcompiler_amd.kernels.moe_gating import moe_topk_softmax_align

    T, H, I, E, k = 24, 384, 256, 16, 4
    gen = torch.Generator().manual_seed(3)
    w1, w2 = torch.randn((E, 2 * I, H), generator=gen) * 0.05, torch.randn((E, H, I), generator=gen) * 0.05
    if fp8:
        (w1, s1), (w2, s2) = ofp8.block_quant_weight(w1), ofp8.block_quant_weight(w2)
        s1, s2 = s1.to(dev), s2.to(dev)
    w1, w2 = (t.to(dev) if fp8 else t.bfloat16().to(dev) for t in (w1, w2))
    x = torch.empty((T, H), dtype=torch.bfloat16, device=dev)
    logits = torch.empty((T, E), device=dev)

    def call():
        tw, ids, slots, _, _, counts = moe_topk_softmax_align(logits, k, ALIGN_BLOCK, return_counts=True)
        if fp8:
            return fused_moe_fp8(x, w1, s1, w2, s2, tw, ids, k, alignment=(slots, counts))
        return fused_moe(x, w1, w2, tw, ids, k, alignment=(slots, counts))

    def fill(seed):
        g = torch.Generator().manual_seed(seed)
        x.copy_(torch.randn((T, H), generator=g).bfloat16())
        logits.copy_(torch.randn((T, E), generator=g))

    fill(0)
    graph, out = _capture(call)
    for rep in range(4):
        fill(20 + rep)
        eager = call().clone()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager) and torch.isfinite(out.float()).all()
