"""GPU parity of the router + alignment around the sizes where the launch changes: one workgroup up to
80 to 128 tokens / 4096 slots, 64- and 128-token chunks beyond."""
import pytest
import torch

from oracle import moe_gating as og

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,E,k,block", [(256, 256, 16, 128), (257, 256, 16, 128), (256, 13, 3, 16), (257, 13, 3, 16),
                                         (128, 64, 16, 128), (129, 64, 16, 128), (96, 128, 8, 64), (97, 128, 8, 64), (80, 200, 8, 64), (81, 200, 8, 64),
                                         (192, 128, 8, 1), (16384, 255, 2, 128), (16448, 256, 16, 64)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_router_and_alignment_at_launch_edges(dev, T, E, k, block, dtype):
    from dlcompiler_amd.kernels.moe_gating import moe_topk_softmax_align

    logits = torch.randn((T, E), generator=torch.Generator().manual_seed(T + E)).to(dtype)
    w, ids, slots, experts, total, counts = moe_topk_softmax_align(logits.to(dev), k, block, return_counts=True)
    rw, rids = og.topk_softmax(logits.float(), k)
    rs, re_, rn, rc = og.align_block_size(rids, block, E)
    assert torch.equal(ids.cpu(), rids) and torch.equal(slots.cpu(), rs) and torch.equal(experts.cpu(), re_)
    assert int(total.item()) == int(rn.item()) and torch.equal(counts.cpu(), rc.to(torch.int32))
    torch.testing.assert_close(w.cpu(), rw, rtol=2e-6, atol=0)


@pytest.mark.parametrize("numel", [0, 1, 63, 1023, 1025, 4096, 4097])
@pytest.mark.parametrize("E,block", [(256, 128), (5, 16)])
def test_alignment_of_given_ids_at_launch_edges(dev, numel, E, block):
    from dlcompiler_amd.kernels.moe_gating import moe_align_block_size

    ids = torch.randint(-1, E + 1, (numel, 1), generator=torch.Generator().manual_seed(numel), dtype=torch.int32)
    slots, experts, total, counts = moe_align_block_size(ids.to(dev), block, E, return_counts=True)
    rs, re_, rn, rc = og.align_block_size(ids, block, E)
    assert torch.equal(slots.cpu(), rs) and torch.equal(experts.cpu(), re_)
    assert int(total.item()) == int(rn.item()) and torch.equal(counts.cpu(), rc.to(torch.int32))


# block sizes whose reciprocal is exact, inexact and the smallest; one expert with more blocks than threads, in one
# launch, in two and in three
@pytest.mark.parametrize("block", [1, 3, 7, 127, 1 << 16])
@pytest.mark.parametrize("numel", [300, 4000, 30000, 530000])
@pytest.mark.parametrize("E", [1, 3, 256])
def test_blocks_of_one_expert(dev, block, numel, E):
    from dlcompiler_amd.kernels.moe_gating import moe_align_block_size

    ids = torch.full((numel, 1), E // 2, dtype=torch.int32)
    ids[::11] = E - 1
    slots, experts, total, counts = moe_align_block_size(ids.to(dev), block, E, return_counts=True)
    rs, re_, rn, rc = og.align_block_size(ids, block, E)
    assert torch.equal(slots.cpu(), rs) and torch.equal(experts.cpu(), re_)
    assert int(total.item()) == int(rn.item()) and torch.equal(counts.cpu(), rc.to(torch.int32))


# either side of: one launch or two, 16 / 32 / 64 / 128 tokens per workgroup of the router
@pytest.mark.parametrize("T,E,k", [(36, 256, 8), (37, 256, 8), (56, 128, 8), (57, 100, 8), (96, 64, 6), (97, 64, 16),
                                   (1024, 256, 8), (1025, 256, 8), (2048, 128, 8), (2049, 128, 8), (4096, 64, 6),
                                   (4097, 60, 4), (8192, 129, 8), (8193, 256, 8), (8192, 16, 2), (16385, 8, 2)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_router_and_alignment_at_chunk_edges(dev, T, E, k, dtype):
    from dlcompiler_amd import _lib
    from dlcompiler_amd.kernels.moe_gating import moe_topk_softmax_align

    logits = torch.randn((T, E), generator=torch.Generator().manual_seed(T + E)).to(dtype)
    x = logits.to(dev)
    w, ids, slots, experts, total, counts = moe_topk_softmax_align(x, k, 64, return_counts=True)
    rw, rids = og.topk_softmax(logits.float(), k)
    rs, re_, rn, rc = og.align_block_size(rids, 64, E)
    assert torch.equal(ids.cpu(), rids) and torch.equal(slots.cpu(), rs) and torch.equal(experts.cpu(), re_)
    assert int(total.item()) == int(rn.item()) and torch.equal(counts.cpu(), rc.to(torch.int32))
    torch.testing.assert_close(w.cpu(), rw, rtol=2e-6, atol=0)
    # a scratch with room for chunks of 64 tokens, and for the 128 that many tokens take, gives the same
    rows = -(-T // (64 if T <= 16384 else 128))
    ws = torch.empty(rows * ((E + 3) // 4) * 4, dtype=torch.uint8, device=dev)
    again = [torch.empty_like(t) for t in (w, ids, slots, experts, counts, total)]
    st = _lib.load().dlb_moe_topk_softmax_align_f32(
        x.data_ptr(), again[0].data_ptr(), again[1].data_ptr(), T, E, k, E, _lib.torch_dtype_code(dtype), 1, 64,
        again[2].data_ptr(), slots.numel(), again[3].data_ptr(), experts.numel(), again[4].data_ptr(),
        again[5].data_ptr(), ws.data_ptr(), ws.numel(), _lib.current_stream_ptr(x.device))
    assert st == 0
    for a, b in zip(again, (w, ids, slots, experts, counts, total)):
        assert torch.equal(a, b)
