"""A few tokens through the fp8 MoE layer: the intermediate handed over in fp32 and quantised by the down GEMM (one
token's experts, and about one column tile with rows per CU), activations quantised ahead of the main loop, and the
sizes next to either rule.  The alignment handed over or not, the result has the same bits."""
import pytest
import torch

from oracle import fp8 as ofp8
from oracle import fused_moe as ofm
from oracle import moe_gating as og

pytestmark = pytest.mark.gpu


def _layer(dev, T, H, I, E, k, shuffled, dtype, first=0, local=None, skew=False):
    from dlcompiler_amd.kernels.fused_moe import ALIGN_BLOCK, fused_moe_fp8, shuffle_moe_weight
    from dlcompiler_amd.kernels.moe_gating import moe_align_block_size

    local = local or E
    g = torch.Generator().manual_seed(T * H + I)
    # (an outlier of about 90 makes gate and up about 5, so |h| stays below 100 and outputs, sums of up to 4224 of them
    # with weights of 0.05, far below fp16's 65504)
    x = torch.randn((T, H), generator=g) * torch.logspace(-2, 0, T)[:, None]
    if H > 128:
        x[0, :128] = 0.0                 # a group of zeros
    x[-1, 5] *= 30.0                     # an outlier
    x = x.to(dtype)
    w1, s1 = ofp8.block_quant_weight(torch.randn((local, 2 * I, H), generator=g) * 0.05)
    w2, s2 = ofp8.block_quant_weight(torch.randn((local, H, I), generator=g) * 0.05)
    logits = torch.randn((T, E), generator=g)
    if skew:
        logits[:, 1] += 20.0             # every token at one expert
    tw, ids = og.topk_softmax(logits, k, renormalize=False)
    ref = ofm.fused_moe_fp8(x, w1, s1, w2, s2, tw, ids, expert_offset=first).double()
    x, w1, s1, w2, s2, tw, ids = (t.to(dev) for t in (x, w1, s1, w2, s2, tw, ids))
    if shuffled:
        w1, w2 = shuffle_moe_weight(w1), shuffle_moe_weight(w2)
    slots, _, _, counts = moe_align_block_size(ids, ALIGN_BLOCK, E, return_counts=True)
    args = (x, w1, s1, w2, s2, tw, ids, k, first, E)
    own = fused_moe_fp8(*args, weights_shuffled=shuffled)
    out = fused_moe_fp8(*args, weights_shuffled=shuffled, alignment=(slots, counts))
    assert torch.equal(out, own)
    # (bits of one call after another are the same)
    assert torch.equal(out, fused_moe_fp8(*args, weights_shuffled=shuffled, alignment=(slots, counts)))
    # a value next to a rounding boundary of the fp8 intermediate falls to either side: 2^-4 of it, few of a row's
    rows = (out.cpu().double() - ref).norm(dim=1) / ref.norm(dim=1).clamp_min(1e-9)
    assert (rows[ref.norm(dim=1) > 0] < 3e-2).all() and (rows > 0).any(), rows
    assert (out.cpu()[ref.norm(dim=1) == 0] == 0).all()


@pytest.mark.parametrize("T,H,I,E,k", [(1, 128, 128, 1, 1), (1, 2048, 384, 64, 6), (1, 2176, 256, 8, 2),
                                       (3, 4096, 128, 16, 4), (1, 4224, 128, 8, 2), (2, 256, 4096, 4, 2),
                                       (1, 256, 4224, 4, 1), (2, 512, 2176, 8, 2), (16, 640, 256, 16, 4)])
@pytest.mark.parametrize("shuffled", [False, True])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_few_column_tiles(dev, T, H, I, E, k, shuffled, dtype):
    _layer(dev, T, H, I, E, k, shuffled, dtype)


# 256 CUs, 257 to 548 tiles with rows: quantised ahead of the main loop, rows of up to 2048 and of 4096
@pytest.mark.parametrize("T,H,I,E,k", [(10, 384, 1024, 40, 6), (8, 384, 1024, 64, 8), (12, 256, 1024, 64, 8),
                                       (30, 2048, 640, 128, 8), (20, 2304, 640, 64, 8)])
def test_more_column_tiles(dev, T, H, I, E, k):
    _layer(dev, T, H, I, E, k, True, torch.bfloat16)


# rows of 1536 and more: 256 tiles with rows, fp32 intermediate, and 224, quantised in every step
@pytest.mark.parametrize("T,H", [(12, 1536), (12, 2304), (9, 1536)])
def test_a_tile_per_cu(dev, T, H):
    _layer(dev, T, H, 1280, 32, 4, True, torch.bfloat16)


@pytest.mark.parametrize("T,E", [(20, 64), (33, 16), (7, 8)])
def test_one_expert_with_several_row_tiles(dev, T, E):
    _layer(dev, T, 384, 256, E, 2, True, torch.bfloat16, skew=True)


@pytest.mark.parametrize("first", [0, 8])
def test_shard(dev, first):
    _layer(dev, 4, 512, 256, 16, 4, True, torch.bfloat16, first=first, local=8)
