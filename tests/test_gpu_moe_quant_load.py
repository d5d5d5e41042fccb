"""A few rows per expert: the gate_up GEMM quantises the activations that it loads.  With an alignment that
the caller brings it does; without one the quantiser runs in the alignment's launch: the same bytes."""
import pytest
import torch

from oracle import fp8 as ofp8
from oracle import fused_moe as ofm
from oracle import moe_gating as og

pytestmark = pytest.mark.gpu


# (T, H, I, E, k): K loops of one chunk and more, split over two waves or not, 7 rows per expert and past it
@pytest.mark.parametrize("T,H,I,E,k", [(1, 128, 128, 8, 2), (2, 384, 256, 64, 6), (28, 256, 384, 8, 2),
                                       (29, 256, 384, 8, 2), (74, 1152, 640, 64, 6)])
@pytest.mark.parametrize("shuffled", [False, True])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_same_as_the_quantiser(dev, T, H, I, E, k, shuffled, dtype):
    from dlcompiler_amd.kernels.fused_moe import ALIGN_BLOCK, fused_moe_fp8, shuffle_moe_weight
    from dlcompiler_amd.kernels.moe_gating import moe_align_block_size

    g = torch.Generator().manual_seed(T * H)
    x = torch.zeros((T, H + 8))          # rows that are not packed
    x[:, :H] = torch.randn((T, H), generator=g) * torch.logspace(-2, 1, T)[:, None]
    x[0, :128] = 0.0                     # a group of zeros
    x[-1, 5] *= 300.0                    # an outlier
    x = x.to(dtype)
    w1, s1 = ofp8.block_quant_weight(torch.randn((E, 2 * I, H), generator=g) * 0.05)
    w2, s2 = ofp8.block_quant_weight(torch.randn((E, H, I), generator=g) * 0.05)
    tw, ids = og.topk_softmax(torch.randn((T, E), generator=g), k, renormalize=False)
    ref = ofm.fused_moe_fp8(x[:, :H].contiguous(), w1, s1, w2, s2, tw, ids).double()
    xd, w1, s1, w2, s2, tw, ids = (t.to(dev) for t in (x, w1, s1, w2, s2, tw, ids))
    if shuffled:
        w1, w2 = shuffle_moe_weight(w1), shuffle_moe_weight(w2)
    slots, _, _, counts = moe_align_block_size(ids, ALIGN_BLOCK, E, return_counts=True)
    args = (xd[:, :H], w1, s1, w2, s2, tw, ids, k)
    own = fused_moe_fp8(*args, weights_shuffled=shuffled)
    out = fused_moe_fp8(*args, weights_shuffled=shuffled, alignment=(slots, counts))
    assert torch.equal(out, own)
    rows = (out.cpu().double() - ref).norm(dim=1) / ref.norm(dim=1).clamp_min(1e-9)
    assert rows.max().item() < 3e-2, rows.max().item()
