"""GPU parity of the grouped GEMMs from few rows per expert to many: tile heights of 16 to 128 rows, waves
side by side or splitting K, chunk counts that do not divide by the waves, experts without rows, skewed
routing (several row tiles of one expert), rows just past a tile, and the edge to the tiled fp8 kernel."""
import pytest
import torch

from oracle import fp8 as ofp8
from oracle import fused_moe as ofm
from oracle import moe_gating as og

pytestmark = pytest.mark.gpu


def _routing(T, E, k, skew, g):
    logits = torch.randn((T, E), generator=g)
    if skew:
        logits[:, 1] += 8.0   # every token goes to expert 1 as well
    return og.topk_softmax(logits, k, renormalize=False)


# (T, H, I, E, k): mean rows per expert 0.2 .. 315
SHAPES = [(1, 128, 128, 8, 2), (3, 640, 384, 64, 6), (40, 2048, 256, 64, 6), (17, 256, 1408, 8, 2),
          (75, 384, 128, 8, 2), (100, 1152, 640, 16, 4), (168, 256, 256, 8, 2), (169, 256, 256, 8, 2),
          (224, 192, 320, 8, 2), (225, 192, 320, 8, 2), (300, 64, 192, 4, 2), (333, 512, 128, 4, 2),
          (420, 128, 384, 4, 3)]
# on either side of each limit: 7, 22, 32 (fp8: the tiled kernel from there on) and 52 rows per expert where waves split
# K, 19 and 36 where they run side by side
SHAPES += [(T, 256, 384, 8, 2) for T in (28, 29, 88, 89, 128, 129, 208, 209)]
SHAPES += [(T, 128, 1088, 64, 4) for T in (304, 305, 576, 577)]
# rows of 4096 fp8 bytes, in either GEMM, where waves start at other chunks: tiles of 16, 32 and 64 rows
SHAPES += [(T, H, I, 4, 2) for T in (6, 30, 60) for H, I in ((4096, 256), (256, 4096))]


@pytest.mark.parametrize("T,H,I,E,k", SHAPES)
@pytest.mark.parametrize("skew", [False, True])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_sixteen_bit(dev, T, H, I, E, k, skew, dtype):
    from dlcompiler_amd.kernels.fused_moe import fused_moe, shuffle_moe_weight

    g = torch.Generator().manual_seed(T + H)
    x = torch.randn((T, H), generator=g).to(dtype)
    w1, w2 = (torch.randn(s, generator=g).mul_(0.05).to(dtype) for s in ((E, 2 * I, H), (E, H, I)))
    tw, ids = _routing(T, E, k, skew, g)
    ref = ofm.fused_moe(x, w1, w2, tw, ids, renormalize=True).double()
    args = (x.to(dev), w1.to(dev), w2.to(dev), tw.to(dev), ids.to(dev))
    for out in (fused_moe(*args, k, renormalize=True),
                fused_moe(args[0], shuffle_moe_weight(args[1]), shuffle_moe_weight(args[2]), args[3],
                          args[4].to(torch.int64), k, renormalize=True, weights_shuffled=True)):
        err = ((out.cpu().double() - ref).norm() / ref.norm()).item()
        assert err < 5e-3, err


@pytest.mark.parametrize("T,H,I,E,k", [s for s in SHAPES if s[1] % 128 == 0])
@pytest.mark.parametrize("skew", [False, True])
def test_fp8(dev, T, H, I, E, k, skew):
    from dlcompiler_amd.kernels.fused_moe import ALIGN_BLOCK, fused_moe_fp8, shuffle_moe_weight
    from dlcompiler_amd.kernels.moe_gating import moe_align_block_size

    g = torch.Generator().manual_seed(T + H)
    I = -(-I // 128) * 128
    x = torch.randn((T, H), generator=g).to(torch.bfloat16)
    w1, s1 = ofp8.block_quant_weight(torch.randn((E, 2 * I, H), generator=g) * 0.05)
    w2, s2 = ofp8.block_quant_weight(torch.randn((E, H, I), generator=g) * 0.05)
    tw, ids = _routing(T, E, k, skew, g)
    ref = ofm.fused_moe_fp8(x, w1, s1, w2, s2, tw, ids).double()
    xd, w1, s1, w2, s2, tw, ids = (t.to(dev) for t in (x, w1, s1, w2, s2, tw, ids))
    slots, _, _, counts = moe_align_block_size(ids, ALIGN_BLOCK, E, return_counts=True)
    for out in (fused_moe_fp8(xd, w1, s1, w2, s2, tw, ids, k),
                fused_moe_fp8(xd, shuffle_moe_weight(w1), s1, shuffle_moe_weight(w2), s2, tw, ids, k,
                              weights_shuffled=True, alignment=(slots, counts))):
        err = ((out.cpu().double() - ref).norm() / ref.norm()).item()
        assert err <= 3e-2, err


@pytest.mark.parametrize("topk", [2, 3])
def test_expert_shards_add_up(dev, topk):
    """Two halves of an expert-parallel group: slots of experts held elsewhere are not read."""
    from dlcompiler_amd.kernels.fused_moe import fused_moe

    g = torch.Generator().manual_seed(topk)
    T, H, I, E = 50, 256, 128, 8
    x = torch.randn((T, H), generator=g).to(torch.bfloat16)
    w1, w2 = (torch.randn(s, generator=g).mul_(0.05).to(torch.bfloat16) for s in ((E, 2 * I, H), (E, H, I)))
    tw, ids = og.topk_softmax(torch.randn((T, E), generator=g), topk, renormalize=False)
    xd, tw, ids = x.to(dev), tw.to(dev), ids.to(dev)
    halves = [fused_moe(xd, w1[o:o + 4].to(dev), w2[o:o + 4].to(dev), tw, ids, topk, o, E, True).double()
              for o in (0, 4)]
    whole = fused_moe(xd, w1.to(dev), w2.to(dev), tw, ids, topk, renormalize=True).double()
    assert ((halves[0] + halves[1] - whole).norm() / whole.norm()).item() < 1e-2
