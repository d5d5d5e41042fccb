"""fp8 MoE with many rows per expert: row tiles with one row and on either side of 32, 64, 96 and 128, slots per token
whose reciprocal is exact and inexact, reductions of 64 and 65 chunks (the block scales of a tile come in strips of 64),
routing weights as they are and divided by their sum."""
import pytest
import torch

from oracle import fp8 as ofp8
from oracle import fused_moe as ofm

pytestmark = pytest.mark.gpu

# the layer's bound against the dequantised fp32 evaluation: two fp8 roundings (2^-4 each way, averaged over the sums)
REL = 3e-2


def _check(dev, ids, E, H, I, renormalize, shuffled):
    from dlcompiler_amd.kernels.fused_moe import fused_moe_fp8, shuffle_moe_weight

    T, k = ids.shape
    assert T * k > 32 * E  # the tiled kernel
    g = torch.Generator().manual_seed(T + H)
    x = torch.randn((T, H), generator=g).to(torch.bfloat16)
    w1, s1 = ofp8.block_quant_weight(torch.randn((E, 2 * I, H), generator=g) * 0.02)
    w2, s2 = ofp8.block_quant_weight(torch.randn((E, H, I), generator=g) * 0.02)
    tw = torch.rand((T, k), generator=g) + 0.1
    ref = ofm.fused_moe_fp8(x, w1, s1, w2, s2, tw, ids, renormalize=renormalize).double()
    d = [t.to(dev) for t in (x, w1, s1, w2, s2, tw, ids)]
    if shuffled:
        d[1], d[3] = shuffle_moe_weight(d[1]), shuffle_moe_weight(d[3])
    out = fused_moe_fp8(*d, k, renormalize=renormalize, weights_shuffled=shuffled).cpu().double()
    assert ((out - ref).norm() / ref.norm()).item() <= REL
    # every row by itself: one that took another's slot, weight or scale is off by its whole size
    rows = (out - ref).norm(dim=1) / ref.norm(dim=1).clamp_min(1e-6)
    assert rows.max().item() <= 4 * REL


@pytest.mark.parametrize("counts", [[1, 31, 32, 33, 129], [63, 64, 65, 1, 0], [95, 96, 97, 127], [128, 130, 257]])
@pytest.mark.parametrize("renormalize", [False, True])
@pytest.mark.parametrize("shuffled", [False, True])
def test_row_tiles(dev, counts, renormalize, shuffled):
    ids = torch.cat([torch.full((n,), e, dtype=torch.int32) for e, n in enumerate(counts)])
    ids = ids[torch.randperm(len(ids), generator=torch.Generator().manual_seed(1))]
    _check(dev, ids[:, None], len(counts), 384, 256, renormalize, shuffled)


@pytest.mark.parametrize("T,E,k", [(70, 4, 2), (80, 5, 3), (90, 7, 5), (120, 8, 7)])
@pytest.mark.parametrize("renormalize", [False, True])
def test_slots_per_token(dev, T, E, k, renormalize):
    g = torch.Generator().manual_seed(T)
    ids = torch.stack([torch.randperm(E, generator=g)[:k] for _ in range(T)]).to(torch.int32)
    _check(dev, ids, E, 256, 128, renormalize, True)


@pytest.mark.parametrize("H,I", [(8192, 128), (8320, 128), (128, 8192), (128, 8320)])
def test_long_reductions(dev, H, I):
    ids = torch.tensor([0] * 40 + [1] * 33, dtype=torch.int32)[:, None]
    _check(dev, ids, 2, H, I, False, False)
