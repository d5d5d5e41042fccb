"""A NaN activation reaches the output whichever kernel quantises it, and only its token's row."""
import pytest
import torch

from oracle import fp8 as ofp8
from oracle import fused_moe as ofm
from oracle import moe_gating as og

pytestmark = pytest.mark.gpu
NAN = float("nan")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_quantiser(dev, dtype):
    from dlcompiler_amd.kernels.fused_moe import per_token_group_quant_fp8

    x = torch.randn((5, 384), generator=torch.Generator().manual_seed(1)).to(dtype)
    clean_q, clean_s = per_token_group_quant_fp8(x.to(dev))
    x[1, 3] = x[4, 130] = NAN
    x[2, 128:256] = NAN
    q, s = per_token_group_quant_fp8(x.to(dev))
    assert torch.equal(torch.isnan(q.float()).cpu(), torch.isnan(x))
    assert torch.isfinite(s).all()
    # groups without a NaN: the bytes that they have anyway
    same = ~torch.isnan(x).view(5, 3, 128).any(-1)
    assert torch.equal(s.cpu()[same], clean_s.cpu()[same])
    bytes_ = lambda t: t.view(torch.uint8).view(5, 3, 128).cpu()[same]
    assert torch.equal(bytes_(q), bytes_(clean_q))


# about 3, 20 and 64 rows per expert: quantised while loading (with an alignment at hand) or before, and
# the GEMMs for few and for many rows
@pytest.mark.parametrize("T", [12, 80, 256])
@pytest.mark.parametrize("shuffled", [False, True])
@pytest.mark.parametrize("aligned", [False, True])
def test_layer(dev, T, shuffled, aligned):
    from dlcompiler_amd.kernels.fused_moe import ALIGN_BLOCK, fused_moe_fp8, shuffle_moe_weight
    from dlcompiler_amd.kernels.moe_gating import moe_align_block_size

    H, I, E, k = 384, 256, 8, 2
    g = torch.Generator().manual_seed(T)
    x = torch.randn((T, H), generator=g).to(torch.bfloat16)
    w1, s1 = ofp8.block_quant_weight(torch.randn((E, 2 * I, H), generator=g) * 0.05)
    w2, s2 = ofp8.block_quant_weight(torch.randn((E, H, I), generator=g) * 0.05)
    tw, ids = og.topk_softmax(torch.randn((T, E), generator=g), k)
    bad = x.clone()
    bad[3, 7] = bad[T - 1, 300] = NAN
    ref = ofm.fused_moe_fp8(bad, w1, s1, w2, s2, tw, ids)
    rows = torch.isnan(ref).any(1)
    assert torch.equal(rows.nonzero().flatten(), torch.tensor([3, T - 1])) and torch.isnan(ref[rows]).all()
    x, bad, w1, s1, w2, s2, tw, ids = (t.to(dev) for t in (x, bad, w1, s1, w2, s2, tw, ids))
    if shuffled:
        w1, w2 = shuffle_moe_weight(w1), shuffle_moe_weight(w2)
    slots, _, _, counts = moe_align_block_size(ids, ALIGN_BLOCK, E, return_counts=True)
    run = lambda t: fused_moe_fp8(t, w1, s1, w2, s2, tw, ids, k, weights_shuffled=shuffled,
                                  alignment=(slots, counts) if aligned else None).cpu()
    out, clean = run(bad), run(x)
    assert torch.isnan(out[rows]).all()
    assert torch.equal(out[~rows], clean[~rows]) and torch.isfinite(clean).all()
