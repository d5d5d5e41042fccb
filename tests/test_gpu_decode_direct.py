"""GPU parity of paged decode around the rule that picks one launch or two: context lengths from 0 keys to
past the limits, fewer keys than wavefronts, sliding windows longer and shorter than the context,
head sizes with an instance of their own (64, 96, 128) and masked ones, groups wider than 16 heads."""
import pytest
import torch

from oracle import attention as oatt

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lens", [[0, 1, 31, 32, 33], [129, 700, 5], [701, 64], [1024] * 26, [1025] * 26, [2000, 300]])
@pytest.mark.parametrize("Hq,Hkv,D", [(8, 8, 64), (16, 4, 96), (32, 8, 128), (8, 2, 72), (40, 2, 104)])
@pytest.mark.parametrize("window,cap", [(None, None), (100, 20.0)])
def test_one_and_two_launches(dev, lens, Hq, Hkv, D, window, cap):
    from dlcompiler_amd.kernels.paged_attention import paged_attention_fwd

    g = torch.Generator().manual_seed(sum(lens) + D)
    ks, vs = ([torch.randn((n, Hkv, D), generator=g).to(torch.bfloat16) for n in lens] for _ in range(2))
    kc, vc, table = oatt.make_paged_cache(ks, vs, 16)
    q = torch.randn((len(lens), Hq, D), generator=g).to(torch.bfloat16)
    ctx = torch.tensor(lens)
    out = torch.full_like(q, 7.0).to(dev)
    paged_attention_fwd(q.to(dev), kc.to(dev), vc.to(dev), out, table.to(dev), None,
                        torch.ones(len(lens), dtype=torch.int64, device=dev), ctx.to(dev), 1,
                        window_size=window, logit_softcapping=cap)
    ref = oatt.paged_decode(q, kc, vc, table, ctx, window=window, softcap=cap)
    torch.testing.assert_close(out.cpu().float(), ref.float(), rtol=2e-2, atol=2e-2)
