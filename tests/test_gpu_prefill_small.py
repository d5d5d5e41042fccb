"""GPU parity of prefill launches too small to fill the chip (64-row workgroups, two key groups) and just
past the limit, the head-size-96 instance, and sliding windows whose open tiles skip the mask."""
import pytest
import torch

from oracle import attention as oatt

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lens", [[129], [1, 64, 65, 700], [200, 33], [2000], [513, 513, 513]])
@pytest.mark.parametrize("Hq,Hkv,D", [(8, 2, 64), (4, 4, 96), (16, 4, 128), (8, 1, 80), (6, 2, 104)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_packed(dev, lens, Hq, Hkv, D, dtype):
    from dlcompiler_amd.kernels.prefill_attention import context_attention_fwd

    g = torch.Generator().manual_seed(sum(lens) + D)
    n = sum(lens)
    q, k, v = (torch.randn((n, h, D), generator=g).to(dtype) for h in (Hq, Hkv, Hkv))
    start = torch.tensor([sum(lens[:i]) for i in range(len(lens))])
    o = torch.full_like(q, 3.0).to(dev)
    context_attention_fwd(q.to(dev), k.to(dev), v.to(dev), o, start.to(dev), torch.tensor(lens).to(dev), max(lens))
    ref = oatt.prefill_attention(q, k, v, start, torch.tensor(lens))
    torch.testing.assert_close(o.cpu().float(), ref.float(), rtol=2e-2, atol=2e-2)


@pytest.mark.parametrize("new,history", [([16, 3], [300, 0]), ([1, 130, 64], [900, 63, 2000]), ([300], [1500]), ([40] * 9, [500] * 9),
                                         ([100], [3000]), ([33, 7], [2500, 10]), ([1, 2], [1300, 0])])
@pytest.mark.parametrize("page", [16, 64])
@pytest.mark.parametrize("Hq,Hkv,D", [(8, 2, 96), (8, 1, 128), (4, 4, 64)])
@pytest.mark.parametrize("window,cap", [(None, None), (200, None), (64, 15.0), (None, 15.0)])
def test_paged(dev, new, history, page, Hq, Hkv, D, window, cap):
    from dlcompiler_amd.kernels.paged_attention import paged_attention_fwd

    g = torch.Generator().manual_seed(sum(new) + page + D)
    ctx = [a + b for a, b in zip(new, history)]
    ks, vs = ([torch.randn((c, Hkv, D), generator=g).to(torch.bfloat16) for c in ctx] for _ in range(2))
    kc, vc, table = oatt.make_paged_cache(ks, vs, page)
    q = torch.randn((sum(new), Hq, D), generator=g).to(torch.bfloat16)
    start = torch.tensor([sum(new[:i]) for i in range(len(new))])
    o = torch.full_like(q, 3.0).to(dev)
    paged_attention_fwd(q.to(dev), kc.to(dev), vc.to(dev), o, table.to(dev), start.to(dev), torch.tensor(new).to(dev),
                        torch.tensor(ctx).to(dev), max(new), window_size=window, logit_softcapping=cap)
    ref = oatt.paged_prefill(q, kc, vc, table, start, torch.tensor(new), torch.tensor(ctx), window=window, softcap=cap)
    torch.testing.assert_close(o.cpu().float(), ref.float(), rtol=2e-2, atol=2e-2)
