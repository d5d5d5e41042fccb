"""Paged decode of long contexts in few sequences: 64- and 128-key pieces, and partials per head around the 64 that
the merge takes at a time."""
import pytest
import torch

from oracle import attention as oa

pytestmark = pytest.mark.gpu


# 64-key pieces up to 4096 keys of room and four wavefronts per CU, else 128: 1 .. 160 partials
@pytest.mark.parametrize("lens", [[1100], [4095], [4096], [4033, 3], [3, 4096], [8191], [8193], [20300], [64, 2300, 1, 700]])
@pytest.mark.parametrize("hq,hkv,d", [(4, 1, 128), (8, 4, 64), (2, 2, 96), (4, 2, 80), (2, 1, 256)])
@pytest.mark.parametrize("window", [None, 900])
def test_partials(dev, lens, hq, hkv, d, window):
    from dlcompiler_amd.kernels.paged_attention import paged_attention_fwd

    g = torch.Generator().manual_seed(sum(lens) + d)
    ks, vs = ([torch.randn((n, hkv, d), generator=g).to(torch.bfloat16) for n in lens] for _ in range(2))
    q = (2 * torch.randn((len(lens), hq, d), generator=g)).to(torch.bfloat16)
    kc, vc, table = oa.make_paged_cache(ks, vs, 64, dtype=torch.bfloat16)
    kv_len = torch.tensor(lens)
    ref = oa.paged_decode(q, kc, vc, table, kv_len, window=window)
    o = torch.full_like(q, 9.0).to(dev)
    paged_attention_fwd(q.to(dev), kc.to(dev), vc.to(dev), o, table.to(dev), torch.arange(len(lens), device=dev),
                        torch.ones(len(lens), dtype=torch.int64, device=dev), kv_len.to(dev), 1, window_size=window)
    # 16-bit P and outputs: 2^-8 of values of a few units
    torch.testing.assert_close(o.cpu().float(), ref.float(), rtol=2e-2, atol=2e-2)
