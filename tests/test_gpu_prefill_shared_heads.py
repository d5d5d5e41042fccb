"""GPU parity of prefill where the heads of a KV group share workgroups (launches of several rounds): a
workgroup's waves take 32-query blocks in the order (block, head), so with group sizes that do not divide
the waves one workgroup holds blocks of two to four kinds.  Lengths on either side of a block, windows."""
import pytest
import torch

from oracle import attention as oatt

pytestmark = pytest.mark.gpu

# 16-bit inputs and outputs, P rounded to 16 bits before the second product: 2^-8 per rounding of values of
# order one, a few of which add up
TOL = {"rtol": 2e-2, "atol": 2e-2}


def _repeated(lens, Hq, rounds, D):
    """``lens`` over and over, until the launch has more than ``rounds`` rounds of 128-row workgroups."""
    slots = 256 * (4 if D <= 64 else 2)
    tiles = -(-max(lens) // 128) * Hq
    return lens * (rounds * slots // (tiles * len(lens)) + 1)


@pytest.mark.parametrize("Hq,Hkv,D", [(12, 2, 128), (10, 2, 64), (28, 4, 128), (24, 8, 96), (16, 1, 128), (6, 2, 72)])
@pytest.mark.parametrize("lens", [[1, 31, 32, 33, 0], [63, 64, 65, 95, 97], [129, 223, 5]])
def test_packed(dev, lens, Hq, Hkv, D):
    from dlcompiler_amd.kernels.prefill_attention import context_attention_fwd

    lens = _repeated(lens, Hq, 2, D)
    g = torch.Generator().manual_seed(sum(lens) + Hq)
    n = sum(lens)
    q, k, v = (torch.randn((n, h, D), generator=g).to(torch.bfloat16) for h in (Hq, Hkv, Hkv))
    start = torch.tensor([sum(lens[:i]) for i in range(len(lens))])
    o = torch.full_like(q, 3.0).to(dev)
    context_attention_fwd(q.to(dev), k.to(dev), v.to(dev), o, start.to(dev), torch.tensor(lens).to(dev), max(lens))
    ref = oatt.prefill_attention(q, k, v, start, torch.tensor(lens))
    torch.testing.assert_close(o.cpu().float(), ref.float(), **TOL)


@pytest.mark.parametrize("Hq,Hkv", [(40, 8), (28, 4), (16, 1), (48, 16)])
@pytest.mark.parametrize("window", [None, 40, 200])
@pytest.mark.parametrize("page", [16, 64])
def test_paged(dev, Hq, Hkv, window, page):
    from dlcompiler_amd.kernels.paged_attention import paged_attention_fwd

    D = 128
    new = _repeated([150, 65, 97, 131], Hq, 3, D)
    history = [70, 0, 333, 64] * (len(new) // 4)
    g = torch.Generator().manual_seed(Hq)
    ctx = [a + b for a, b in zip(new, history)]
    ks, vs = ([torch.randn((c, Hkv, D), generator=g).to(torch.bfloat16) for c in ctx] for _ in range(2))
    kc, vc, table = oatt.make_paged_cache(ks, vs, page)
    q = torch.randn((sum(new), Hq, D), generator=g).to(torch.bfloat16)
    start = torch.tensor([sum(new[:i]) for i in range(len(new))])
    o = torch.full_like(q, 3.0).to(dev)
    paged_attention_fwd(q.to(dev), kc.to(dev), vc.to(dev), o, table.to(dev), start.to(dev), torch.tensor(new).to(dev),
                        torch.tensor(ctx).to(dev), max(new), window_size=window)
    ref = oatt.paged_prefill(q, kc, vc, table, start, torch.tensor(new), torch.tensor(ctx), window=window)
    torch.testing.assert_close(o.cpu().float(), ref.float(), **TOL)
