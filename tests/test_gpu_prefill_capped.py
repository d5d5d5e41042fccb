"""GPU parity of soft-capped prefill over a history: tiles under the diagonal, which have no mask, beside those on it
and at the window's edge; scores far below the cap, and some of a wave beyond it; each shape of workgroup."""
import pytest
import torch

from oracle import attention as oatt

pytestmark = pytest.mark.gpu

# 16-bit inputs and outputs, P rounded to 16 bits before the second product: 2^-8 per rounding of values of
# order one, a few of which add up
TOL = {"rtol": 2e-2, "atol": 2e-2}


def _check(dev, Hq, Hkv, D, page, new, history, cap, window, dtype=torch.bfloat16):
    from dlcompiler_amd.kernels.paged_attention import paged_attention_fwd

    g = torch.Generator().manual_seed(Hq + D + sum(new))
    ctx = [a + b for a, b in zip(new, history)]
    ks, vs = ([torch.randn((c, Hkv, D), generator=g).to(dtype) for c in ctx] for _ in range(2))
    kc, vc, table = oatt.make_paged_cache(ks, vs, page)
    q = torch.randn((sum(new), Hq, D), generator=g)
    q[::7] *= 6.0  # some queries of a wave beyond the polynomial's range
    q = q.to(dtype)
    start = torch.tensor([sum(new[:i]) for i in range(len(new))])
    o = torch.full_like(q, 3.0).to(dev)
    paged_attention_fwd(q.to(dev), kc.to(dev), vc.to(dev), o, table.to(dev), start.to(dev), torch.tensor(new).to(dev),
                        torch.tensor(ctx).to(dev), max(new), window_size=window, logit_softcapping=cap)
    ref = oatt.paged_prefill(q, kc, vc, table, start, torch.tensor(new), torch.tensor(ctx), window=window, softcap=cap)
    torch.testing.assert_close(o.cpu().float(), ref.float(), **TOL)


@pytest.mark.parametrize("D", [64, 80, 96, 128, 160])
@pytest.mark.parametrize("page", [16, 64])
@pytest.mark.parametrize("cap", [1.5, 40.0])
@pytest.mark.parametrize("new,history,window", [([129, 64, 1], [63, 0, 192], None), ([127, 65], [129, 320], None),
                                                ([300], [200], 130), ([200, 31], [0, 500], 64)])
def test_few_row_tiles(dev, D, page, cap, new, history, window):
    _check(dev, 4, 2, D, page, new, history, cap, window)


# enough workgroups for 128-row tiles, and for heads that share them without a cap
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("cap", [1.5, 40.0])
@pytest.mark.parametrize("window", [None, 100])
def test_many_row_tiles(dev, D, cap, window):
    _check(dev, 32, 8, D, 64, [150, 64, 97] * 11, [70, 0, 130] * 11, cap, window, torch.float16)


# packed heads with split keys
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("cap", [1.5, 40.0])
def test_packed_heads(dev, D, cap):
    _check(dev, 8, 2, D, 64, [17, 3], [2500, 640], cap, None)
