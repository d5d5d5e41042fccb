"""GPU parity of paged decode of one sequence, whose pieces start at fixed keys and whose page numbers come in one
vector load: contexts on either side of a piece, pages of several sizes, the longest table of the route."""
import pytest
import torch

from oracle import attention as oa

pytestmark = pytest.mark.gpu

# 16-bit inputs and outputs, P rounded to 16 bits: 2^-8 per rounding of values of order one
TOL = {"rtol": 2e-2, "atol": 2e-2}


def _run(dev, ctx, page, room, hq, hkv, d, dv=None, idx=torch.int64, softcap=None, dtype=torch.bfloat16):
    from dlcompiler_amd.kernels.paged_attention import paged_attention_fwd

    dv = dv or d
    g = torch.Generator().manual_seed(ctx + page)
    mk = lambda *shape: torch.randn(shape, generator=g).to(dtype)
    k, v, q = mk(max(ctx, 1), hkv, d)[:ctx], mk(max(ctx, 1), hkv, dv)[:ctx], mk(1, hq, d)
    kc, vc, table = oa.make_paged_cache([k], [v], page)
    blocks = max(room // page, table.shape[1])
    wide = torch.zeros((1, blocks), dtype=torch.int64)
    wide[:, :table.shape[1]] = table
    wide = torch.where(wide < 0, 0, wide)
    ref = oa.paged_decode(q, kc, vc, table, torch.tensor([ctx]), softcap=softcap)
    o = torch.full((1, hq, dv), 3.0, dtype=dtype, device=dev)
    paged_attention_fwd(q.to(dev), kc.to(dev), vc.to(dev), o, wide.to(idx).to(dev), torch.tensor([0], device=dev),
                        torch.tensor([1], device=dev), torch.tensor([ctx]).to(idx).to(dev), 1, logit_softcapping=softcap)
    torch.testing.assert_close(o.cpu().float(), ref.float(), **TOL)


@pytest.mark.parametrize("ctx", [1, 31, 32, 33, 63, 64, 65, 127, 128, 129, 513, 1000, 2047, 2048])
@pytest.mark.parametrize("page", [16, 48, 64, 128])
def test_pieces(dev, ctx, page):
    _run(dev, ctx, page, 2048, 8, 2, 128)


@pytest.mark.parametrize("hq,hkv,d,dv", [(8, 8, 64, 64), (8, 1, 96, 96), (20, 1, 128, 128), (4, 2, 72, 40)])
@pytest.mark.parametrize("idx", [torch.int32, torch.int64])
def test_heads_and_index_types(dev, hq, hkv, d, dv, idx):
    _run(dev, 1333, 64, 1536, hq, hkv, d, dv, idx, dtype=torch.float16)
    _run(dev, 700, 16, 1536, hq, hkv, d, dv, idx, softcap=20.0)


# 8 heads: 256 teams of 128-key pieces reach 32768 keys; one page more takes the general route
@pytest.mark.parametrize("room", [4096, 8192, 32768, 32768 + 64])
def test_long_tables(dev, room):
    for ctx in (room - 64, 4097, 5):
        _run(dev, ctx, 64, room, 8, 8, 128)


def test_empty(dev):
    from dlcompiler_amd.kernels.paged_attention import paged_attention_fwd

    kc = torch.randn(16, 64, 2, 128, device=dev, dtype=torch.bfloat16)
    q = torch.randn(1, 8, 128, device=dev, dtype=torch.bfloat16)
    o = torch.full_like(q, 3.0)
    paged_attention_fwd(q, kc, kc, o, torch.arange(16, device=dev)[None], torch.tensor([0], device=dev),
                        torch.tensor([1], device=dev), torch.tensor([0], device=dev), 1)
    assert (o == 0).all()
