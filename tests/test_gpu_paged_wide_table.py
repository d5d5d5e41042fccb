"""Chunked prefill with a block table wider than the contexts, as engines keep it: the launch is planned for
what the table has room for, the work follows the contexts."""
import pytest
import torch

from oracle import attention as oatt

pytestmark = pytest.mark.gpu


def _case(new, history, page, Hq, Hkv, D, width, dtype=torch.bfloat16):
    g = torch.Generator().manual_seed(sum(new) + page + D)
    ctx = [a + b for a, b in zip(new, history)]
    ks, vs = ([torch.randn((c, Hkv, D), generator=g).to(dtype) for c in ctx] for _ in range(2))
    kc, vc, table = oatt.make_paged_cache(ks, vs, page)
    # entries past a context name one more page, of NaN
    wide = torch.full((len(new), width), kc.shape[0], dtype=table.dtype)
    for i, c in enumerate(ctx):
        wide[i, :-(-c // page)] = table[i, :-(-c // page)]
    nan = torch.full_like(kc[:1], float("nan"))
    kc, vc = torch.cat([kc, nan]), torch.cat([vc, nan])
    q = torch.randn((sum(new), Hq, D), generator=g).to(dtype)
    start = torch.tensor([sum(new[:i]) for i in range(len(new))])
    return q, kc, vc, wide, start, torch.tensor(new), torch.tensor(ctx)


# contexts of one part, around 16 tiles of 64 keys (two parts from there on), of several parts, mixed
@pytest.mark.parametrize("new,history", [([32], [68]), ([1, 5], [959, 955]), ([1, 8], [960, 600]), ([16], [1200]),
                                         ([3, 32, 1], [0, 5000, 800]), ([100, 7], [900, 3]), ([128], [2000])])
@pytest.mark.parametrize("page,width", [(64, 512), (16, 1024)])
@pytest.mark.parametrize("Hq,Hkv,D", [(8, 2, 64), (8, 1, 128), (4, 4, 80)])
@pytest.mark.parametrize("window,cap", [(None, None), (700, None), (40, 15.0)])
def test_results(dev, new, history, page, width, Hq, Hkv, D, window, cap):
    from dlcompiler_amd.kernels.paged_attention import paged_attention_fwd

    q, kc, vc, table, start, lens, ctx = _case(new, history, page, Hq, Hkv, D, width)
    o = torch.full_like(q, 3.0).to(dev)
    paged_attention_fwd(q.to(dev), kc.to(dev), vc.to(dev), o, table.to(dev), start.to(dev), lens.to(dev),
                        ctx.to(dev), max(new), window_size=window, logit_softcapping=cap)
    ref = oatt.paged_prefill(q, kc, vc, table, start, lens, ctx, window=window, softcap=cap)
    torch.testing.assert_close(o.cpu().float(), ref.float(), rtol=2e-2, atol=2e-2)


@pytest.mark.parametrize("history,parts", [(68, 0), (928, 0), (929, 2), (1200, 2), (1505, 3)])
def test_parts_without_keys_write_nothing(dev, history, parts):
    from dlcompiler_amd import _lib

    new, Hq, Hkv, D, page, width = 32, 8, 2, 64, 64, 512
    q, kc, vc, table, start, lens, ctx = _case([new], [history], page, Hq, Hkv, D, width)
    ref = oatt.paged_prefill(q, kc, vc, table, start, lens, ctx)
    q, kc, vc, table, start, lens, ctx = (t.to(dev) for t in (q, kc, vc, table, start, lens, ctx))
    lib = _lib.load()
    ws_bytes = lib.dlb_paged_prefill_ws_bytes(new, 1, Hq, Hkv, D, D, page, width, new, -1)
    nsplit = ws_bytes // (4 * new * Hq * (D + 2))
    assert nsplit > 3
    ws = torch.full((ws_bytes // 4,), float("nan"), device=dev)
    o = torch.empty_like(q)
    (table, start, lens, ctx), mask = _lib.index_arrays(table, start, lens, ctx)
    _lib.check(lib.dlb_paged_prefill_attn_ws(
        q.data_ptr(), kc.data_ptr(), vc.data_ptr(), o.data_ptr(), table.data_ptr(), start.data_ptr(), lens.data_ptr(),
        ctx.data_ptr(), mask, 1, Hq, Hkv, D, D, page, width, new, q.stride(0), q.stride(1), kc.stride(0), kc.stride(1),
        kc.stride(2), vc.stride(0), vc.stride(1), vc.stride(2), o.stride(0), o.stride(1), table.stride(0), D ** -0.5,
        -1, -1.0, 0, new, ws.data_ptr(), ws_bytes, _lib.current_stream_ptr(q.device)), "paged prefill")
    torch.testing.assert_close(o.cpu().float(), ref.float(), rtol=2e-2, atol=2e-2)
    rows = ws[:nsplit * new * Hq * D].view(nsplit, -1)
    assert not torch.isnan(rows[:parts]).any() and torch.isnan(rows[parts:]).all()
