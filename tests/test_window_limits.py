"""A sliding window larger than any context plans the same launch as none, up to the largest int."""
import pytest
import torch

from dlcompiler_amd import _lib

LARGEST = 2 ** 31 - 1


@pytest.mark.parametrize("window", [LARGEST, LARGEST - 31, 1 << 30, 16000])
@pytest.mark.parametrize("tokens,B", [(32, 1), (100, 2)])
def test_chunked_scratch(window, tokens, B):
    args = (tokens * B, B, 32, 8, 128, 128, 64, 250, tokens)
    lib = _lib.load()
    assert lib.dlb_paged_prefill_ws_bytes(*args, window) == lib.dlb_paged_prefill_ws_bytes(*args, -1) > 0


@pytest.mark.gpu
@pytest.mark.parametrize("window", [-1, LARGEST, LARGEST - 31, 3000])
def test_decode_route(dev, window):
    """2000 keys of 128 dims take the split kernel, which leaves partials in the scratch."""
    from oracle import attention as oatt

    g = torch.Generator().manual_seed(1)
    Hq, Hkv, D, page, ctx = 8, 2, 128, 16, 2000
    ks, vs = ([torch.randn((ctx, Hkv, D), generator=g).to(torch.bfloat16)] for _ in range(2))
    kc, vc, table = oatt.make_paged_cache(ks, vs, page)
    q, lens = torch.randn((1, Hq, D), generator=g).to(torch.bfloat16), torch.tensor([ctx])
    ref = oatt.paged_decode(q, kc, vc, table, lens)
    q, kc, vc, table, lens = (t.to(dev) for t in (q, kc, vc, table, lens))
    (table, lens), mask = _lib.index_arrays(table, lens)
    lib = _lib.load()
    ws_bytes = lib.dlb_paged_decode_ws_bytes(1, Hq, Hkv, D, page, table.size(1))
    ws = torch.full((-(-ws_bytes // 4),), float("nan"), device=dev)
    o = torch.empty_like(q)
    _lib.check(lib.dlb_paged_decode_attn(
        q.data_ptr(), kc.data_ptr(), vc.data_ptr(), o.data_ptr(), table.data_ptr(), lens.data_ptr(), mask, 1, Hq, Hkv,
        D, D, page, table.size(1), q.stride(0), q.stride(1), kc.stride(0), kc.stride(1), kc.stride(2), vc.stride(0),
        vc.stride(1), vc.stride(2), o.stride(0), o.stride(1), table.stride(0), D ** -0.5, window, -1.0, 0,
        ws.data_ptr(), ws.numel() * 4, _lib.current_stream_ptr(q.device)), "decode")
    torch.testing.assert_close(o.cpu().float(), ref.float(), rtol=2e-2, atol=2e-2)
    assert not torch.isnan(ws).all()
