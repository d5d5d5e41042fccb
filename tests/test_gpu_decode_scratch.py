"""Paged decode with a caller's scratch: one sized for a larger batch or a wider table, whose pieces are longer, also
serves smaller ones, which would rather have more of it."""
import pytest
import torch

from dlcompiler_amd import _lib
from oracle import attention as oatt

pytestmark = pytest.mark.gpu
PAGE, D = 64, 128


def _need(B, Hq, keys):
    """Partials of pieces of 128 keys."""
    return B * Hq * (keys // 128 + 2) * (D + 2) * 4 + 4 * B


# sequences, query heads, key heads, keys in the table; then the sequences and keys that the scratch is sized for
@pytest.mark.parametrize("B,Hq,Hkv,keys,sized_B,sized_keys",
                         [(2, 32, 8, 4096, 3, 4096), (16, 8, 1, 4096, 17, 4096), (1, 32, 8, 4096, 1, 5120), (3, 8, 2, 2048, 3, 2048)])
def test_smaller_calls_in_the_scratch_of_a_larger_one(dev, B, Hq, Hkv, keys, sized_B, sized_keys):
    lib, g = _lib.load(), torch.Generator().manual_seed(B + keys)
    lens = [keys - 37 * i for i in range(B)]
    ks, vs = ([torch.randn((n, Hkv, D), generator=g).to(torch.bfloat16) for n in lens] for _ in range(2))
    kc, vc, table = oatt.make_paged_cache(ks, vs, PAGE)
    q, lens = torch.randn((B, Hq, D), generator=g).to(torch.bfloat16), torch.tensor(lens)
    ref = oatt.paged_decode(q, kc, vc, table, lens)
    q, kc, vc, table, lens = (t.to(dev) for t in (q, kc, vc, table, lens))
    (table, lens), mask = _lib.index_arrays(table, lens)
    sized = lib.dlb_paged_decode_ws_bytes(sized_B, Hq, Hkv, D, PAGE, sized_keys // PAGE)
    own = lib.dlb_paged_decode_ws_bytes(B, Hq, Hkv, D, PAGE, keys // PAGE)
    assert _need(B, Hq, keys) < own
    for ws_bytes in (own, own - 4, min(sized, own), _need(B, Hq, keys), _need(B, Hq, keys) - 4):
        ws = torch.full((own // 4 + 64,), 7.0, device=dev)
        o = torch.full_like(q, 9.0)
        status = lib.dlb_paged_decode_attn(
            q.data_ptr(), kc.data_ptr(), vc.data_ptr(), o.data_ptr(), table.data_ptr(), lens.data_ptr(), mask, B, Hq,
            Hkv, D, D, PAGE, table.size(1), q.stride(0), q.stride(1), kc.stride(0), kc.stride(1), kc.stride(2),
            vc.stride(0), vc.stride(1), vc.stride(2), o.stride(0), o.stride(1), table.stride(0), D ** -0.5, -1, -1.0, 0,
            ws.data_ptr(), ws_bytes, _lib.current_stream_ptr(q.device))
        if ws_bytes < _need(B, Hq, keys):
            assert status == -4 and (o == 9.0).all()
            continue
        _lib.check(status, "decode")
        # 16-bit P and outputs: 2^-8 of values of a few units
        torch.testing.assert_close(o.cpu().float(), ref.float(), rtol=2e-2, atol=2e-2)
        assert (ws[ws_bytes // 4:] == 7.0).all()
