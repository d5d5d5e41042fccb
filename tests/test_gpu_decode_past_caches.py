"""Paged decode of more keys than go through the caches: K comes in whole lines there, two operand rows a line.  Short
contexts beside filling ones, whose table rows name one page over and over; slots past the contexts, which share their
pages, hold NaN."""
import pytest
import torch

from oracle import attention as oa

pytestmark = pytest.mark.gpu

LAYOUTS = {
    "contiguous": lambda c: c,
    "head_major": lambda c: c.transpose(1, 2).contiguous().transpose(1, 2),
    "gaps": lambda c: torch.cat([c, torch.full_like(c, float("nan"))], -1)[..., :c.shape[-1]],
}


def _inputs(lens, fillers, filling, page, hq, hkv, d, dtype, layout):
    """The sequences of ``lens``, one of a full page, and ``fillers`` of ``filling`` keys, all on that page."""
    g = torch.Generator().manual_seed(sum(lens) + page + d)
    ks, vs = ([torch.randn((n, hkv, d), generator=g).to(dtype) for n in [*lens, page]] for _ in range(2))
    q = torch.randn((len(lens) + 1 + fillers, hq, d), generator=g).to(dtype)
    kc, vc, table = oa.make_paged_cache(ks, vs, page, dtype=dtype)
    wide = torch.full((q.shape[0], max(-(-filling // page), table.shape[1])), int(table[-1, 0]), dtype=table.dtype)
    wide[:len(lens), :table.shape[1]] = table[:-1]
    kv_len = torch.tensor([*lens, page] + [filling] * fillers)
    return q, LAYOUTS[layout](kc), LAYOUTS[layout](vc), wide, kv_len


def _run(dev, q, kc, vc, table, kv_len, window=None, cap=None):
    from dlcompiler_amd.kernels.paged_attention import paged_attention_fwd

    o = torch.full_like(q, 9.0).to(dev)
    # (to a device as it is: .to() would keep the strides of dense views only)
    kd, vd = (torch.empty_strided(c.shape, c.stride(), dtype=c.dtype, device=dev).copy_(c) for c in (kc, vc))
    paged_attention_fwd(q.to(dev), kd, vd, o, table.to(dev), torch.arange(len(kv_len), device=dev),
                        torch.ones(len(kv_len), dtype=torch.int64, device=dev), kv_len.to(dev), 1, window_size=window,
                        logit_softcapping=cap)
    return o.cpu()


def _check(dev, lens, fillers, filling, page, hq, hkv, d, dtype, layout, window, cap):
    q, kc, vc, table, kv_len = _inputs(lens, fillers, filling, page, hq, hkv, d, dtype, layout)
    visible = sum(min(n, window + 1) if window else n for n in kv_len.tolist())
    assert visible * hkv * d * 4 > 128 * 2**20 and len(kv_len) * min(filling, window or filling) * hkv * d * 4 > 256 * 2**20
    n = len(lens)
    ref = oa.paged_decode(q[:n], kc, vc, table[:n], kv_len[:n], window=window, softcap=cap)
    # 16-bit P and outputs: 2^-8 of values of a few units
    torch.testing.assert_close(_run(dev, q, kc, vc, table, kv_len, window, cap)[:n].float(), ref.float(), rtol=2e-2, atol=2e-2)


@pytest.mark.parametrize("lens", [[1, 2, 3, 15, 16, 17, 31, 0], [33, 47, 63, 64, 65, 96, 127, 129], [511, 513, 1000, 2049]])
@pytest.mark.parametrize("page", [16, 48, 64])
@pytest.mark.parametrize("hq,hkv,d,dtype", [(8, 2, 128, torch.bfloat16), (16, 1, 64, torch.float16), (40, 2, 128, torch.float16),
                                            (4, 4, 64, torch.bfloat16)])
@pytest.mark.parametrize("window,cap", [(None, None), (600000, None), (None, 5.0)])
def test_wide_tables(dev, lens, page, hq, hkv, d, dtype, window, cap):
    _check(dev, lens, 1, 150 * 2**20 // (hkv * d * 4), page, hq, hkv, d, dtype, "contiguous", window, cap)


@pytest.mark.parametrize("layout", ["head_major", "gaps"])
@pytest.mark.parametrize("page", [16, 48])
@pytest.mark.parametrize("hq,hkv,d", [(8, 2, 128), (8, 4, 64)])
def test_strided_caches(dev, layout, page, hq, hkv, d):
    _check(dev, [1, 17, 64, 95, 700, 1111], 1, 150 * 2**20 // (hkv * d * 4), page, hq, hkv, d, torch.bfloat16, layout, None, None)


# the window starts inside a 16-key sub-tile, at its edge, and before the context
@pytest.mark.parametrize("page", [16, 64])
@pytest.mark.parametrize("layout", ["contiguous", "head_major"])
@pytest.mark.parametrize("hkv,d,fillers", [(8, 128, 21), (4, 64, 86)])
def test_windows(dev, page, layout, hkv, d, fillers):
    _check(dev, [3002, 3003, 3009, 3018, 3034, 3100, 3517, 3001, 40], fillers, 3333, page, 2 * hkv, hkv, d, torch.bfloat16,
           layout, 3001, 6.0 if page == 16 else None)


@pytest.mark.parametrize("hq,hkv,d", [(32, 8, 128), (160, 4, 64)])
def test_the_keys_decide_and_not_the_table(dev, hq, hkv, d):
    """Few keys take the same loads, and add in the same order, in tables with room for less and for more than the
    caches hold (which split them alike: pieces of 128 and of 512 keys)."""
    lens, page = [1100, 3000, 40, 777, 2222, 1, 64, 500], 64
    q, kc, vc, table, kv_len = _inputs(lens, 0, page, page, hq, hkv, d, torch.bfloat16, "contiguous")
    results = []
    for room in (230, 290):
        wide = torch.zeros((len(kv_len), room * 2**20 // (len(kv_len) * page * hkv * d * 4)), dtype=table.dtype)
        wide[:, :table.shape[1]] = table
        results.append(_run(dev, q, kc, vc, wide, kv_len))
    assert torch.equal(*results)


@pytest.mark.parametrize("hkv,d", [(2, 128), (4, 64)])
def test_replays_follow_the_keys(dev, hkv, d):
    """Captured with few keys and replayed with more than go through the caches, and back."""
    from dlcompiler_amd.kernels.paged_attention import paged_attention_fwd

    filling = 300 * 2**20 // (hkv * d * 4)
    q, kc, vc, table, kv_len = (t.to(dev) for t in _inputs([1100, 40, 3000], 1, filling, 64, 4 * hkv, hkv, d, torch.bfloat16,
                                                           "contiguous"))
    start, new, o = torch.arange(5, device=dev), torch.ones(5, dtype=torch.int64, device=dev), torch.empty_like(q)

    def call():
        paged_attention_fwd(q, kc, vc, o, table, start, new, kv_len, 1)

    kv_len[-1] = 500
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call()
    for keys in (filling, 500, filling // 2 - 40, filling // 3, filling):
        kv_len[-1] = keys
        call()
        eager = o.clone()
        o.fill_(7.0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(o, eager), keys
