"""The native host path of each operator against the general Python path on the same arguments: bit
for bit the same results, and arguments it does not cover still go through."""
import pytest
import torch

import dlcompiler_amd as d
from dlcompiler_amd import _lib

pytestmark = pytest.mark.gpu


class _Declines:
    """Stands for the native module: covers nothing."""

    def __getattr__(self, name):
        return lambda *args: None


def _r(*shape, dtype=torch.bfloat16):
    return torch.randn(shape, device="cuda:0").to(dtype)


def _ints(values, dtype=torch.int32):
    return torch.tensor(values, dtype=dtype, device="cuda:0")


def _rotary(T, strided=False, dtype=torch.bfloat16):
    q = _r(T, 8, 128, dtype=dtype)[:, ::2] if strided else _r(T, 4, 64, dtype=dtype)
    D = q.size(-1)
    return d.apply_rotary_pos_emb, (q, _r(T, 2, D, dtype=dtype), _r(T, D, dtype=dtype), _r(T, D, dtype=dtype))


def _fill(idx):
    table = _ints([[3, 1, 9], [0, 2, 9]], idx)[:, :2]  # rows of a wider table
    kc, vc = _r(4, 16, 2, 64), _r(4, 16, 2, 64)

    def call(k, v):
        caches = kc.clone(), vc.clone()
        assert d.fill_kv_cache(k, v, *caches, _ints([0, 3]), _ints([3, 1], idx), _ints([20, 17]), 3, table) is None
        return caches

    return call, (_r(4, 2, 64), _r(4, 2, 64))


def _paged(idx, decode, window=None, cap=None):
    table, kv = _ints([[3, 1], [0, 2]], idx), _ints([20, 31], idx)
    lens = [1, 1] if decode else [3, 2]
    q, k, v = _r(sum(lens), 4, 64), _r(4, 16, 2, 64), _r(4, 16, 2, 64)

    def call(q):
        o = torch.full_like(q, 7.0)
        assert d.paged_attention_fwd(q, k, v, o, table, _ints([0, lens[0]]), _ints(lens), kv, max(lens), window, None,
                                     cap) is None
        return o

    return call, (q,)


def _prefill(idx):
    def call(q, k, v):
        o = torch.full_like(q, 7.0)
        assert d.context_attention_fwd(q, k, v, o, _ints([0, 5], idx), _ints([5, 70]), 70) is None
        return o

    return call, (_r(75, 4, 64), _r(75, 2, 64), _r(75, 2, 64))


def _moe(fp8, ids_type=torch.int64, aligned=False, shard=False, renorm=False, strided=False):
    from dlcompiler_amd.kernels.fused_moe import ALIGN_BLOCK

    T, H, I, E, k = 9, 256, 128, 4, 2
    x = _r(T, 2 * H)[:, :H] if strided else _r(T, H)
    weights, ids = torch.rand((T, k), device="cuda:0"), torch.randint(0, 8 if shard else E, (T, k), device="cuda:0")
    ids = ids.to(ids_type)
    experts = 8 if shard else None
    alignment = None
    if aligned:
        slots, _, _, counts = d.moe_align_block_size(ids, ALIGN_BLOCK, experts or E, return_counts=True)
        alignment = slots, counts
    w1, w2 = _r(E, 2 * I, H) * 0.05, _r(E, H, I) * 0.05
    if fp8:
        quantised = [w.to(torch.float8_e4m3fn) for w in (w1, w2)]
        s1, s2 = torch.rand((E, 2, 2), device="cuda:0"), torch.rand((E, 2, 1), device="cuda:0")
        return (lambda x: d.fused_moe_fp8(x, quantised[0], s1, quantised[1], s2, weights, ids, k, 4 if shard else 0, experts,
                                          renorm, alignment=alignment)), (x,)
    return (lambda x: d.fused_moe(x, w1, w2, weights, ids, k, 4 if shard else 0, experts, renorm,
                                  alignment=alignment)), (x,)


CASES = {
    "silu": lambda: (d.silu_and_mul, (_r(3, 2 * 40),)),
    "silu_out": lambda: (d.silu_and_mul, (_r(3, 2 * 41, dtype=torch.float32), _r(3, 50, dtype=torch.float32)[:, :41])),
    "silu_columns_strided": lambda: (d.silu_and_mul, (_r(80, 3).t(),)),
    "rms": lambda: (d.rms_norm, (_r(2, 5, 128), _r(128))),
    "rms_rows_strided": lambda: (d.rms_norm, (_r(5, 256)[:, :128], _r(128), 1e-5)),
    "add_rms": lambda: (d.add_rms_norm, (_r(5, 72, dtype=torch.float16), _r(72, dtype=torch.float16), 1e-6,
                                         _r(5, 72, dtype=torch.float16))),
    "rotary": lambda: _rotary(5),
    "rotary_strided": lambda: _rotary(5, strided=True),
    "rotary_f32": lambda: _rotary(1, dtype=torch.float32),
    "fill_32": lambda: _fill(torch.int32),
    "fill_64": lambda: _fill(torch.int64),
    "fill_16": lambda: _fill(torch.int16),  # converted by the general path
    "decode": lambda: _paged(torch.int32, True),
    "decode_window_cap": lambda: _paged(torch.int64, True, 8, 20.0),
    "chunked": lambda: _paged(torch.int64, False),
    "chunked_window_cap": lambda: _paged(torch.int32, False, 8, 20),
    "prefill_32": lambda: _prefill(torch.int32),
    "prefill_64": lambda: _prefill(torch.int64),
    "gate": lambda: (lambda x: d.moe_topk_softmax_align(x, 3, 16, return_counts=True), (_r(37, 12),)),
    "gate_one_token": lambda: (lambda x: d.moe_topk_softmax_align(x, 1, 128, 8, False), (_r(1, 8, dtype=torch.float32),)),
    "moe": lambda: _moe(False),
    "moe_aligned_renormalised": lambda: _moe(False, torch.int32, aligned=True, renorm=True),
    "moe_shard": lambda: _moe(False, shard=True),
    "moe_rows_strided": lambda: _moe(False, strided=True),   # copied by the general path
    "moe_ids_16": lambda: _moe(False, torch.int16),          # converted by the general path
    "moe_fp8": lambda: _moe(True),
    "moe_fp8_aligned": lambda: _moe(True, torch.int32, aligned=True),
    "moe_fp8_rows_strided_shard": lambda: _moe(True, shard=True, strided=True),
    "gate_columns_strided": lambda: (lambda x: d.moe_topk_softmax_align(x, 2, 64), (_r(12, 9).t(),)),
}


@pytest.mark.parametrize("name", list(CASES))
def test_native_path_equals_general_path(dev, name, monkeypatch):
    torch.manual_seed(3)
    call, args = CASES[name]()
    native = call(*args)
    native = native if isinstance(native, tuple) else (native,)
    native = [t.clone() for t in native]
    if not name.startswith("gate"):  # (its general path ends in the two separate operators, below)
        monkeypatch.setattr(_lib, "_host", _Declines())
        general = call(*args)
    else:
        k, block = {"gate": (3, 16), "gate_one_token": (1, 128), "gate_columns_strided": (2, 64)}[name]
        general = d.moe_topk_softmax(args[0], k, name != "gate_one_token")
        general += d.moe_align_block_size(general[1], block, args[0].shape[1], return_counts=len(native) == 6)
    general = general if isinstance(general, tuple) else (general,)
    assert len(native) == len(general)
    for a, b in zip(native, general):
        assert a.dtype == b.dtype and a.shape == b.shape and torch.equal(a, b)


def test_side_stream_and_errors(dev):
    x = _r(64, 2 * 256)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        y = d.silu_and_mul(x)
    side.synchronize()
    assert torch.equal(y, d.silu_and_mul(x))
    with pytest.raises(AssertionError):
        d.silu_and_mul(x[0])
    with pytest.raises(TypeError):
        d.silu_and_mul(x.double())
    with pytest.raises(ValueError):
        d.rms_norm(x, torch.ones(512, dtype=x.dtype))
    with pytest.raises(_lib.DlblasHipError):
        d.context_attention_fwd(_r(4, 2, 20), _r(4, 2, 20), _r(4, 2, 20), _r(4, 2, 20), _ints([0]), _ints([4]), 4)
