"""The cache of operand-order weight copies: a copy lives and dies with the weights it was made from (no GPU)."""
import gc

import torch

from dlcompiler_amd.kernels import fused_moe as fm


def _weights(memory):
    return torch.frombuffer(memory, dtype=torch.bfloat16).view(2, 16, 64)


def test_other_weights_in_the_same_memory(monkeypatch):
    monkeypatch.setattr(fm, "_OPERAND_ORDER_CACHE", {})
    memory = bytearray(torch.randn(2 * 16 * 64).bfloat16().view(torch.uint8).numpy().tobytes())
    first = _weights(memory)
    assert torch.equal(fm._operand_order_cached(first), fm.shuffle_moe_weight(first))
    memory[:] = torch.randn(2 * 16 * 64).bfloat16().view(torch.uint8).numpy().tobytes()
    where = first.data_ptr()
    del first
    gc.collect()
    second = _weights(memory)   # same address, shape and version counter
    assert second.data_ptr() == where and second._version == 0
    assert torch.equal(fm._operand_order_cached(second), fm.shuffle_moe_weight(second))
    assert len(fm._OPERAND_ORDER_CACHE) == 1   # the first one's copy went with it


def test_kept_while_unmodified(monkeypatch):
    monkeypatch.setattr(fm, "_OPERAND_ORDER_CACHE", {})
    w = torch.randn((2, 16, 64)).bfloat16()
    copy = fm._operand_order_cached(w)
    assert fm._operand_order_cached(w) is copy and fm._operand_order_cached(w.view(2, 16, 64)) is copy
    w[0, 0, 0] = 3.0
    again = fm._operand_order_cached(w)
    assert again is not copy and torch.equal(again, fm.shuffle_moe_weight(w))
