"""Allocations of the native host path go through torch's dispatcher: dispatch modes see them, and the
deterministic fill of uninitialised memory reaches them."""
import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

import dlcompiler_amd as d

pytestmark = pytest.mark.gpu


class _Log(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.allocations = 0

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.allocations += func is torch.ops.aten.empty.memory_format
        return func(*args, **(kwargs or {}))


def _calls(dev):
    bf = lambda *shape: torch.randn(shape, device=dev).bfloat16()
    ints = lambda *v: torch.tensor(v, dtype=torch.int32, device=dev)
    x, w = bf(4, 128), bf(128)
    tw, ids = torch.rand((4, 2), device=dev), torch.randint(0, 4, (4, 2), device=dev)
    q, cache = bf(1, 4, 64), bf(2, 16, 2, 64)
    return {
        "silu_and_mul": (lambda: d.silu_and_mul(bf(4, 128)), 1),
        "rms_norm": (lambda: d.rms_norm(x, w), 1),
        "add_rms_norm": (lambda: d.add_rms_norm(x, w, 1e-6, x), 2),
        "rotary": (lambda: d.apply_rotary_pos_emb(bf(4, 2, 64), bf(4, 1, 64), bf(4, 64), bf(4, 64)), 2),
        "gate": (lambda: d.moe_topk_softmax_align(x, 2, 64), 1),
        "decode": (lambda: d.paged_attention_fwd(q, cache, cache, torch.empty_like(q), ints(0, 1)[None], None,
                                                 ints(1), ints(20), 1), 1),
        "moe": (lambda: d.fused_moe(x, bf(4, 256, 128), bf(4, 128, 128), tw, ids, 2), 2),
    }


@pytest.mark.parametrize("name", ["silu_and_mul", "rms_norm", "add_rms_norm", "rotary", "gate", "decode", "moe"])
def test_a_mode_sees_the_allocations(dev, name, monkeypatch):
    from dlcompiler_amd import _lib

    call, count = _calls(dev)[name]
    native, done = _lib.host(), []

    class Spy:
        """The native module, noting that it did not decline."""

        def __getattr__(self, attr):
            def entry(*args):
                before = log.allocations
                result = getattr(native, attr)(*args)
                done.append((result, log.allocations - before))
                return result
            return entry

    monkeypatch.setattr(_lib, "_host", Spy())
    with _Log() as log:
        call()
    assert len(done) == 1 and done[0][0] is not None and done[0][1] == count


def test_deterministic_fill(dev):
    logits = torch.randn((3, 5), device=dev)
    d.moe_topk_softmax_align(logits, 2, 16)
    torch.use_deterministic_algorithms(True)
    assert torch.utils.deterministic.fill_uninitialized_memory
    try:
        weights, *_ = d.moe_topk_softmax_align(logits, 2, 16)
    finally:
        torch.use_deterministic_algorithms(False)
    # the results are pieces of one byte buffer, which the fill sets to 255; the two unused words between
    # the 6 weights and the ids keep that
    words = torch.empty(0, dtype=torch.int32, device=dev).set_(weights.untyped_storage(), 6, (2,))
    assert torch.equal(words.cpu(), torch.full((2,), -1, dtype=torch.int32))
