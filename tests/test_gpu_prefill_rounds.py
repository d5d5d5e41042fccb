"""GPU parity of packed prefill where 64-row workgroups take several rounds, and on both sides of the rule that
prefers them: long chains in few sequences, short ones in many, one workgroup per CU and two."""
import pytest
import torch

from oracle import attention as oatt

pytestmark = pytest.mark.gpu


# (Hq, Hkv, D, lengths): 64-row with one round / two / three, 128-row for several short prompts
@pytest.mark.parametrize("Hq,Hkv,D,lens", [
    (4, 2, 128, [4095]), (16, 4, 128, [1537]), (32, 8, 128, [513]), (16, 2, 96, [2113]),
    (8, 8, 128, [300] * 8), (8, 8, 128, [300, 17, 256, 129, 300]), (16, 4, 64, [2177]), (4, 4, 72, [640] * 10),
    (32, 8, 64, [1281]), (8, 2, 64, [300] * 13), (16, 4, 64, [639, 590, 276])])
def test_packed(dev, Hq, Hkv, D, lens):
    from dlcompiler_amd.kernels.prefill_attention import context_attention_fwd

    g = torch.Generator().manual_seed(sum(lens) + D)
    n = sum(lens)
    q, k, v = (torch.randn((n, h, D), generator=g).to(torch.bfloat16) for h in (Hq, Hkv, Hkv))
    start = torch.tensor([sum(lens[:i]) for i in range(len(lens))])
    o = torch.full_like(q, 3.0).to(dev)
    context_attention_fwd(q.to(dev), k.to(dev), v.to(dev), o, start.to(dev), torch.tensor(lens).to(dev), max(lens))
    ref = oatt.prefill_attention(q, k, v, start, torch.tensor(lens))
    torch.testing.assert_close(o.cpu().float(), ref.float(), rtol=2e-2, atol=2e-2)
