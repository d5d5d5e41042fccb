"""fused_moe divides routing weights by their token's sum where it stores the slot rows, loading up to four or eight of a
token's weights at once: the same bits as with the weights divided in advance, summed in the order of the slots."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [1, 2, 3, 4, 5, 7, 8, 9, 16, 17])
@pytest.mark.parametrize("rows", [3, 20, 80])  # per expert: tiles of 16 rows, of 32, tall ones (fp8: the tiled kernel)
@pytest.mark.parametrize("fp8", [False, True])
def test_same_bits_as_divided_weights(dev, k, rows, fp8):
    from dlcompiler_amd.kernels.fused_moe import fused_moe, fused_moe_fp8

    E, H, I = 20, 256, 128
    T = max(1, rows * E // k)
    g = torch.Generator(device=dev).manual_seed(k)
    x = torch.randn((T, H), generator=g, device=dev, dtype=torch.bfloat16)
    w1 = torch.randn((E, 2 * I, H), generator=g, device=dev, dtype=torch.bfloat16) * 0.1
    w2 = torch.randn((E, H, I), generator=g, device=dev, dtype=torch.bfloat16) * 0.1
    ids = torch.rand((T, E), generator=g, device=dev).argsort(dim=1)[:, :k].to(torch.int32).contiguous()
    tw = torch.rand((T, k), generator=g, device=dev) + 0.1
    total = torch.zeros(T, device=dev)
    for j in range(k):
        total = total + tw[:, j]
    divided = (tw / total[:, None]).contiguous()
    if fp8:
        s1, s2 = torch.full((E, 2 * I // 128, H // 128), 0.25, device=dev), torch.full((E, H // 128, I // 128), 0.5, device=dev)
        w1, w2 = w1.to(torch.float8_e4m3fn), w2.to(torch.float8_e4m3fn)
        got = fused_moe_fp8(x, w1, s1, w2, s2, tw, ids, k, renormalize=True)
        want = fused_moe_fp8(x, w1, s1, w2, s2, divided, ids, k, renormalize=False)
    else:
        got = fused_moe(x, w1, w2, tw, ids, k, renormalize=True)
        want = fused_moe(x, w1, w2, divided, ids, k, renormalize=False)
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
