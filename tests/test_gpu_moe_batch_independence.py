"""A token's result does not depend on where the other tokens of its batch are routed: in the streaming grouped GEMM,
and in the tiled one, the order of a row's sums follows from its experts alone."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# mean rows per expert of 16 / 8 experts: 16-, 32- and 64-row tiles, the tiled fp8 kernel; K split and not; K of 4096
@pytest.mark.parametrize("T,H,I,E", [(20, 2048, 1408, 16), (60, 2048, 1408, 16), (120, 2048, 1408, 16),
                                     (400, 640, 384, 16), (10, 4096, 512, 8), (60, 4096, 512, 8), (20, 1152, 896, 64)])
@pytest.mark.parametrize("form", ["fp8", "fp8_row_major", "bf16"])
def test_other_tokens_routed_elsewhere(dev, T, H, I, E, form):
    from dlcompiler_amd.kernels.fused_moe import fused_moe, fused_moe_fp8, shuffle_moe_weight

    k, mine = 2, 6
    g = torch.Generator(device=dev).manual_seed(T + H)
    x = torch.randn((T, H), generator=g, device=dev).to(torch.bfloat16)
    w1, w2 = (torch.randn(s, generator=g, device=dev).mul_(0.05).to(torch.bfloat16) for s in ((E, 2 * I, H), (E, H, I)))
    weights = torch.rand((T, k), generator=g, device=dev)
    ids = torch.rand((T, E), generator=g, device=dev).argsort(-1)[:, :k]
    if form != "bf16":
        w1, w2 = (w.mul_(50).to(torch.float8_e4m3fn) for w in (w1, w2))
        s1, s2 = (torch.rand((E, w.shape[1] // 128, w.shape[2] // 128), generator=g, device=dev) * 0.03 + 0.01
                  for w in (w1, w2))
        if form == "fp8":
            w1, w2 = shuffle_moe_weight(w1), shuffle_moe_weight(w2)

    def first_rows(ids):
        if form == "bf16":
            return fused_moe(x, w1, w2, weights, ids, k)[:mine].clone()
        return fused_moe_fp8(x, w1, s1, w2, s2, weights, ids, k, weights_shuffled=form == "fp8")[:mine].clone()

    want = first_rows(ids)
    for first in (0, E // 2):  # all the others to two experts, ahead of and behind these tokens' own
        other = ids.clone()
        other[mine:] = torch.tensor([first, first + 1], device=dev)
        assert torch.equal(first_rows(other), want)
