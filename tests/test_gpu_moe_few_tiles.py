"""16-bit grouped GEMMs whose column tiles are fewer than the CUs, by twos, fours and eights: row tiles of 16 to 128 rows
with the waves side by side, in two pairs and all splitting K, on either side of the limits between them."""
import pytest
import torch

from oracle import fused_moe as ofm
from oracle import moe_gating as og

pytestmark = pytest.mark.gpu

# (tokens, hidden, intermediate, output width, experts, k), for 256 CUs.  20 tiles of 128 columns: K split four ways, 16
# rows, then in two pairs, 32 and 64; 64 side by side; 128
SIZES = [(T, 192, 576, 1040, 4, 2) for T in (20, 24, 25, 60, 130, 400, 1500, 4000)]
# 128 and (half the experts) 64 tiles: 32 and 64 rows in two pairs, 128 rows
SIZES += [(T, 128, 448, 784, 32, 4) for T in (60, 130, 200, 420, 700)]
# 160 and 224, side by side, 32, 64 and 128 rows, and 80 and 112; 256 and 160, 128 and 80
SIZES += [(T, 64, 640, 1552, 32, 4) for T in (57, 150, 153, 288, 290, 416, 420)] + [(200, 64, 1024, 1040, 32, 4)]
# 288 and 448, where the down GEMM alone goes to 128 rows, and 144 and 224
SIZES += [(T, 64, 1152, 3336, 32, 4) for T in (170, 190, 300)]

# half the experts: 80 gate_up tiles of 32 rows side by side, 112 down tiles of 128 rows, then of 64, which a long K hides
SIZES += [(540, 64, 640, 1552, 32, 4), (700, 64, 640, 1552, 32, 4), (700, 64, 1024, 1552, 32, 4)]


@pytest.mark.parametrize("T,H,I,O,E,k", SIZES)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("local", [False, True])
def test_few_tiles(dev, T, H, I, O, E, k, dtype, local):
    from dlcompiler_amd.kernels.fused_moe import fused_moe, shuffle_moe_weight

    g = torch.Generator().manual_seed(T + O)
    n, first = (E // 2, E // 2) if local else (E, 0)
    x = torch.randn((T, H), generator=g).to(dtype)
    w1, w2 = (torch.randn(s, generator=g).mul_(0.05).to(dtype) for s in ((n, 2 * I, H), (n, O, I)))
    tw, ids = og.topk_softmax(torch.randn((T, E), generator=g), k, renormalize=False)
    ref = ofm.fused_moe(x, w1, w2, tw, ids, expert_offset=first, renormalize=True).double()
    x, w1, w2, tw, ids = (t.to(dev) for t in (x, w1, w2, tw, ids))
    out = fused_moe(x, w1, w2, tw, ids, k, first, E, True)
    # two 16-bit roundings of the intermediate and one of the slot rows, 2^-9 each in bf16, and their sum's
    err = ((out.cpu().double() - ref).norm() / ref.norm()).item()
    assert err < 5e-3, err
    if O % 16 == 0:
        assert torch.equal(out, fused_moe(x, shuffle_moe_weight(w1), shuffle_moe_weight(w2), tw, ids, k, first, E, True,
                                          weights_shuffled=True))
