"""The tanh of the logit soft-cap is an fp32 function: its error, seen through the public entry point.

Two keys with scores x1, x2 a few units in the last place apart and a cap of 2^20 (scale 2^20, so that the
cap's argument is the score itself): the logits 2^20 tanh(x) differ by less than 3, the values are 1 and 0,
and the output is the weight of the first key, from which the difference of the two logits follows to
within 2^-11 / (1 - w) < 0.01.  One ulp of tanh is 0.03 (results in [0.25, 0.5)) or 0.06 ([0.5, 1))."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
CAP = 2.0 ** 20


def _pairs(lo, hi, sign, n, seed):
    """x1, x2: multiples of an fp32 ulp or two, exact as head + rest * 2^-12 with 16-bit head and rest."""
    step = 2.0 ** (-24 if hi <= 0.5 else -23 if hi <= 1.0 else -22)
    rng = np.random.default_rng(seed)
    x1 = np.round(rng.uniform(lo, hi, n) / step)
    slope = 1.0 - np.tanh(x1 * step) ** 2
    x2 = x1 + np.round(rng.uniform(-2.0, 2.0, n) / slope / step / CAP)
    return sign * x1 * step, sign * x2 * step


@pytest.mark.parametrize("lo,hi", [(0.251, 0.3), (0.3, 0.5), (0.55, 0.99), (1.01, 1.3), (1.3, 1.9)])
@pytest.mark.parametrize("sign", [1.0, -1.0])
@pytest.mark.parametrize("decode", [True, False])
def test_error_of_a_logit(dev, lo, hi, sign, decode):
    from dlcompiler_amd.kernels.paged_attention import paged_attention_fwd

    B, D, page = 1024, 64, 16
    xs = _pairs(lo, hi, sign, B, int(100 * hi))
    k = torch.zeros((B, page, 1, D), dtype=torch.float16)
    for slot, x in enumerate(xs):
        head = torch.from_numpy(x).to(torch.float16)
        rest = ((torch.from_numpy(x) - head.double()) * 2.0 ** 12).to(torch.float16)
        assert torch.equal(head.double() + rest.double() * 2.0 ** -12, torch.from_numpy(x))
        k[:, slot, 0, 0], k[:, slot, 0, 1] = head, rest
    v = torch.zeros_like(k)
    v[:, 0, 0, :] = 1.0
    new = 1 if decode else 2   # the last query sees both keys
    q = torch.zeros((B * new, 1, D), dtype=torch.float16)
    q[:, 0, 0], q[:, 0, 1] = 1.0, 2.0 ** -12
    out = torch.empty_like(q).to(dev)
    ints = lambda t: torch.as_tensor(t, dtype=torch.int32, device=dev)
    paged_attention_fwd(q.to(dev), k.to(dev), v.to(dev), out, ints(torch.arange(B)[:, None]),
                        ints(torch.arange(B) * new), ints([new] * B), ints([2] * B), new, sm_scale=CAP,
                        logit_softcapping=CAP)
    w = out[new - 1::new, 0, 0].double().cpu().numpy()
    assert w.min() > 0.05 and w.max() < 0.95
    t1, t2 = np.tanh(xs[0]), np.tanh(xs[1])
    ulps = (np.log(w / (1.0 - w)) - CAP * (t1 - t2)) / (CAP * np.spacing(np.abs(t1).astype(np.float32)).astype(np.float64))
    # Each logit: tanh to 1.41 ulp (what tanhf gives on this hardware), then one rounding in base 2 (half an
    # ulp, up to one where the factor 1.44 leaves the binade); output and difference 0.3 between them.
    # A tanh of 6 to 10 ulp exceeds this many times over in a thousand pairs.
    assert np.abs(ulps).max() < 2 * (1.41 + 1.0) + 0.3, np.abs(ulps).max()
    assert np.sqrt((ulps ** 2).mean()) < 1.2, np.sqrt((ulps ** 2).mean())
