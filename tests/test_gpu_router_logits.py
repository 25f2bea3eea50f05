"""Router logits of many tokens (several experts per wave) against one-token
calls: the same fixed summation order, so the same bits, whatever the batch."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("tokens,experts,h", [(16, 256, 2304), (64, 77, 72), (65, 256, 2304),
                                              (130, 6, 2560), (200, 33, 4096), (1100, 256, 520)])
def test_many_tokens_match_one_token_calls(tokens, experts, h, dtype):
    from local_kimi_amd.kernels import router_logits

    gen = torch.Generator(device=DEV).manual_seed(tokens + h)
    x = torch.randn(tokens, h, device=DEV, generator=gen).to(torch.bfloat16)
    w = torch.randn(experts, h, device=DEV, generator=gen).to(dtype)
    out = router_logits(x, w)
    rows = sorted({0, 1, tokens // 2, tokens - 2, tokens - 1})
    one = torch.cat([router_logits(x[t:t + 1], w) for t in rows])
    assert torch.equal(out[rows], one)
    # fp32 sums of h products: each within h ulps of the magnitudes' sum
    want = x.double() @ w.double().T
    bound = h * 2.0**-24 * (x.double().abs() @ w.double().abs().T)
    assert bool(((out.double() - want).abs() <= bound).all())
