"""Choice of experts for many tokens: a token's logits are summed in one order, however many tokens there are."""
import pytest
import torch

from turboquant_cpp_amd.csrc import ops

pytestmark = pytest.mark.gpu
DEVICE = "cuda:0"


# 239 and 240 lie on both sides of the change of form; 1,002 elements are not whole groups of four; 5,120 fill the LDS, 5,124 pass it
@pytest.mark.parametrize("tokens,experts,width,shared,dtype", [
    (239, 60, 2048, True, torch.bfloat16), (240, 60, 2048, True, torch.bfloat16), (241, 60, 2048, False, torch.float32),
    (1001, 8, 1000, True, torch.bfloat16), (300, 33, 1002, True, torch.bfloat16), (2500, 130, 512, False, torch.bfloat16),
    (250, 31, 5120, True, torch.float32), (250, 31, 5124, True, torch.bfloat16),
])
def test_choice_of_many_tokens_is_that_of_a_few(tokens, experts, width, shared, dtype):
    gen = torch.Generator().manual_seed(tokens + experts)
    x = torch.randn(tokens, width, generator=gen).to(DEVICE)
    router = (torch.randn(experts, width, generator=gen) * 0.05).to(dtype).to(DEVICE)
    gate = (torch.randn(width, generator=gen) * 0.05).to(dtype).to(DEVICE) if shared else None
    bias = torch.randn(experts, generator=gen).to(DEVICE)
    ids, weights, gates = ops.router_topk(x, router, gate, 4, False, "bfloat16", bias=bias)
    for first in range(0, tokens, 100):
        few = ops.router_topk(x[first:first + 100], router, gate, 4, False, "bfloat16", bias=bias)
        assert torch.equal(ids[first:first + 100], few[0])
        assert torch.equal(weights[first:first + 100], few[1])
        if shared:
            assert torch.equal(gates[first:first + 100], few[2])
    # a logit is a sum of `width` products of about 0.05 in 32 bits: 1e-5 is far above its rounding, and softmax weights follow it
    logits = x.double() @ router.double().t() + bias.double()
    exact = torch.softmax(logits, -1).gather(1, ids.long())
    assert (weights.double() - exact).abs().max().item() < 2e-5
    best = torch.topk(logits, 4, -1).values
    assert (logits.gather(1, ids.long()) - best).abs().max().item() < 2e-5
    if shared:
        assert (gates.double() - torch.sigmoid(x.double() @ gate.double())).abs().max().item() < 2e-5
