"""The router's logits of wide rows: the same numbers however many tokens go to a workgroup."""
import pytest
import torch

from turboquant_cpp_amd.csrc import ops

pytestmark = pytest.mark.gpu
DEVICE = "cuda:0"


# rows beyond 2,560 and more than 2,048 tokens, 4 or 8 to a workgroup: 64 experts and 65, the first and the second half of a round of 2,048 tokens,
# more than 12,288 tokens of 129 and of 128 experts
@pytest.mark.parametrize("tokens,experts,width", [(2048, 65, 3072), (2049, 65, 3072), (3072, 130, 2561), (3073, 65, 3072), (3073, 64, 5120), (4097, 129, 3584),
                                                  (12288 - 1023, 129, 2570), (14337, 129, 2564), (14337, 128, 2564)])
def test_logits_of_wide_rows(tokens, experts, width):
    """A logit is summed in one order, however many tokens go to a workgroup: as for the same tokens 239 at a time; and against 64 bits."""
    gen = torch.Generator(DEVICE).manual_seed(tokens + experts)
    x = torch.randn(tokens, width, generator=gen, device=DEVICE)
    router = (torch.randn(experts, width, generator=gen, device=DEVICE) * 0.05).bfloat16()
    got = ops.router_topk(x, router, None, 4, False, "bfloat16")
    for at in (0, tokens // 2, tokens - 239):
        part = ops.router_topk(x[at:at + 239].contiguous(), router, None, 4, False, "bfloat16")
        assert torch.equal(got[0][at:at + 239], part[0]) and torch.equal(got[1][at:at + 239], part[1]), at
    scores = torch.softmax(x.double() @ router.double().t(), -1)
    worst, chosen = torch.topk(scores, 4, -1).values[:, -1:], scores.gather(1, got[0].long())
    assert (chosen >= worst - 1e-6).all() and (got[1].double() - chosen).abs().max() < 2e-5
