"""Choice and order of many tokens in two launches: the numbers of the choice and of the order apart, on both sides of every line of the rule."""
import pytest
import torch

from turboquant_cpp_amd.csrc import ops

pytestmark = pytest.mark.gpu
DEVICE = "cuda:0"


# tokens: where 2, 4 and 8 go to a workgroup, and remainders; (192 experts, eight a token: the choice through LDS); rows of 5,120 and of 1,002;
# 72 experts of which the last 18 have no matrices; 33 experts at 13,000 tokens are beyond the table's size, 32 at 16,384 just within
@pytest.mark.parametrize("tokens,experts,top,width,unit,options", [
    (511, 60, 4, 512, 64, {}), (512, 60, 4, 512, 64, {"shared": True}), (513, 60, 4, 512, 64, {}), (1024, 60, 4, 512, 64, {"four": True}),
    (1025, 60, 4, 512, 16, {"shared": True}), (2047, 64, 2, 512, 128, {"groups": (8, 2)}), (2049, 64, 8, 512, 64, {"sigmoid": True}),
    (1024, 192, 8, 512, 64, {}), (1027, 192, 8, 512, 32, {"bias": True}), (2100, 30, 2, 5120, 64, {}), (700, 31, 4, 1002, 64, {"shared": True}),
    (1999, 72, 4, 512, 64, {"identity": 18}), (4096, 8, 8, 512, 64, {}), (13000, 33, 1, 512, 64, {}), (16384, 32, 1, 512, 256, {}),
    (600, 1, 1, 512, 64, {}), (1025, 64, 4, 512, 64, {"ties": True}), (777, 40, 4, 512, 64, {"nan": True}),
])
@pytest.mark.parametrize("act", ["bfloat16", "float32"])
def test_choice_and_order_are_those_apart(tokens, experts, top, width, unit, options, act):
    gen = torch.Generator().manual_seed(tokens * 7 + experts)
    dtype = torch.bfloat16 if act == "bfloat16" else torch.float32
    x = torch.randn(tokens, width, generator=gen)
    router = (torch.randn(experts, width, generator=gen) * 0.05).to(dtype)
    if "ties" in options:
        router = router[:1].expand(experts, width).contiguous()
    if "nan" in options:
        x[5, 3] = float("nan")
    x, router = x.to(DEVICE), router.to(DEVICE)
    shared = (torch.randn(1, width, generator=gen) * 0.05).to(dtype).to(DEVICE) if "shared" in options else None
    identity = options.get("identity", 0)
    units = 4 if "four" in options else 2
    row_unit = ops.RowUnit(unit, units)
    if identity:
        correction = (torch.randn(experts, generator=gen) * 0.01).to(DEVICE)
        got = ops.route(x, router, None, top, False, row_unit, act, correction=correction, identity=identity)
        # the oracle's choice by corrected scores, in 64 bits
        scores = torch.softmax(x.double() @ router.double().t(), -1)
        worst = torch.topk(scores + correction.double(), top, -1).values[:, -1:]
        assert ((scores + correction.double()).gather(1, got[0].long()) >= worst - 1e-6).all()
        assert (got[1].double() - scores.gather(1, got[0].long())).abs().max() < 2e-5
        real = got[0] < experts - identity
        assert (got[2].double() - (got[1].double() * ~real).sum(-1)).abs().max() < 1e-6
        assert torch.equal(got[4] < 0, ~real)
        rows = got[4][real].long()
        assert torch.equal(got[3][rows].long(), torch.arange(tokens, device=DEVICE)[:, None].expand(tokens, top)[real])
        assert int((got[3] >= 0).sum()) == rows.numel() == rows.unique().numel()
        assert torch.equal(got[5][(rows // unit)], got[0][real])
        return
    args = {k: v for k, v in options.items() if k == "groups"}
    if "bias" in options:
        args["bias"] = torch.randn(experts, generator=gen).to(DEVICE)
    if "sigmoid" in options:
        args["sigmoid"] = True
    renormalize = "sigmoid" in options or "groups" in options
    got = ops.route(x, router, shared, top, renormalize, row_unit, act, **args)
    ids, weights, gate = ops.router_topk(x, router, shared, top, renormalize, act, **args)
    sorted_token, pair_slot, tile_expert, n_tiles = ops.moe_align(ids, experts, unit, act, units)
    assert torch.equal(got[0], ids) and torch.equal(torch.nan_to_num(got[1], -1.0), torch.nan_to_num(weights, -1.0))
    if shared is not None:
        assert torch.equal(torch.nan_to_num(got[2], -1.0), torch.nan_to_num(gate, -1.0))
    assert torch.equal(got[3], sorted_token) and torch.equal(got[4], pair_slot) and torch.equal(got[6][:2], n_tiles[:2])
    tiles, items, behind = int(n_tiles[0]), int(n_tiles[1]), sorted_token.numel() // unit
    assert torch.equal(got[5][:tiles], tile_expert[:tiles])
    assert torch.equal(got[5][behind:behind + items], tile_expert[behind:behind + items])
    if unit == 64:
        whole = got[6].queues.whole
        assert int(whole[2]) == ids.unique().numel() and int(whole[16:].abs().sum()) == 0
