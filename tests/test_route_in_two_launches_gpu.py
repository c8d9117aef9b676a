"""Choice and order of many tokens in one call, in two launches or in more: the numbers of the choice and of the order apart, and the choice
against 64 bits, on both sides of the lines of the rule."""
import pytest
import torch

from turboquant_cpp_amd.csrc import ops

pytestmark = pytest.mark.gpu
DEVICE = "cuda:0"


# two: whether the host's rule says two launches.  Where 2, 4 and 8 tokens go to a workgroup, and remainders; (192 experts, eight a token: the choice
# through LDS); rows of 5,120 and of 1,002, and of 10,700 (2 tokens, and from 2,049 on 1); 72 experts of which the last 18 have no matrices.  More
# launches: fewer tokens, few experts or pairs, tables of more than 65,536 counts (33 experts at 16,384 tokens) or 8 a pair, rows of 5,120 of more than
# 3,072 tokens; among them the order by 8 and by 11 to 16 workgroups and by one, units of 16, and more than 64 and 128 experts.
@pytest.mark.parametrize("tokens,experts,top,width,unit,options,two", [
    (511, 60, 4, 512, 64, {}, 0), (512, 60, 4, 512, 64, {"shared": True}, 1), (513, 60, 4, 512, 64, {}, 1), (1024, 60, 4, 512, 64, {"four": True}, 1),
    (1025, 60, 4, 512, 16, {"shared": True}, 1), (2047, 64, 2, 512, 128, {"groups": (8, 2)}, 1), (2049, 64, 8, 512, 64, {"sigmoid": True}, 1),
    (1024, 192, 8, 512, 64, {}, 1), (1027, 192, 8, 512, 32, {"bias": True}, 1), (2100, 30, 4, 5120, 64, {}, 1), (700, 31, 4, 1002, 64, {"shared": True}, 1),
    (1999, 72, 4, 512, 64, {"identity": 18}, 1), (4096, 8, 8, 512, 64, {}, 1), (13000, 33, 1, 512, 64, {}, 1), (16384, 32, 1, 512, 256, {}, 1),
    (600, 1, 1, 512, 64, {}, 0), (1025, 64, 4, 512, 64, {"ties": True}, 1), (777, 40, 4, 512, 64, {"nan": True}, 1),
    (2051, 30, 4, 10700, 64, {"shared": True}, 1), (701, 16, 2, 10700, 64, {}, 1), (1280, 15, 4, 10700, 64, {}, 0), (3073, 16, 4, 5120, 64, {}, 0),
    (16384, 33, 1, 512, 64, {}, 0), (2000, 300, 4, 512, 64, {"shared": True}, 0), (4000, 192, 3, 512, 16, {"bias": True}, 0),
    (2731, 260, 3, 512, 16, {}, 0), (8201, 72, 4, 512, 64, {"identity": 18}, 0), (3000, 7, 4, 512, 64, {}, 0), (1183, 8, 2, 512, 64, {}, 0),
    (1030, 160, 1, 512, 32, {}, 0), (13197, 64, 8, 512, 64, {"four": True}, 0),
])
@pytest.mark.parametrize("act", ["bfloat16", "float32"])
def test_choice_and_order_are_those_apart(tokens, experts, top, width, unit, options, two, act):
    assert bool(ops.library(act).tq_route_in_two(tokens, experts, "shared" in options, top, width)) is bool(two)
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
    if not set(options) - {"shared", "four"}:
        scores = torch.softmax(x.double() @ router.double().t(), -1)
        worst = torch.topk(scores, top, -1).values[:, -1:]
        chosen = scores.gather(1, ids.long())
        assert (chosen >= worst - 1e-6).all() and (ids.sort(-1).values.diff(dim=-1) > 0).all()
        assert (weights.double() - chosen).abs().max() < 2e-5
        if shared is not None:
            assert (gate.double() - torch.sigmoid(x.double() @ shared[0].double())).abs().max() < 2e-5
