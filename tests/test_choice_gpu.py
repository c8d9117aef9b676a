"""The choice of experts where a lane holds one or two of them, and beyond (general search): against logits in 64 bits with ties by the
highest index, the same whatever tokens are beside, and the order of one token's pairs as the general order gives it."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    from turboquant_cpp_amd.csrc import ops as module
    return module


def drawn(shape, seed, scale=1.0):
    return (torch.randn(shape, generator=torch.Generator().manual_seed(seed)) * scale).to(DEV)


FORMS = [dict(), dict(renormalize=True), dict(renormalize=True, sigmoid=True, weight_scale=2.5), dict(renormalize=True, groups=(4, 2)),
         dict(renormalize=True, groups=(4, 2), sigmoid=True, pair_groups=True), dict(correction=True), dict(correction=True, identity=3)]


@pytest.mark.parametrize("E", [4, 8, 60, 64, 65, 80, 128, 132])
@pytest.mark.parametrize("form", range(len(FORMS)))
def test_choice_and_order(ops, E, form):
    form = dict(FORMS[form])
    if "groups" in form and E % 4:
        pytest.skip("groups of equal size")
    H, T, topk, act = 64, 33, min(4, E // 2), "float32"
    x, router = drawn((T, H), 1), drawn((E, H), 2, 0.3)
    router[E - 1] = router[0]            # an exact tie between the first and the last expert
    shared = None if "correction" in form else drawn((1, H), 3, 0.3)
    correction = drawn((E,), 4, 0.01) if form.pop("correction", False) else None
    if correction is not None:
        correction[E - 1] = correction[0]
        form["correction"] = correction
    renorm = form.pop("renormalize", False)
    ids, weights, gate, *order = ops.route(x, router, shared, topk, renorm, 16, act, **form)
    # the scores in 64 bits
    z = x.double() @ router.double().T
    s = torch.sigmoid(z) if form.get("sigmoid") else torch.softmax(z, -1)
    by = s + correction.double() if correction is not None else s.clone() if form.get("sigmoid") else z.clone()
    by[:, 0], s[:, 0] = by[:, E - 1], s[:, E - 1]
    if "groups" in form:
        count, keep = form["groups"]
        per = by.view(T, count, -1)
        best = per.topk(2, -1).values.sum(-1) if form.get("pair_groups") and E // count > 1 else per.amax(-1)
        rank = torch.argsort(best + torch.arange(count, device=DEV) * 1e-13, -1, descending=True)[:, :keep]
        kept = torch.zeros(T, count, dtype=torch.bool, device=DEV).scatter_(1, rank, True)
        by = torch.where(kept.repeat_interleave(E // count, 1), by, -torch.inf)
    want = torch.argsort(by + torch.arange(E, device=DEV) * 1e-13, -1, descending=True)[:, :topk]
    gap = by.sort(-1, descending=True).values
    gap = torch.where(gap[:, :topk] - gap[:, 1:topk + 1] == 0.0, torch.inf, gap[:, :topk] - gap[:, 1:topk + 1])
    sure = (gap > 1e-5).all(-1)          # no two scores so close that 32 bits may order them otherwise (but for the exact tie)
    assert sure.sum() > T // 2
    assert torch.equal(ids.long()[sure], want[sure])
    w = s.gather(1, want)
    if form.get("sigmoid"):
        w = w / (w.sum(-1, keepdim=True) + 1e-20) * form.get("weight_scale", 1.0)
    elif renorm:
        w = w / w.sum(-1, keepdim=True)
    assert (weights.double() - w)[sure].abs().max() < 1e-5
    # token by token: the same bits, and the order that the general kernel makes of the same choice
    for t in range(T):
        one = ops.route(x[t:t + 1].contiguous(), router, shared, topk, renorm, 16, act, **form)
        assert torch.equal(one[0], ids[t:t + 1]) and torch.equal(one[1], weights[t:t + 1])
        if gate is not None:
            assert torch.equal(one[2], gate[t:t + 1])
        real = ids[t:t + 1].clone()
        n_real = E - form.get("identity", 0)
        if (real < n_real).all():
            st, slot, te, nt = ops.moe_align(real, E, 16, act)
            n = int(nt[0])
            half = st.numel() // 16
            assert torch.equal(one[3], st) and torch.equal(one[4], slot) and torch.equal(one[6], nt)
            assert torch.equal(one[5][:n], te[:n]) and torch.equal(one[5][half:half + n], te[half:half + n])
        else:
            assert ((one[4] < 0) == (real >= n_real)).all() and int(one[6][0]) == int((real < n_real).sum())
    nine = ops.route(x[:9].contiguous(), router, shared, topk, renorm, 16, act, **form)
    assert torch.equal(nine[0], ids[:9]) and torch.equal(nine[1], weights[:9])


@pytest.mark.parametrize("E", [8, 60, 80])
def test_logits_that_are_no_numbers(ops, E):
    """A token of NaN or infinities chooses as it does beside others, and its pairs are ordered."""
    H, topk = 64, 3
    x, router = drawn((20, H), 1), drawn((E, H), 2, 0.3)
    x[3], x[7, 0], x[11, 5] = torch.nan, torch.inf, -torch.inf
    router[1] = 0.0                        # infinity times nothing: one NaN among infinities
    for renorm in (False, True):
        ids, weights, *_ = ops.route(x, router, None, topk, renorm, 16, "float32")
        assert ((ids >= 0) & (ids < E)).all()
        for t in (0, 3, 7, 11):
            one = ops.route(x[t:t + 1].contiguous(), router, None, topk, renorm, 16, "float32")
            assert torch.equal(one[0], ids[t:t + 1]) and torch.equal(one[1].isnan(), weights[t:t + 1].isnan())
            assert ((one[4] >= 0) & (one[4] < one[3].numel())).all()


@pytest.mark.parametrize("E", [8, 60, 80, 132])
@pytest.mark.parametrize("renorm", [False, True])
def test_logits_that_are_infinite(ops, E, renorm):
    """Infinities without a NaN among them: the search by the rule, the highest index first among equals, a chosen expert then the least."""
    H, topk = 64, 3
    x, router = drawn((20, H), 1), drawn((E, H), 2, 0.3)
    router[:, 0], router[1, 0] = -router[:, 0].abs(), 0.5      # one expert at +infinity and the others at -infinity, or the other way about
    x[3, 0], x[7, 0], x[11, 5] = torch.inf, -torch.inf, torch.inf
    ids, weights, *_ = ops.route(x, router, None, topk, renorm, 16, "float32")
    z = (x.double() @ router.double().T).cpu()
    for t in (3, 7, 11):
        v, want = z[t].clone(), []
        assert v.isinf().all()
        for _ in range(topk):
            want.append(max(range(E), key=lambda e: (v[e].item(), e)))
            v[want[-1]] = -torch.inf
        one = ops.route(x[t:t + 1].contiguous(), router, None, topk, renorm, 16, "float32")
        assert ids[t].tolist() == want and one[0][0].tolist() == want and torch.equal(one[1].isnan(), weights[t:t + 1].isnan())
        assert ((one[4] >= 0) & (one[4] < one[3].numel())).all()


@pytest.mark.parametrize("E", [8, 60, 64, 80, 128, 132])
def test_corrections_that_are_no_numbers(ops, E):
    """Experts whose correction is NaN are not chosen; where all are, it is the first one, with its own score as its weight."""
    H, topk = 64, 3
    x, router = drawn((20, H), 1), drawn((E, H), 2, 0.3)
    score = torch.softmax(x.double() @ router.double().T, -1)
    for real in ([], [1], [0, E - 2, E - 1, 2]):
        correction = torch.full((E,), torch.nan, device=DEV)
        correction[real] = 0.0
        ids, weights, *_ = ops.route(x, router, None, topk, False, 16, "float32", correction=correction)
        if not real:
            assert (ids == 0).all()
        assert torch.isin(ids[:, :len(real)], torch.tensor(real or [0], dtype=torch.int32, device=DEV)).all()
        assert (weights.double() - score.gather(1, ids.long()))[:, :max(len(real), 1)].abs().max() < 1e-6
        for t in (0, 7):
            one = ops.route(x[t:t + 1].contiguous(), router, None, topk, False, 16, "float32", correction=correction)
            assert torch.equal(one[0], ids[t:t + 1]) and torch.equal(one[1], weights[t:t + 1])
