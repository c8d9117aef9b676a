"""Products of up to 16 rows a tile with k in whole lines of 64 and columns in whole tiles of 16: the kernel without a test per load.
One column less goes to the general streaming kernel, which splits k alike and adds in the same order: the same bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    from turboquant_cpp_amd.csrc import ops as module
    return module


def drawn(shape, seed, scale=1.0):
    gen = torch.Generator().manual_seed(seed)
    return (torch.randn(shape, generator=gen) * scale).to(torch.bfloat16).to(DEV)


def forms(w2, pair_limit=None):
    if w2 is None:
        return [dict(out_act=True), dict(), dict(out_act=True, activation="relu2", act_alone=True)]
    return [dict(w2=w2, out_act=True), dict(w2=w2), dict(w2=w2, out_act=True, activation="gelu_tanh", pair_limit=0.5)]


# k: one line; fewer lines than a round; a round and a remainder over two waves; shares of sixteen waves of which one has none;
# columns: one tile, a few, every compute unit a workgroup of 16 columns, one and a half, many
@pytest.mark.parametrize("K,N", [(64, 16), (192, 48), (1408, 208), (5632, 512), (2048, 4096), (128, 6144), (320, 17408)])
@pytest.mark.parametrize("M", [1, 7, 8, 9, 16])
@pytest.mark.parametrize("gated", [True, False])
def test_one_matrix(ops, K, N, M, gated):
    x, w, w2 = drawn((M, K), 1), drawn((N, K), 2, 0.1), drawn((N, K), 3, 0.1)
    bias = torch.randn(N, generator=torch.Generator().manual_seed(4)).to(DEV)
    for form, b in [(f, b) for f in forms(w2 if gated else None) for b in (None, bias)]:
        got = ops.gemm(x, w, "bfloat16", bias=b, **form)
        less = dict(form, w2=w2[:N - 1]) if gated else form
        want = ops.gemm(x, w[:N - 1], "bfloat16", bias=None if b is None else b[:N - 1], **less)
        assert torch.equal(got[:, :N - 1], want), form
    if not gated:      # and the formula, all columns: K products of bfloat16 factors and K - 1 sums in 32 bits
        exact = x.double() @ w.double().t()
        bound = K * 2.0 ** -23 * (x.double().abs() @ w.double().abs().t())
        assert ((ops.gemm(x, w, "bfloat16").double() - exact).abs() <= bound).all()


def rows_of(ops, counts, T):
    """counts[e] tokens for expert e, in a mixed order; the row order in units of 16."""
    ids = torch.tensor([e for e, n in enumerate(counts) for _ in range(n)], dtype=torch.int32)
    ids = ids[torch.randperm(len(ids), generator=torch.Generator().manual_seed(7))].view(T, -1)
    st, _slot, te, nt = ops.moe_align(ids.contiguous().to(DEV), len(counts), 16, "bfloat16")
    return dict(a_rows=st, tile_group=te, n_tiles=nt, tile_rows=16)


# experts with one row, eight, nine, sixteen, seventeen (a second tile of one), none; more row tiles than the narrow columns are for
@pytest.mark.parametrize("counts,T", [([0, 1, 0, 0], 1), ([1, 8, 0, 9, 16, 17, 1], 52), ([1] * 20 + [12], 16)])
@pytest.mark.parametrize("K,N", [(64, 16), (1408, 240), (2048, 1408)])
def test_experts_and_a_second_product_beside_them(ops, counts, T, K, N):
    E = len(counts)
    order = rows_of(ops, counts, T)
    live = order["a_rows"] >= 0
    x, w, w2 = drawn((T, K), 1), drawn((E, N, K), 2, 0.1), drawn((E, N, K), 3, 0.1)
    wl, w2l = w[:, :N - 1].contiguous(), w2[:, :N - 1].contiguous()
    for gated in (True, False):
        for form in forms(w2 if gated else None):
            less = dict(form, w2=w2l) if gated else form
            got, want = ops.gemm(x, w, "bfloat16", **order, **form), ops.gemm(x, wl, "bfloat16", **order, **less)
            assert torch.equal(got[live][:, :N - 1], want[live]), form
    # rows by place, as the second product of an expert takes them; what padding holds must not matter
    h = drawn((order["a_rows"].numel(), K), 5)
    h[~live] = float("nan")
    got, want = (ops.gemm(h, m, "bfloat16", gather=False, **order) for m in (w, wl))
    assert torch.equal(got[live][:, :N - 1], want[live]) and got[live].isfinite().all()
    if T > 16:
        return
    s, s2 = drawn((48, K), 6, 0.1), drawn((48, K), 8, 0.1)
    for a, b in ((dict(w2=w2, out_act=True), dict(w2=s2, out_act=True)), ({}, {}), ({}, dict(partial_sums=True))):
        al = dict(a, w2=w2l) if a else a
        bl = dict(b, w2=s2[:47]) if "w2" in b else b
        got = ops.gemm_pair(dict(a=x, w=w, **order, **a), dict(a=x, w=s, **b), "bfloat16")
        want = ops.gemm_pair(dict(a=x, w=wl, **order, **al), dict(a=x, w=s[:47], **bl), "bfloat16")
        assert torch.equal(got[0][live][:, :N - 1], want[0][live])
        assert torch.equal(got[1][..., :47], want[1])
