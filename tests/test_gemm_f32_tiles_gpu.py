"""32-bit products in tiles: k that is no multiple of a tile's 16, rows and columns that do not fill a tile, runs of k, gated pairs in tiles of
their own width, and experts' row tiles, against sums in 64 bits within the rounding of the sum."""
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


def within(got, a, b):
    """K roundings of 32 bits to the largest partial sum."""
    a, b = a.double(), b.double()
    return ((got.double() - a @ b.T).abs() <= a.shape[1] * 2.0 ** -24 * (a.abs() @ b.abs().T)).all()


@pytest.mark.parametrize("M,N,K", [(17, 64, 4), (33, 130, 12), (64, 200, 16), (65, 127, 20), (129, 128, 36), (300, 260, 48), (200, 1, 1004),
                                   (40, 2048, 2044)])
def test_products_in_tiles(ops, M, N, K):
    a, w, w2, bias = drawn((M, K), 1), drawn((N, K), 2, 0.2), drawn((N, K), 3, 0.2), drawn((N,), 4)
    assert within(ops.gemm(a, w, "float32"), a, w)
    got = ops.gemm(a, w, "float32", bias=bias).double()
    assert (got - (a.double() @ w.double().T + bias.double())).abs().max() <= (K + 1) * 2.0 ** -24 * ((a.abs().double() @ w.abs().double().T).max() + bias.abs().max())
    u, v = (a.double() @ x.double().T for x in (w, w2))
    bound = K * 2.0 ** -24 * (a.abs().double() @ w.abs().double().T)
    bound2 = K * 2.0 ** -24 * (a.abs().double() @ w2.abs().double().T)
    got = ops.gemm(a, w, "float32", w2=w2, activation="relu2").double()
    # relu(u)^2 v: an error of e in u and f in v moves it by at most (2 |u| e + e^2)(|v| + f) + u^2 f, and three roundings
    exact = u.clamp(min=0) ** 2 * v
    assert ((got - exact).abs() <= (2 * u.abs() * bound + bound ** 2) * (v.abs() + bound2) + u ** 2 * bound2 + 4 * 2.0 ** -24 * exact.abs() + 1e-30).all()


@pytest.mark.parametrize("N", [4194240, 4194241, 8388480])
def test_gated_pairs_of_as_many_columns_as_the_grid_has_room_for(ops, N):
    """The last width in tiles of 64 columns, the first in tiles of 128 and the last of those: the same bits, column by column."""
    M, K = 65, 4
    a, w, w2 = drawn((M, K), 1), drawn((4096, K), 2, 0.2), drawn((4096, K), 3, 0.2)
    many = [m.repeat(-(-N // 4096), 1)[:N].contiguous() for m in (w, w2)]
    want = ops.gemm(a, w, "float32", w2=w2)
    got = ops.gemm(a, many[0], "float32", w2=many[1])
    whole = N // 4096 * 4096
    assert (got[:, :whole].view(M, -1, 4096) == want[:, None]).all() and torch.equal(got[:, whole:], want[:, :N - whole])
    with pytest.raises(Exception, match="not supported"):
        ops.gemm(a, w.repeat(2049, 1)[:8388481].contiguous(), "float32", w2=w2.repeat(2049, 1)[:8388481].contiguous())


def test_an_experts_pair_in_either_width(ops):
    """Experts' gated pairs go in tiles of 64 columns and, where those are many, of 128: a column's bits are the same."""
    K, N, E = 36, 8192, 3
    ids = torch.tensor([0] * 700 + [1] * 65 + [2], dtype=torch.int32)[torch.randperm(766, generator=torch.Generator().manual_seed(7))].to(DEV)
    st, _slot, te, nt = ops.moe_align(ids[:, None].contiguous(), E, 64, "float32")
    assert st.numel() // 64 * (N // 128) <= 5 * 512 < st.numel() // 64 * (4 * N // 128)
    x, w, w2 = drawn((766, K), 1), drawn((E, N, K), 2, 0.2), drawn((E, N, K), 3, 0.2)
    order = dict(a_rows=st, tile_group=te, n_tiles=nt, tile_rows=64)
    want = ops.gemm(x, w, "float32", w2=w2, **order)
    got = ops.gemm(x, w.repeat(1, 4, 1), "float32", w2=w2.repeat(1, 4, 1), **order)
    live = st >= 0
    assert (got[live].view(-1, 4, N) == want[live][:, None]).all()


@pytest.mark.parametrize("K,N", [(12, 40), (52, 129), (64, 128)])
@pytest.mark.parametrize("gated", [True, False])
def test_experts_in_row_tiles(ops, K, N, gated):
    """Every expert's rows as a product of its own gives them: the sums' order hangs on k alone."""
    counts = [1, 64, 0, 65, 130, 700]
    ids = torch.tensor([e for e, n in enumerate(counts) for _ in range(n)], dtype=torch.int32)
    ids = ids[torch.randperm(len(ids), generator=torch.Generator().manual_seed(7))].to(DEV)
    st, _slot, te, nt = ops.moe_align(ids[:, None].contiguous(), len(counts), 64, "float32")
    x, w = drawn((len(ids), K), 1), drawn((len(counts), N, K), 2, 0.2)
    w2 = drawn((len(counts), N, K), 3, 0.2) if gated else None
    got = ops.gemm(x, w, "float32", w2=w2, a_rows=st, tile_group=te, n_tiles=nt, tile_rows=64)
    for e, n in enumerate(counts):
        if n > 64:      # (up to 64 rows a plain product may be cut into runs of k)
            rows = (st >= 0) & (te[:st.numel() // 64].repeat_interleave(64) == e)
            rows[64 * int(nt[0]):] = False
            want = ops.gemm(x[st[rows].long()].contiguous(), w[e].contiguous(), "float32", w2=w2[e].contiguous() if gated else None)
            assert torch.equal(got[rows], want)
            if not gated:
                assert within(got[rows], x[st[rows].long()], w[e])
