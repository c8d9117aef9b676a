"""Products over experts by items of up to four units of 64 rows: the tile of 64 MI rows by 256 columns (128 of a gated pair)
whose two groups of waves take turns.  Its sums run over k as in the tile kernel, so its bits are the tile kernel's."""
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


def order(ops, counts, unit=64, item_units=4):
    """A token per pair, experts in turn with counts[e] tokens each, in a mixed order."""
    ids = torch.tensor([e for e, n in enumerate(counts) for _ in range(n)], dtype=torch.int32)
    ids = ids[torch.randperm(len(ids), generator=torch.Generator().manual_seed(7))]
    return ops.moe_align(ids[:, None].contiguous().to(DEV), len(counts), unit, "bfloat16", item_units=item_units)


# rows per expert: items of 1, 2, 3 and 4 units, full and with padding, an item of one row behind full ones, an empty expert
COUNTS = [1, 63, 64, 65, 129, 192, 0, 255, 256, 257, 700]


def test_items_of_four_units(ops):
    """From one workgroup and, from 8,192 pairs on, from several: an expert's row tiles four at a time."""
    for counts in (COUNTS, [3000, 0, 1, 5000, 191]):
        st, _slot, te, nt = order(ops, counts)
        units, items = nt.tolist()
        of = [-(-n // 64) for n in counts]
        assert units == sum(of) and te[:units].tolist() == [e for e, n in enumerate(of) for _ in range(n)]
        first = [sum(of[:e]) for e in range(len(of))]
        assert te[st.numel() // 64:][:items].tolist() == [first[e] + u for e, n in enumerate(of) for u in range(0, n, 4)]


@pytest.mark.parametrize("item_units", [2, 4])
@pytest.mark.parametrize("unit", [1, 2047, 2048, 2112, 4096])
def test_items_of_any_unit(ops, unit, item_units):
    """A unit is a number of rows, small or large, whatever its items hold."""
    counts = [1, 2049, 0, 9000, 4096]
    st, slot, te, nt = order(ops, counts, unit, item_units)
    of = [-(-n // unit) for n in counts]
    first = [sum(of[:e]) for e in range(len(of))]
    units, items = nt.tolist()
    assert st.numel() % unit == 0 and units == sum(of) and te[:units].tolist() == [e for e, n in enumerate(of) for _ in range(n)]
    assert te[st.numel() // unit:][:items].tolist() == [first[e] + u for e, n in enumerate(of) for u in range(0, n, item_units)]
    assert sorted(slot.flatten().tolist()) == [first[e] * unit + i for e, n in enumerate(counts) for i in range(n)]


@pytest.mark.parametrize("form", [{}, {"shared_size": 128}, {"sigmoid_scores": True, "renormalize": True}, {"score_correction": True, "identity": 2},
                                  {"gated": False}, {"expert_size": 4104}])
def test_the_feed_forward_asks_for_items_of_four(ops, monkeypatch, form):
    """Every kind of routed experts has its row order list items of up to four units where four suit, else of two (both give the same
    results, so that only the order shows it)."""
    from types import SimpleNamespace
    from turboquant_cpp_amd.parts.ffn import SparseMoE
    form = dict({"expert_size": 4096}, **form)
    part = SparseMoE(128, 5, 2, **form)
    for i, (name, spec) in enumerate(part.param_specs().items()):
        setattr(part, name, drawn(spec.shape, i, 0.1))
    part.prepare(DEV, "bfloat16")
    seen, route = [], ops.route
    monkeypatch.setattr(ops, "route", lambda *a, **k: seen.append(route(*a, **k)) or seen[-1])
    # (beside the shared expert's tiles, as tall as they are, items of four from 88 rows per expert on, whatever their number)
    for T, per in ((2100, 4), (900, 4 if "shared_size" in form else 2), (215, 2)):
        x = drawn((T, 128), 50)
        part.forward(x, x.float(), SimpleNamespace(act="bfloat16"))
        ids, _w, _g, st, _slot, _te, nt = seen.pop()
        of = [-(-int((ids == e).sum()) // 64) for e in range(5)]
        assert nt.tolist() == [sum(of), sum(-(-n // per) for n in of)]
        assert T == 215 or max(of) > 2


def test_a_unit_of_half_a_thousand_million_rows(ops):
    """What says that there are queues is no number of rows: an order of 2 GB, one unit with one row."""
    st, slot, te, nt = order(ops, [1], 1 << 29, 2)
    assert nt.tolist() == [1, 1] and te.tolist() == [0, 0] and slot.tolist() == [[0]]
    assert st.numel() == 1 << 29 and st[0] == 0 and (st[1:] == -1).all()
    ids = torch.zeros((1, 1), dtype=torch.int32, device=DEV)
    out = torch.zeros(64, dtype=torch.int32, device=DEV)
    for bad in (0, -1, ops.ORDER_QUEUES, ops.ORDER_QUEUES + 63, ops.ORDER_QUEUES + ops.ITEMS_OF_FOUR + 65):
        assert ops.library("bfloat16").tq_moe_align(ids.data_ptr(), 1, 1, 1, bad, 64, out.data_ptr(), out.data_ptr(), out.data_ptr(), out.data_ptr(),
                                                    torch.cuda.current_stream().cuda_stream) == -1


# k: 2, 3, 4, 5 and 9 steps of 64 (the rings hold 2 to 4 tiles); columns: less than a wave's 32, no multiple of 8, one more than a tile
@pytest.mark.parametrize("K,N", [(128, 24), (192, 100), (256, 129), (320, 256), (576, 263)])
@pytest.mark.parametrize("gated", [True, False])
def test_products_by_items_of_four(ops, K, N, gated):
    T, E = sum(COUNTS), len(COUNTS)
    st, _slot, te, nt = order(ops, COUNTS)
    x, w = drawn((T, K), 1), drawn((E, N, K), 2, 0.1)
    w2 = drawn((E, N, K), 3, 0.1) if gated else None
    live = st >= 0
    bias = torch.randn(N, generator=torch.Generator().manual_seed(4)).to(DEV)
    forms = [dict(w2=w2, out_act=True, activation=a, **more) for a in ("silu", "gelu_tanh") for more in ({}, {"pair_limit": 0.5}, {"bias": bias})] if gated \
        else [dict(out_act=True), dict(), dict(out_act=True, activation="gelu", act_alone=True), dict(bias=bias), dict(out_act=True, bias=bias.bfloat16())]
    for form in forms:
        got, want = (ops.gemm(x, w, "bfloat16", a_rows=st, tile_group=te, n_tiles=nt, tile_rows=rows, **form)
                     for rows in (64 + ops.TILE_PAIRS, 64))
        assert torch.equal(got[live], want[live]), form
    # and the formula: a sum of K products of bfloat16 factors is off by at most K roundings of 32 bits to its largest partial sum
    if not gated:
        tokens, expert = st[live].long(), te[torch.nonzero(live)[:, 0] // 64].long()
        got = ops.gemm(x, w, "bfloat16", a_rows=st, tile_group=te, n_tiles=nt, tile_rows=64 + ops.TILE_PAIRS)[live].double()
        for e in range(E):
            rows = expert == e
            a, b = x[tokens[rows]].double(), w[e].double()
            assert ((got[rows] - a @ b.T).abs() <= K * 2.0 ** -24 * (a.abs() @ b.abs().T)).all()


# a result whose rows stand further apart than it is wide: by whole runs of 16 bytes, and not
@pytest.mark.parametrize("N,ldc", [(200, 208), (200, 203), (263, 264), (256, 512)])
@pytest.mark.parametrize("out_act", [True, False])
def test_rows_in_place_and_a_wider_result(ops, N, ldc, out_act):
    """The second product reads row m for row m.  What padding holds does not matter, and neither its rows nor what lies beside a row
    of the result are written."""
    K, act = 192, "bfloat16"
    st, _slot, te, nt = order(ops, COUNTS)
    live = st >= 0
    h, w = drawn((st.numel(), K), 4), drawn((len(COUNTS), N, K), 5, 0.1)
    h[~live] = float("nan")
    lib, outs = ops.library(act), []
    for rows in (64 + ops.TILE_PAIRS, 64):
        out = torch.full((st.numel(), ldc), 7.5, dtype=torch.bfloat16 if out_act else torch.float32, device=DEV)
        assert lib.tq_gemm_mfma(h.data_ptr(), K, st.data_ptr(), 0, w.data_ptr(), None, N * K, te.data_ptr(), nt.data_ptr(), None, 0,
                                out.data_ptr(), ldc, int(out_act), st.numel(), N, K, rows, 1, 0, torch.cuda.current_stream().cuda_stream) == 0
        outs.append(out)
    got, want = outs
    assert torch.equal(got, want) and got[live].isfinite().all()
    assert (got[~live] == 7.5).all() and (got[:, N:] == 7.5).all()


# the second product: fewer rows than a tile, more than one row of tiles; k in one run and (5,632 beside 192) in several, the last shorter
@pytest.mark.parametrize("T,K,N,K2,N2", [(65, 192, 100, 128, 130), (300, 256, 263, 640, 72), (777, 192, 64, 5632, 200), (515, 128, 40, 2112, 256)])
@pytest.mark.parametrize("gated", [True, False])
def test_a_product_beside_the_experts(ops, T, K, N, K2, N2, gated):
    """Both products of gemm_pair in one launch: the experts' rows bit for bit as alone, the other's as unit by unit in one run of k, and
    its partial sums in as many runs as it says, each within the rounding of its sum and of the bias added to the first."""
    st, _slot, te, nt = order(ops, COUNTS)
    x, w = drawn((sum(COUNTS), K), 1), drawn((len(COUNTS), N, K), 2, 0.1)
    a, b = drawn((T, K2), 6), drawn((N2, K2), 7, 0.1)
    first = dict(a=x, w=w, a_rows=st, tile_group=te, n_tiles=nt, tile_rows=64 + ops.TILE_PAIRS)
    second = dict(a=a, w=b)
    if gated:
        first.update(w2=drawn(w.shape, 3, 0.1), out_act=True, activation="silu", pair_limit=0.7)
        second.update(w2=drawn(b.shape, 8, 0.1), out_act=True, activation="gelu_tanh")
    else:
        bias = torch.randn(N2, generator=torch.Generator().manual_seed(9)).to(DEV)
        second.update(partial_sums=True, bias=bias)
    y1, y2 = ops.gemm_pair(dict(first), dict(second), "bfloat16")
    want = ops.gemm(first.pop("a"), first.pop("w"), "bfloat16", **first)
    assert torch.equal(y1[st >= 0], want[st >= 0])
    if gated:
        alone = ops.gemm(a, b, "bfloat16", w2=second["w2"], out_act=True, activation="gelu_tanh")
        assert torch.equal(y2, alone)
    else:
        runs = y2.shape[0]
        assert (runs > 1) == (K2 >= 2048)
        per = -(-(K2 // 64) // runs) * 64
        for z in range(runs):
            az, bz = a[:, z * per:(z + 1) * per].double(), b[:, z * per:(z + 1) * per].double()
            exact = az @ bz.T + (bias.double() if z == 0 else 0.0)      # the bias goes with the first run alone
            assert ((y2[z].double() - exact).abs() <= K2 * 2.0 ** -24 * (az.abs() @ bz.abs().T) + 2.0 ** -23 * exact.abs()).all()


# rows, columns, k and the height of the tiles that suits (0: it goes in others): each height; the fewest rows of each rule (65 and 129, 513 to
# 1,024, 1,025); a few columns past a tile, less than a wave's 32; two and three steps of k; a last tile of one row; columns and a k left to the tile kernel
@pytest.mark.parametrize("M,N,K,rows", [(1025, 24, 2048, 64), (1025, 40, 128, 64), (1100, 4200, 128, 128), (700, 3104, 512, 64), (65, 66048, 512, 128), (1030, 4104, 192, 128),
                                        (515, 16600, 512, 192), (130, 33000, 576, 192), (2049, 6400, 192, 256), (3001, 5000, 128, 256), (2999, 8000, 320, 192),
                                        (1025, 4100, 128, 0), (1025, 24, 128, 0)])
def test_products_of_one_matrix(ops, M, N, K, rows):
    """Plain products in these tiles are the tile kernel's bits (which gathered rows keep to), with a bias, into either type, through an
    activation and in runs of k; and the formula's values."""
    assert ops.library("bfloat16").tq_gemm_phases_rows(M, N, K, 0, 1) == rows
    a, w = drawn((M, K), 1), drawn((N, K), 2, 0.1)
    every = torch.arange(M, dtype=torch.int32, device=DEV)
    bias = torch.randn(N, generator=torch.Generator().manual_seed(4)).to(DEV)
    for form in (dict(), dict(bias=bias), dict(out_act=True, bias=bias.bfloat16()), dict(out_act=True, activation="gelu", act_alone=True, bias=bias)):
        with ops.own_products(True):
            assert torch.equal(ops.gemm(a, w, "bfloat16", **form), ops.gemm(a, w, "bfloat16", a_rows=every, **form)), form
    runs = ops.gemm(a, w, "bfloat16", bias=bias, partial_sums=True)
    x, y = a.double(), w.double()
    assert ((runs.double().sum(0) - (x @ y.T + bias.double())).abs() <= (K + 4) * 2.0 ** -24 * (x.abs() @ y.abs().T + bias.double().abs())).all()


@pytest.mark.parametrize("M,N,K,rows", [(65, 16504, 128, 128), (1500, 2104, 192, 128), (129, 20000, 128, 192), (200, 16504, 192, 256), (2049, 5000, 192, 192),
                                        (1025, 8, 128, 64), (1500, 2100, 192, 0)])
def test_gated_pairs_of_one_matrix(ops, M, N, K, rows):
    """As above, of two matrices behind each other and apart, with and without a limit."""
    assert ops.library("bfloat16").tq_gemm_phases_rows(M, N, K, 1, 1) == rows
    a, both = drawn((M, K), 1), drawn((2 * N, K), 2, 0.1)
    w, w2, every = both[:N], both[N:], torch.arange(M, dtype=torch.int32, device=DEV)
    for form in (dict(out_act=True), dict(), dict(out_act=True, pair_limit=0.6), dict(out_act=True, activation="gelu_tanh")):
        with ops.own_products(True):
            want = ops.gemm(a, w, "bfloat16", w2=w2, a_rows=every, **form)
            assert torch.equal(ops.gemm(a, w, "bfloat16", w2=w2.clone(), **form), want), form
            assert torch.equal(ops.gemm(a, w, "bfloat16", w2=w2, **form), want), form


def test_runs_of_k_of_one_matrix(ops):
    """Many rows of a long k in two runs and more, each within the rounding of its sum, the bias in the first alone."""
    for M, N, K in ((1025, 2048, 8448), (2100, 1024, 4160), (1100, 1504, 6400)):
        a, w = drawn((M, K), 1), drawn((N, K), 2, 0.1)
        bias = torch.randn(N, generator=torch.Generator().manual_seed(4)).to(DEV)
        got = ops.gemm(a, w, "bfloat16", bias=bias, partial_sums=True)
        runs = got.shape[0]
        assert runs > 1 and runs == ops.library("bfloat16").tq_gemm_mfma_splits(M, N, K)
        per = -(-(K // 64) // runs) * 64
        for z in range(runs):
            x, y = a[:, z * per:(z + 1) * per].double(), w[:, z * per:(z + 1) * per].double()
            want = x @ y.T + (bias.double() if z == 0 else 0.0)
            assert ((got[z].double() - want).abs() <= (per + 4) * 2.0 ** -24 * (x.abs() @ y.abs().T + bias.double().abs())).all()


# tiles: fewer than the chip's compute units, some for each of them, and crowded experts that leave one die with more than the others
@pytest.mark.parametrize("counts,N", [([70] * 5, 300), ([130, 1, 64, 200] * 20, 1300), ([2900] + [65] * 30, 1300), ([300] * 9 + [0] * 40 + [60], 4100)])
@pytest.mark.parametrize("gated", [True, False])
def test_tiles_dealt_from_a_queue(ops, counts, N, gated):
    """An order's first two products take their tiles from its queues, a third one a tile to a workgroup, in a captured graph all of
    them: the same results, alone and with another product beside, which the order's next use of its memory does not change."""
    K = 320
    st, _slot, te, nt = order(ops, counts)
    live, T = st >= 0, sum(counts)
    x, w = drawn((T, K), 1), drawn((len(counts), N, K), 2, 0.1)
    form = dict(w2=drawn(w.shape, 3, 0.1), out_act=True) if gated else dict()
    run = lambda nt, rows: ops.gemm(x, w, "bfloat16", a_rows=st, tile_group=te, n_tiles=nt, tile_rows=rows, **form)[live]
    want = run(nt, 64)
    assert nt.queues.left == [2, 1]
    for left in ([2], [], []):
        assert torch.equal(run(nt, 64 + ops.TILE_PAIRS), want) and nt.queues.left == left
    assert torch.equal(run(nt.clone(), 64 + ops.TILE_PAIRS), want)      # numbers without queues
    for _ in range(3):
        nt = order(ops, counts)[3]
        a, b = drawn((700, 128), 6), drawn((N, 128), 7, 0.1)
        first = dict(a=x, w=w, a_rows=st, tile_group=te, n_tiles=nt, tile_rows=64 + ops.TILE_PAIRS, **form)
        second = dict(a=a, w=b, **(dict(w2=drawn(b.shape, 8, 0.1), out_act=True) if gated else {}))
        y1, y2 = ops.gemm_pair(first, dict(second), "bfloat16")
        assert nt.queues.left == [2] and torch.equal(y1[live], want)
        assert torch.equal(y2, ops.gemm(second.pop("a"), second.pop("w"), "bfloat16", **second))
    nt = order(ops, counts)[3]
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = ops.gemm(x, w, "bfloat16", a_rows=st, tile_group=te, n_tiles=nt, tile_rows=64 + ops.TILE_PAIRS, **form)
    assert nt.queues.left == [2, 1]
    for _ in range(3):
        got.zero_()
        graph.replay()
        assert torch.equal(got[live], want)


def test_what_names_no_queue_is_refused(ops):
    st, _slot, te, nt = order(ops, [70])
    h, w, out = drawn((st.numel(), 128), 1), drawn((1, 64, 128), 2), torch.empty((st.numel(), 64), device=DEV)
    call = lambda rows: ops.library("bfloat16").tq_gemm_mfma(h.data_ptr(), 128, st.data_ptr(), 0, w.data_ptr(), None, 64 * 128, te.data_ptr(), nt.data_ptr(),
                                                            None, 0, out.data_ptr(), 64, 0, st.numel(), 64, 128, rows, 1, 0, torch.cuda.current_stream().cuda_stream)
    assert call(64 + ops.TILE_QUEUE) != 0 and call(64 + ops.TILE_PAIRS + 3 * ops.TILE_QUEUE) != 0


@pytest.mark.parametrize("hint", [2048, 4096, 64 + 1024 + 2048, 1 << 30])
def test_a_hint_of_any_size_is_ignored(ops, hint):
    """Products of one matrix take no notice of the rows of a tile, alone and in pairs of few rows."""
    for M in (5, 300, 1100):
        a, w, w2, bias = drawn((M, 128), 1), drawn((256, 128), 2), drawn((128, 128), 3), drawn((256,), 4)
        assert torch.equal(ops.gemm(a, w, "bfloat16", out_act=True, bias=bias, tile_rows=hint), ops.gemm(a, w, "bfloat16", out_act=True, bias=bias))
        if M <= 16:
            both = [ops.gemm_pair(dict(a=a, w=w, tile_rows=r), dict(a=a, w=w2, tile_rows=r), "bfloat16") for r in (16, hint)]
            assert torch.equal(both[0][0], both[1][0]) and torch.equal(both[0][1], both[1][1])


# rows and columns of each kernel of plain products: streaming, tiles of few workgroups, the tile kernel, these tiles by 16 bytes and by pairs
@pytest.mark.parametrize("M,N", [(3, 264), (40, 264), (300, 264), (1025, 261), (1100, 264)])
def test_rounding_to_16_bits(ops, M, N):
    """Results of 16 bits are the nearest, of two as near the even one: biases of 32 bits beside rows of zeros.  Among them both sides of
    ties, the largest that stay finite, subnormal numbers of 16 bits, infinities and NaN."""
    bits = [h << 16 | low for h in (0x3F80, 0x3F81, 0x0000, 0x0001, 0x007F, 0x0080, 0x7F7F, 0x7F7E, 0x4123) for low in (0, 1, 0x7FFF, 0x8000, 0x8001, 0xFFFF)]
    bits += [b | 1 << 31 for b in bits] + [0x7F800000, 0xFF800000, 0x7F800001, 0x7FC00000, 0xFFFFFFFF]
    bias = torch.tensor([bits[i % len(bits)] for i in range(N)], dtype=torch.int64).to(torch.int32).view(torch.float32)
    a, w = torch.zeros(M, 128, dtype=torch.bfloat16, device=DEV), drawn((N, 128), 2)
    with ops.own_products(True):
        got = ops.gemm(a, w, "bfloat16", bias=bias.to(DEV), out_act=True).cpu()
    want = bias.bfloat16().expand(M, N)
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.nan_to_num(7.0, 8.0, 9.0), want.nan_to_num(7.0, 8.0, 9.0))


# Values of a wave of 32 columns beside each other: its form of the gate hangs on whether one of them is 87 or more in size.  To the ends of
# the shorter form; where an exponential one rounding off gives the next float; zeros and the smallest normal floats; NaN; both forms'
# values, and infinities, in one wave.
ROUNDED = [-73.06429, -30.360157, -60.720314, -40.9672, -57.091183, -15.313667, -74.74527, -61.679783, -46.15222, -76.990776, -54.57411,
           -7.829238, -29.549843, -19.86942, -79.04454, 79.04454]
GATED = [[s * v for v in (86.99, 86.5, 86.0, 85.5, 84.0, 83.0, 80.0, 70.0) for s in (1, -1)] * 2,
         ROUNDED * 2,
         [0.0, -0.0, 1e-30, -1e-30, 2.0 ** -126, -(2.0 ** -126), 2.0 ** -110, -(2.0 ** -120)] * 4,
         [float("nan")] * 32,
         [0.0, -0.0, 86.5, -86.5, 87.0, -87.0, 88.0, -88.5, 1e5, -1e5, 1e-30, float("inf"), float("-inf"), float("nan"), 3.0, -3.0] * 2,
         [(i - 15.5) * 0.05 for i in range(32)],
         [(i - 15.5) * 3.0 for i in range(32)],
         [(-1) ** i * 2.0 ** (-i) for i in range(32)]]


@pytest.mark.parametrize("out_act", [True, False])
def test_the_gate_over_its_whole_range(ops, out_act):
    """silu in the tiles' epilogue is the tile kernel's, bit for bit: each value of GATED, and 127 smaller multiples of it, in waves of the
    shorter form, of the longer one, and of values that would take either.  And it is the formula's."""
    x = torch.tensor(GATED).flatten()
    M, K, N = 1280, 128, x.numel()
    a, w, w2 = torch.zeros(M, K), torch.zeros(N, K), torch.zeros(N, K)
    a[:, :3] = (1.0 - torch.arange(M) % 128 / 256.0)[:, None]
    rest = x
    for k in range(3):      # a float is three of 16 bits
        w[:, k] = rest.bfloat16().float()
        rest = torch.where(x.isfinite(), rest - w[:, k], 0.0)
    a[:, 3] = w2[:, 3] = 1.0
    a, w, w2 = (t.to(torch.bfloat16).to(DEV) for t in (a, w, w2))
    assert ops.library("bfloat16").tq_gemm_phases_rows(M, N, K, 1, 1)
    with ops.own_products(True):
        got = ops.gemm(a, w, "bfloat16", w2=w2, out_act=out_act)
        want = ops.gemm(a, w, "bfloat16", w2=w2, out_act=out_act, a_rows=torch.arange(M, dtype=torch.int32, device=DEV))
        z = ops.gemm(a, w, "bfloat16")
    finite = x.isfinite() & (x.abs() > 1e-29)
    assert torch.equal(z[0].cpu()[finite], x[finite])
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.nan_to_num(), want.nan_to_num())
    z = z.double().cpu()
    exact, inside = z * torch.sigmoid(z), z.abs() < 87
    # a rounding to 16 bits; in 32 bits those of the exponential (one place of its own), the sum and the quotient
    bound = exact.abs() * (2.0 ** -8 if out_act else 3 * 2.0 ** -23) + 2.0 ** -126
    assert inside.sum() > 0.8 * inside.numel() and ((got.cpu().double() - exact).abs() <= bound)[inside].all()
