"""The residual sum with norms, for rows that wait in registers and for those that go through LDS: lengths at the edges of the threads'
runs (256 and 512 threads, 1, 2 and 4 runs of four), one that is no multiple of four and one that is too long."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
LENGTHS = [4, 1020, 1024, 1028, 1030, 2044, 2048, 2052, 4096, 4100, 8192, 8196]


@pytest.fixture(scope="module")
def ops():
    from turboquant_cpp_amd.csrc import ops as module
    return module


def drawn(shape, seed, scale=1.0, dtype=torch.float32):
    return (torch.randn(shape, generator=torch.Generator().manual_seed(seed)) * scale).to(dtype).to(DEV)


def rms(v, w, eps):
    return v / torch.sqrt((v * v).mean(-1, keepdim=True) + eps) * w.double()


def experts(ops, T, H, topk, dense, seed):
    """Unsummed rows of experts, one of the pairs without a row, and what they add up to in 64 bits."""
    y = drawn((3 * T, H), seed)
    slot = torch.randint(0, 3 * T, (T, topk), generator=torch.Generator().manual_seed(seed), dtype=torch.int32).to(DEV)
    slot[T // 2, topk - 1] = -1
    weights, gate = drawn((T, topk), seed + 1).abs(), drawn((T,), seed + 2).abs()
    extra = drawn((dense, T, H), seed + 3) if dense else None
    total = (y.double()[slot.clamp(min=0).long()] * (weights * (slot >= 0)).double()[..., None]).sum(1)
    if dense:
        total = total + gate.double()[:, None] * extra.double().sum(0)
    return ops.GatheredSum(y, slot, weights, extra, gate if dense else None), total


def close(got, want, roundings):
    """Within some roundings of 32 bits (and one of the result's type) of values that a row's largest bounds."""
    size = want.abs().amax(-1, keepdim=True) + 1e-20
    eps = roundings * 2.0 ** -24 + (2.0 ** -8 if got.dtype == torch.bfloat16 else 0.0)
    return ((got.double() - want).abs() <= eps * size).all()


@pytest.mark.parametrize("act", ["float32", "bfloat16"])
@pytest.mark.parametrize("H", LENGTHS)
def test_sum_and_norm(ops, act, H):
    T, eps = 5, 1e-5
    dt = torch.float32 if act == "float32" else torch.bfloat16
    w, wd = drawn((H,), 1, 0.1, dt) + 1, drawn((H,), 2, 0.1, dt) + 1
    for kind, topk, parts in (("parts", 0, 1), ("parts", 0, 5), ("experts", 1, 0), ("experts", 4, 2), ("experts", 6, 5)):
        if kind == "parts":
            delta = drawn((parts, T, H), 3)
            total = delta.double().sum(0)
        else:
            delta, total = experts(ops, T, H, topk, parts, 4)
        x0 = drawn((T, H), 5)
        x = x0.clone()
        out, out32 = ops.add_rmsnorm(x, delta, w, eps, act, want_f32=True)
        v = x0.double() + total
        assert close(x, v, 64) and close(out32, rms(v, w, eps), 256) and close(out, rms(v, w, eps), 256)
        rows = torch.tensor([4, 0, 4], dtype=torch.int32, device=DEV)
        x = x0.clone()
        picked, _ = ops.add_rmsnorm(x, delta, w, eps, act, rows=rows)
        assert torch.equal(x, x0) and torch.equal(picked, out[rows.long()])
        # what is added passes a norm of its own first
        normed = ops.NormedDelta(delta, wd, eps)
        x = x0.clone()
        out, out32 = ops.add_rmsnorm(x, normed, w, eps, act, want_f32=True)
        v = x0.double() + rms(total, wd, eps)
        assert close(x, v, 256) and close(out32, rms(v, w, eps), 512) and close(out, rms(v, w, eps), 512)
        x = x0.clone()
        stream, _ = ops.add_rmsnorm(x, normed, None, eps, act, stream=True)
        assert close(stream, v, 256)
        # and the summed row blended with the row that the sequence's slot keeps
        x, state, sw = x0.clone(), drawn((T + 1, H), 6), drawn((H,), 7, 0.1) + 0.5
        slots, kept = torch.tensor([3, 0, 5, 1, 2], dtype=torch.int32, device=DEV), state.clone()
        v = x0.double() + rms(total, wd.float(), eps)
        blended, _ = ops.add_rmsnorm(x, ops.NormedDelta(delta, wd.float(), eps), None, eps, act, stream=True, shift=(sw, state, slots))
        assert close(blended, v + (kept[slots.long()].double() - v) * sw.double(), 512) and torch.equal(state[slots.long()], x)
        if H % 4 == 0 and act == "float32":      # weights that do not start at a whole run
            off = torch.cat([wd[:1], wd])[1:]
            x2 = x0.clone()
            ops.add_rmsnorm(x2, ops.NormedDelta(delta, off, eps), w, eps, act)
            assert close(x2, v, 256)
            # the sums' order does not hang on where anything starts: the same bits, also where a shared part starts so
            x1 = x0.clone()
            want = ops.add_rmsnorm(x1, normed, w, eps, act, want_f32=True)
            cases = [(delta, off)]
            if kind == "experts" and parts:
                dense = torch.cat([delta.dense.flatten()[:1], delta.dense.flatten()])[1:].view_as(delta.dense)
                assert dense.data_ptr() % 16
                cases += [(ops.GatheredSum(delta.y, delta.pair_slot, delta.weights, dense, delta.gate), n) for n in (wd, off)]
            for moved, norm in cases:
                x2 = x0.clone()
                got = ops.add_rmsnorm(x2, ops.NormedDelta(moved, norm, eps), w, eps, act, want_f32=True)
                assert torch.equal(x1, x2) and torch.equal(want[0], got[0]) and torch.equal(want[1], got[1])


@pytest.mark.parametrize("H", LENGTHS)
def test_sum_of_several_parts(ops, H):
    T, eps = 3, 1e-5
    w, vec, x0 = drawn((H,), 1, 0.1) + 1, drawn((H,), 2), drawn((T, H), 3)
    a, b = drawn((1, T, H), 4), drawn((5, T, H), 5)
    gathered, total = experts(ops, T, H, 3, 0, 6)
    x = x0.clone()
    out, out32 = ops.add_rmsnorm(x, ops.Terms([(0.5, a), (2.0, b)], gathered, vec), w, eps, "float32", want_f32=True)
    v = x0.double() + vec.double() + total + 0.5 * a.double().sum(0) + 2.0 * b.double().sum(0)
    assert close(x, v, 64) and close(out, rms(v, w, eps), 256) and torch.equal(out, out32)


@pytest.mark.parametrize("H", [64, 512, 1020, 1024, 4096, 4100, 8192])
def test_parts_of_many_rows(ops, H):
    """Many rows of short or long runs take another kernel than few: a row's bits are the same."""
    T, eps = 257, 1e-5
    w, vec, x0 = drawn((H,), 1, 0.1) + 1, drawn((H,), 2), drawn((T, H), 3)
    a, b = drawn((1, T, H), 4), drawn((5, T, H), 5)
    gathered, _ = experts(ops, T, H, 3, 0, 6)

    def run(n):
        x = x0[:n].clone()
        part = ops.GatheredSum(gathered.y, gathered.pair_slot[:n].contiguous(), gathered.weights[:n].contiguous(), None, None)
        return x, *ops.add_rmsnorm(x, ops.Terms([(0.5, a[:, :n].contiguous()), (2.0, b[:, :n].contiguous())], part, vec), w, eps, "bfloat16", want_f32=True)

    for many, few in zip(run(T), run(T - 1)):
        assert torch.equal(many[:T - 1], few)


@pytest.mark.parametrize("act", ["float32", "bfloat16"])
def test_rows_of_no_numbers(ops, act):
    """Empty rows come back empty; the library's entries read and write nothing for them."""
    import ctypes
    dt = torch.float32 if act == "float32" else torch.bfloat16
    x, w = drawn((5, 0), 1), drawn((0,), 2, dtype=dt)
    rows = torch.tensor([4, 0, 4], dtype=torch.int32, device=DEV)
    for delta in (None, drawn((2, 5, 0), 3), experts(ops, 5, 0, 3, 2, 4)[0]):
        for picked in (None, rows):
            out, out32 = ops.add_rmsnorm(x, delta, w, 1e-5, act, rows=picked, want_f32=True)
            assert out.shape == out32.shape == (5 if picked is None else 3, 0)
    lib, st = ops.library(act), torch.cuda.current_stream().cuda_stream
    buf = [drawn((64,), seed) for seed in range(5)]
    was = [b.clone() for b in buf]
    x, delta, w, out, out32 = (b.data_ptr() for b in buf)
    assert lib.tq_add_rmsnorm(x, delta, 2, 8, None, None, None, 0, None, w, 0, 1e-5, None, 5, out, out32, 0, st) == 0
    assert lib.tq_add_terms_rmsnorm(x, (ctypes.c_int64 * 1)(delta), (ctypes.c_int * 1)(2), (ctypes.c_float * 1)(0.5), 1, 8, None, None,
                                    None, None, 0, w, 0, 1e-5, None, 5, out, out32, 0, st) == 0
    assert lib.tq_add_normed_rmsnorm_shift(x, delta, 2, 8, None, None, None, 0, None, w, 1e-5, w, 0, 1e-5, None, 5, out, out32, 0,
                                           None, None, None, st) == 0
    torch.cuda.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(buf, was))
