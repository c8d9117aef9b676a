"""Prompt attention whose operands are asked for ahead of their products (heads of 64 and 128): sizes around a tile, windows (whose pages
before them are gone), kept first positions, every change of a score, two maps a head.

A probability and an output are each rounded to 8 significant bits (half a unit of the last: 2^-8 of their value at most), so a number of
the output lies within 2^-7 times the weighted sum of the values' magnitudes; 32-bit sums, the hardware's exponential and logarithm add
less than 2^-12."""
import pytest
import torch

from turboquant_cpp_amd.csrc import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
PAGE = 64


def paged(lens, old, nkv, hd, seed, gone=None, width=None):
    """Caches of ``old[i] + lens[i]`` positions; pages before position ``gone[i]`` hold NaN; values are zeros from ``width`` on.  Keys and values
    [n, nkv, hd] too."""
    g = torch.Generator(DEV).manual_seed(seed)
    ends = [a + b for a, b in zip(lens, old)]
    pages = [-(-e // PAGE) for e in ends]
    table = torch.full((len(lens), max(pages)), -1, dtype=torch.int32)
    order = torch.randperm(sum(pages) + 1, generator=torch.Generator().manual_seed(seed))
    kp = torch.full((sum(pages) + 1, nkv, PAGE, hd), float("nan"), dtype=torch.bfloat16, device=DEV)
    vp = torch.full((sum(pages) + 1, nkv, hd, PAGE), float("nan"), dtype=torch.bfloat16, device=DEV)
    ks, vs, at = [], [], 0
    for i, (e, n) in enumerate(zip(ends, pages)):
        k, v = (torch.randn(n * PAGE, nkv, hd, generator=g, device=DEV).bfloat16() for _ in range(2))
        v[..., width or hd:] = 0
        ids = order[at:at + n]
        at += n
        first = gone[i] // PAGE if gone else 0
        table[i, :n] = ids
        table[i, :first] = order[-1]      # a page of NaN
        for p in range(first, n):
            rows = slice(p * PAGE, (p + 1) * PAGE)
            kp[ids[p]] = k[rows].transpose(0, 1)
            vp[ids[p]] = v[rows].permute(1, 2, 0)
        ks.append(k[:e].double())
        vs.append(v[:e].double())
    tokens = sum(lens)
    q = torch.randn(tokens, 1, hd, generator=g, device=DEV)
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)      # noqa: E731
    runs = {"cu_seqlens": i32(cu), "slots": i32(list(range(len(lens)))), "start": i32(old), "max_new": max(lens), "max_end": max(ends),
            "decode": False}
    positions = torch.cat([torch.arange(o, o + n) for n, o in zip(lens, old)]).to(torch.int32).to(DEV)
    seq = torch.cat([torch.full((n,), i) for i, n in enumerate(lens)]).to(torch.int32).to(DEV)
    return kp, vp, table.to(DEV), ks, vs, q, runs, positions, seq


def visible(n, old, window, keep, chunk):
    i, j = torch.arange(old, old + n, device=DEV)[:, None], torch.arange(old + n, device=DEV)[None]
    lo = torch.zeros_like(i)
    if window:
        lo = (i - window + 1).clamp(min=0)
    if chunk:
        lo = torch.maximum(lo, i // chunk * chunk)
    return (j <= i) & ((j >= lo) | (j < keep)), (i - j).clamp(min=0)


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("lens,old,mod", [
    ([193], [0], {}), ([191, 192, 193, 1, 64], [0] * 5, {}), ([256], [0], {}), ([257], [60], {}), ([321], [0], {"sink": 1}), ([700], [0], {"cap": 5.0}),
    ([194], [500], {"window": 70}), ([200, 90], [449, 3], {"window": 100}), ([210], [300], {"window": 66, "keep": 65}),
    ([230], [700], {"window": 130, "keep": 5, "sigmoid": 1}), ([300], [0], {"sigmoid": 1, "gate": 1}), ([400], [0], {"bias": 1}),
    ([200], [100], {"chunk": 192, "bias": 1, "sink": 1}), ([385], [0], {"gate": 1})])
def test_prompts_against_64_bits(hd, lens, old, mod):
    check_prompts(hd, lens, old, mod)


def check_prompts(hd, lens, old, mod, nh=4):
    nkv = 2
    window, keep, chunk = mod.get("window"), mod.get("keep", 0), mod.get("chunk")
    gone = None
    if (window or chunk) and not keep:
        gone = [max(o - window + 1, 0) if window else o // chunk * chunk for o in old]
    kp, vp, table, ks, vs, q, runs, positions, seq = paged(lens, old, nkv, hd, sum(lens) + hd, gone, mod.get("values"))
    g = torch.Generator(DEV).manual_seed(1)
    tokens = sum(lens)
    q = torch.randn(tokens, nh, hd, generator=g, device=DEV).bfloat16()
    f32 = lambda *s: torch.randn(*s, generator=g, device=DEV)      # noqa: E731
    more = {}
    if "sink" in mod:
        more["sink"] = f32(nh)
    if "cap" in mod:
        more["softcap"] = mod["cap"]
    if "bias" in mod:
        more["distance_bias"] = (f32(nh).abs(), f32(nh).abs())
    if "sigmoid" in mod:
        more["sigmoid_bias"] = f32(nh) - 2.0
    if "gate" in mod:
        more["head_gate"] = f32(tokens, nh)
    if "window" in mod or "keep" in mod:
        more["keep_first"] = keep
    if "values" in mod:
        more["value_width"] = mod["values"]
    width = mod.get("values", hd)
    scale = 1.7 * hd ** -0.5
    got = ops.attention(q.reshape(tokens, nh * hd), kp, vp, 0, positions, seq, table, PAGE, nkv * PAGE * hd, nh, nkv, hd, window, scale,
                        "bfloat16", runs=runs, chunk=chunk, **more).double().view(tokens, nh, hd)
    at = 0
    for i, (n, o) in enumerate(zip(lens, old)):
        see, dist = visible(n, o, window, keep, chunk)
        for h in range(nh):
            s = scale * q[at:at + n, h].double() @ ks[i][:, h // (nh // nkv)].T
            if "cap" in mod:
                s = mod["cap"] * torch.tanh(s / mod["cap"])
            if "bias" in mod:
                r1, r2 = (t[h].double() for t in more["distance_bias"])
                s = s - r1 * torch.log1p(r2 * dist)
            if "sigmoid" in mod:
                p = torch.sigmoid(s + more["sigmoid_bias"][h].double()) * see
            else:
                s = s.masked_fill(~see, -torch.inf)
                if "sink" in mod:
                    s = torch.cat([s, more["sink"][h].double().expand(n, 1)], 1)
                p = torch.softmax(s, 1)[:, :o + n]
            if "gate" in mod:
                p = p * torch.sigmoid(more["head_gate"][at:at + n, h].double())[:, None]
            v = vs[i][:, h // (nh // nkv), :width]
            want, bound = p @ v, (2 ** -7 + 2 ** -12) * (p @ v.abs())
            assert ((got[at:at + n, h, :width] - want).abs() <= bound).all(), (i, h)
            assert not got[at:at + n, h, width:].any()
        at += n


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("lens,old", [([193], [0]), ([193, 64, 1], [0] * 3), ([700], [0]), ([200], [130])])
def test_two_maps_a_head(hd, lens, old):
    check_two_maps(hd, lens, old)


def check_two_maps(hd, lens, old):
    nh, nkv, lam, eps, post = 4, 2, 0.4, 1e-5, 0.6
    kp, vp, table, ks, vs, q, runs, positions, seq = paged(lens, old, nkv, hd, 7 + sum(lens) + hd)
    g = torch.Generator(DEV).manual_seed(2)
    tokens = sum(lens)
    q = torch.randn(tokens, nh, hd, generator=g, device=DEV).bfloat16()
    gate = torch.randn(tokens, nh * hd, generator=g, device=DEV)
    scale = 1.7 * (hd // 2) ** -0.5
    got = ops.diff_attention(q.reshape(tokens, nh * hd), kp, vp, 0, positions, seq, table, PAGE, nkv * PAGE * hd, nh, nkv, hd, scale, lam, eps, hd,
                             post, gate, "bfloat16", runs).double().view(tokens, nh, hd)
    at = 0
    for i, (n, o) in enumerate(zip(lens, old)):
        see, _ = visible(n, o, None, 0, None)
        for h in range(nh):
            maps, size = [], 0.0
            for m in range(2):
                part = slice(m * hd // 2, (m + 1) * hd // 2)
                s = scale * q[at:at + n, h, part].double() @ ks[i][:, h // 2, part].T
                p = torch.softmax(s.masked_fill(~see, -torch.inf), 1)
                maps.append(p @ vs[i][:, h // 2])
                size = size + (lam if m else 1.0) * (p @ vs[i][:, h // 2].abs())
            r = maps[0] - lam * maps[1]
            f = post / torch.sqrt((r * r).mean(1, keepdim=True) + eps)
            z = torch.sigmoid(gate[at:at + n, h * hd:(h + 1) * hd].double())
            want = r * f * z
            # the rounded probabilities move r by 2^-8 of `size`, and its root mean square by no more than theirs; the output is rounded
            slack = (2 ** -8 + 2 ** -12) * size
            bound = z * f * (slack + r.abs() * (slack * slack).mean(1, keepdim=True).sqrt() * f / post) + 2 ** -8 * want.abs()
            assert ((got[at:at + n, h] - want).abs() <= 1.1 * bound).all(), (i, h)
        at += n


@pytest.mark.parametrize("hd", [64, 128, 96, 256])
def test_scores_and_sinks_of_minus_infinity(hd):
    """A sink of -inf counts nothing where a key has a finite score; where none has, the sums stay what they began as: 0 over 1."""
    nh, nkv, n = 2, 2, 200
    kp, vp, table, ks, vs, q, runs, positions, seq = paged([n], [0], nkv, hd, hd)
    q = torch.rand(n, nh * hd, generator=torch.Generator(DEV).manual_seed(1), device=DEV).add(0.5).bfloat16()
    kp[table[0].long(), 0, :, 3] = -torch.inf      # the first head's scores are -inf, the second's finite
    sink = torch.full((nh,), -torch.inf, device=DEV)
    got = ops.attention(q, kp, vp, 0, positions, seq, table, PAGE, nkv * PAGE * hd, nh, nkv, hd, None, hd ** -0.5, "bfloat16", runs=runs, sink=sink)
    got = got.double().view(n, nh, hd)
    assert not got[:, 0].any()
    see, _ = visible(n, 0, None, 0, None)
    p = torch.softmax((hd ** -0.5 * q.view(n, nh, hd)[:, 1].double() @ ks[0][:, 1].T).masked_fill(~see, -torch.inf), 1)
    assert ((got[:, 1] - p @ vs[0][:, 1]).abs() <= (2 ** -7 + 2 ** -12) * (p @ vs[0][:, 1].abs())).all()
