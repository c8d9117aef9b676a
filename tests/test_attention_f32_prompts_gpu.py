"""32-bit attention of prompts: heads that fill their last 16 (a tile of keys and values ahead in registers) and others, head counts and
sequences that do not divide among the dies, a first block and a last one, windows that leave pages out."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("hd", [16, 32, 64, 128, 256, 12, 100])
@pytest.mark.parametrize("lens,starts,nh,nkv,window", [([1, 64, 65, 200], [0, 0, 3, 0], 3, 3, None), ([130, 1], [70, 500], 6, 2, 100), ([300], [0], 9, 3, 64)])
def test_prompts_against_64_bits(hd, lens, starts, nh, nkv, window):
    from turboquant_cpp_amd.csrc import ops
    page, gen = 64, torch.Generator().manual_seed(hd + nh)
    ends = [a + n for a, n in zip(starts, lens)]
    pages = [-(-e // page) for e in ends]
    order = torch.randperm(sum(pages), generator=gen)
    table = torch.zeros((len(lens), max(pages)), dtype=torch.int32)
    stride = nkv * page * hd
    kp, vp = torch.randn(sum(pages), nkv, page, hd, generator=gen), torch.randn(sum(pages), nkv, hd, page, generator=gen)
    q = torch.randn(sum(lens), nh * hd, generator=gen)
    want, at, first = [], 0, 0
    for i, (n, s) in enumerate(zip(lens, starts)):
        mine = order[first:first + pages[i]]
        table[i, :pages[i]] = mine.int()
        first += pages[i]
        k = kp[mine].permute(1, 0, 2, 3).reshape(nkv, -1, hd).double().repeat_interleave(nh // nkv, 0)
        v = vp[mine].permute(1, 0, 3, 2).reshape(nkv, -1, hd).double().repeat_interleave(nh // nkv, 0)
        x = q[at:at + n].view(n, nh, hd).permute(1, 0, 2).double()
        pos, j = torch.arange(s, s + n)[:, None], torch.arange(k.shape[1])[None]
        see = (j <= pos) & (j > pos - (window or 1 << 30))
        p = torch.softmax((x @ k.transpose(1, 2) * hd ** -0.5).masked_fill(~see, float("-inf")), -1)
        want.append((p @ v).permute(1, 0, 2).reshape(n, nh * hd))
        if window:      # pages that no token of the run reaches are given back
            table[i, :max(0, s - window + 1) // page] = -1
        at += n
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    runs = dict(cu_seqlens=i32(cu), slots=i32(range(len(lens))), start=i32(starts), max_new=max(lens), max_end=max(ends), decode=False)
    pos = i32([p for n, s in zip(lens, starts) for p in range(s, s + n)])
    seq = i32([i for i, n in enumerate(lens) for _ in range(n)])
    got = ops.attention(q.to(DEV), kp.flatten().to(DEV), vp.flatten().to(DEV), 0, pos, seq, table.to(DEV), page, stride, nh, nkv, hd, window,
                        hd ** -0.5, "float32", runs=runs)
    # scores are off by some roundings of sums of hd products, weights and their sums by as much: 1e-5 of values of about one
    assert (got.cpu().double() - torch.cat(want)).abs().max().item() < 1e-5


def test_more_workgroups_than_a_dimension_of_the_grid_holds():
    """The longest run is an upper bound: 17 million workgroups, most of them with nothing to do, whose threads are more than 32 bits count."""
    from turboquant_cpp_amd.csrc import ops
    page, hd, nh, lens = 64, 32, 3, [70, 5]
    gen = torch.Generator().manual_seed(1)
    kp, vp, q = (torch.randn(*s, generator=gen).to(DEV) for s in ((3, nh, page, hd), (3, nh, hd, page), (sum(lens), nh * hd)))
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    table, pos, seq = i32([[2, 0], [1, 0]]), i32([p for n in lens for p in range(n)]), i32([i for i, n in enumerate(lens) for _ in range(n)])
    def attend(longest):
        runs = dict(cu_seqlens=i32([0, 70, 75]), slots=i32([0, 1]), start=i32([0, 0]), max_new=longest, max_end=70, decode=False)
        return ops.attention(q, kp.flatten(), vp.flatten(), 0, pos, seq, table, page, nh * page * hd, nh, nh, hd, None, hd ** -0.5, "float32", runs=runs)
    assert torch.equal(attend(64 * 2_900_000), attend(70))


def test_16_bit_prompts_refuse_more_workgroups_than_a_grid_holds():
    """Their launch has one dimension: beyond what 32 bits count it would leave its output as it was, so it is an error."""
    from turboquant_cpp_amd.csrc import ops
    page, hd, nh, lens = 64, 32, 3, [70, 5]
    gen = torch.Generator().manual_seed(1)
    kp, vp, q = (torch.randn(*s, generator=gen).bfloat16().to(DEV) for s in ((3, nh, page, hd), (3, nh, hd, page), (sum(lens), nh * hd)))
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    table, pos, seq = i32([[2, 0], [1, 0]]), i32([p for n in lens for p in range(n)]), i32([i for i, n in enumerate(lens) for _ in range(n)])
    def attend(longest):
        runs = dict(cu_seqlens=i32([0, 70, 75]), slots=i32([0, 1]), start=i32([0, 0]), max_new=longest, max_end=70, decode=False)
        return ops.attention(q, kp.flatten(), vp.flatten(), 0, pos, seq, table, page, nh * page * hd, nh, nh, hd, None, hd ** -0.5, "bfloat16", runs=runs)
    with pytest.raises(Exception):
        attend(128 * 2_900_000)
    assert torch.equal(attend(64 * 2_700_000 // nh), attend(70))
