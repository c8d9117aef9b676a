"""Convolution and unit vectors of a long step by runs of eight tokens: the bits of the kernel that takes a token to a wave, which a
sequence's tokens get when they come in a short step of their own."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
# sequences of the step: shorter than the taps, one token to each side of a run of eight and of a step of 128; in all tokens enough for
# runs with the fewest heads, and none of them alone
LENGTHS = [1, 2, 3, 4, 7, 8, 9, 1, 1, 127, 16, 100] * 8


@pytest.mark.parametrize("act", ["float32", "bfloat16"])
@pytest.mark.parametrize("heads,groups,dim,vdim", [(2, 2, 128, 128), (3, 1, 64, 256), (4, 2, 256, 64)])
@pytest.mark.parametrize("head_decay", [False, True])
def test_runs_against_tokens(act, heads, groups, dim, vdim, head_decay):
    from turboquant_cpp_amd.csrc import ops
    dims = ops.DeltaDims(heads, groups, dim, vdim, 4, *((0, 0, True) if head_decay else (24, 40, False)))
    gen = torch.Generator().manual_seed(3)
    draw = lambda *shape: torch.randn(shape, generator=gen).to(DEV)
    n_slots = len(LENGTHS) + 2
    slots = torch.randperm(n_slots, generator=gen)[:len(LENGTHS)].tolist()
    state, conv, proj = draw(n_slots, dims.state_floats + 5), draw(dims.channels, 4), draw(sum(LENGTHS), dims.projections)
    more = (draw(heads), draw(heads)) if head_decay else ()
    prep = ops.delta_prep_h if head_decay else ops.delta_prep
    run = lambda rows, of: prep(rows.contiguous(), torch.tensor(of, dtype=torch.int32, device=DEV), state, conv, *more, dims, act)
    got = run(proj, [s for s, n in zip(slots, LENGTHS) for _ in range(n)])
    at = 0
    for s, n in zip(slots, LENGTHS):
        for a, b in zip(got, run(proj[at:at + n], [s] * n)):
            assert torch.equal(a[at:at + n], b), (n, at)
        at += n
