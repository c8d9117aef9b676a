"""The scan over chunks of the delta rule goes through them in pairs behind the first or the first two: a run's first chunks are the same
whether the run ends there or goes on, and its state is the same in one step and in two."""
import pytest
import torch

from turboquant_cpp_amd.csrc import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# heads of which every wave has the same number of key tiles (64, 128, 256), and others
@pytest.mark.parametrize("D,V", [(64, 32), (128, 128), (256, 16), (48, 16), (112, 48)])
def test_a_run_that_ends_and_one_that_goes_on(D, V):
    H, n = 2, 224
    dims = ops.DeltaDims(H, H, D, V, 4, 8, 8)
    g = torch.Generator().manual_seed(D + V)
    rnd = lambda *s: torch.randn(s, generator=g)      # noqa: E731
    unit = lambda x: (x / x.norm(dim=-1, keepdim=True)).flatten(1)      # noqa: E731
    rows = [t.to(DEV) for t in (unit(rnd(n, H, D)) * D ** -0.5, unit(rnd(n, H, D) + 0.3), rnd(n, H * V), torch.sigmoid(rnd(n, H)), rnd(n, H * D + H * V))]
    a_log, dt_bias, start = (0.5 * rnd(H)).to(DEV), (0.5 * rnd(H * D) - 3).to(DEV), (0.1 * rnd(1, dims.state_floats)).to(DEV)

    def run(lo, hi, state):
        runs = {"cu_seqlens": torch.tensor([0, hi - lo], dtype=torch.int32, device=DEV), "slots": torch.zeros(1, dtype=torch.int32, device=DEV),
                "decode": False}
        return ops.delta_scan(*(t[lo:hi].contiguous() for t in rows), a_log, dt_bias, runs, state, dims, "bfloat16")
    whole = start.clone()
    o = run(0, n, whole)
    for at in (64, 96, 128, 160, 192):      # two to six chunks of 32
        state = start.clone()
        assert torch.equal(run(0, at, state), o[:at]), at
        if n - at >= 64:      # (fewer than 48 tokens would go token by token)
            assert torch.equal(run(at, n, state), o[at:]), at
            assert torch.equal(state[:, :H * D * V], whole[:, :H * D * V]), at
