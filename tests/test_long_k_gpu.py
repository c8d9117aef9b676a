"""Plain products of a long k whose partial sums are wanted apart: which way they go, and how close to 64 bits they are."""
import pytest
import torch

from turboquant_cpp_amd.csrc import ops

pytestmark = pytest.mark.gpu
DEVICE = "cuda:0"


# both sides of 1,024 rows, of 1,024 and 8,192 columns and of k 8,192; remainders of rows and columns
@pytest.mark.parametrize("rows,cols,k,here", [
    (1024, 1024, 8192, False), (1025, 1024, 8192, True), (1025, 1016, 8192, False), (1025, 1024, 8128, False), (1091, 1032, 8256, True),
    (2049, 1280, 12288, True), (1030, 8192, 8192, False),
])
def test_partial_sums_of_a_long_k(rows, cols, k, here):
    gen = torch.Generator().manual_seed(rows + k)
    a = torch.randn(rows, k, generator=gen).to(torch.bfloat16).to(DEVICE)
    w = (torch.randn(cols, k, generator=gen) * 0.02).to(torch.bfloat16).to(DEVICE)
    assert ops._vendor_here("bfloat16", a, w, rows, cols, k, 3) is not here
    parts = ops.gemm(a, w, "bfloat16", partial_sums=True)
    assert (parts.shape[0] > 1) is here
    exact = a.double() @ w.double().t()
    error = ((parts.double().sum(0) - exact).norm() / exact.norm()).item()
    # sums of 32 bits over k / 8 steps that round down: 6.2e-9 sqrt(k) as measured in one run of k, less in several
    assert error < 7e-9 * (k / parts.shape[0]) ** 0.5, error


@pytest.mark.parametrize("first", [(4, 0), (0, 4)])
def test_operands_between_16_bytes(first):
    """Contiguous views that begin 8 bytes into memory: the tiles refuse them, the vendor's library does not."""
    rows, cols, k = 1091, 1032, 8256
    gen = torch.Generator().manual_seed(sum(first))

    def at(rows, first, scale):
        flat = (torch.randn(rows * k + 8, generator=gen) * scale).to(torch.bfloat16).to(DEVICE)
        return flat[first:first + rows * k].view(rows, k)
    a, w = at(rows, first[0], 1.0), at(cols, first[1], 0.02)
    parts = ops.gemm(a, w, "bfloat16", partial_sums=True)
    exact = a.double() @ w.double().t()
    assert parts.shape[0] == 1 and ((parts[0].double() - exact).norm() / exact.norm()).item() < 7e-9 * k ** 0.5
