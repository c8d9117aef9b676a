"""Products of many rows: into how many runs of k they go and which leave for the vendor's library, as the rules say without a GPU."""
import ctypes

import pytest

from turboquant_cpp_amd.csrc import build


@pytest.fixture(scope="module")
def lib():
    return ctypes.CDLL(build.find_library("bfloat16") or build.build("bfloat16"))


def tile_kernel_runs(M, N, K):
    """Tiles of 128 x 128 that do not fill the chip twice, runs of 1,024 of k at least."""
    runs = 1
    while runs < 4 and -(-M // 128) * -(-N // 128) * runs < 512 and K // (2 * runs) >= 1024:
        runs *= 2
    return runs


def test_many_rows_go_in_no_fewer_and_bounded_runs(lib):
    """A run fewer is a longer sum of 32 bits, with a larger error; a run more is as much again for the next kernel to read.  Every run
    has two steps of 64 and more."""
    for M in (1025, 1500, 2048, 3001, 4096, 6000, 8192, 13197, 28000):
        for N in (64, 128, 184, 1024, 2048, 3072, 3584, 4096, 5824, 6144, 8192, 20480):
            for K in (128, 192, 512, 960, 2048, 2112, 3584, 4096, 5632, 8192, 11008, 19520, 20480):
                runs, least = lib.tq_gemm_mfma_splits(M, N, K), tile_kernel_runs(M, N, K)
                assert least <= runs <= 4, (M, N, K)
                assert runs == least or runs * M * N * 4 <= 256 << 20, (M, N, K)
                steps, per = K // 64, -(-(K // 64) // runs)
                assert runs == 1 or steps - per * (runs - 1) >= 2, (M, N, K)


@pytest.mark.parametrize("M,N,K", [(13197, 3584, 3584), (12000, 6144, 5632), (8192, 3584, 20480), (13197, 3584, 20480), (9000, 2048, 16384), (3258, 8224, 4096)])
def test_plain_products_of_a_long_k_stay_with_the_library_that_adds_it_in_parts(lib, M, N, K):
    """Its sums of 32 bits are the closer ones to 64 bits; an activation or a gate's result of 16 bits keeps nothing of that."""
    assert not lib.tq_gemm_here_rather(M, N, K, 0)
    assert lib.tq_gemm_here_rather(2048, 6288, 2048, 0) and lib.tq_gemm_here_rather(2048, 5632, 2048, 2)


@pytest.mark.parametrize("N", [8, 16, 32])
def test_few_columns_stay_in_the_tile_kernel(lib, N):
    """Tiles of 256 columns are nearly empty there: only a long k in one run and one round of tiles makes up for it, and a gated pair."""
    for M in (1025, 4096, 16384, 16385, 65536):
        for K in (128, 512, 1024, 1984, 2048, 4096):
            here = lib.tq_gemm_phases_rows(M, N, K, 0, 1)
            assert (here > 0) == (K >= 2048 and M <= 16384), (M, K)
            assert not lib.tq_gemm_phases_rows(M, N, K, 0, 2) and lib.tq_gemm_phases_rows(M, N, K, 1, 1)
            assert lib.tq_gemm_mfma_splits(M, N, K) == tile_kernel_runs(M, N, K)
            assert lib.tq_gemm_phases_rows(M, 40, K, 0, 1)


def test_one_round_of_the_tile_kernel_stays_its_own(lib):
    """Partial sums of up to 128 columns in the tile kernel's runs; more runs than its are for the other tiles."""
    for M, N, K, here in ((16384, 64, 2048, 0), (14000, 128, 2048, 0), (8192, 40, 4096, 0), (16384, 136, 2048, 1), (12000, 64, 2048, 1), (20000, 64, 2048, 1)):
        runs = lib.tq_gemm_mfma_splits(M, N, K)
        assert runs > 1 and (lib.tq_gemm_phases_rows(M, N, K, 0, runs) > 0) == bool(here), (M, N, K)
        assert runs == tile_kernel_runs(M, N, K) or lib.tq_gemm_phases_rows(M, N, K, 0, runs)


@pytest.mark.parametrize("kind,M,N,K", [(0, 2048, 6288, 2048), (1, 3001, 8448, 2048), (2, 2048, 5632, 2048), (3, 1091, 1032, 8256)])
def test_operands_that_begin_between_16_bytes_leave_for_the_library(lib, monkeypatch, kind, M, N, K):
    """The tiles refuse them, whatever their size says; the vendor's library takes any address."""
    import torch

    from turboquant_cpp_amd.csrc import ops
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.setattr(ops, "library", lambda act: lib)

    def at(rows, first):
        return torch.empty(rows * K + 8, dtype=torch.bfloat16)[first:first + rows * K].view(rows, K)
    for a_first, w_first, leaves in ((0, 0, False), (8, 8, False), (4, 0, True), (0, 4, True), (1, 8, True)):
        a, w = at(M, a_first), at(N, w_first)
        assert a.is_contiguous() and w.is_contiguous()
        assert ops._vendor_here("bfloat16", a, w, M, N, K, kind) is leaves, (a_first, w_first)


@pytest.mark.parametrize("M,N,K,here", [
    (2048, 4096, 8192, True), (2049, 4096, 8192, False), (1280, 6144, 8192, True), (1281, 6144, 8192, False),      # 256 tiles in two runs, and more
    (1091, 7168, 14336, False), (2713, 2944, 12928, False), (3258, 5120, 8192, False), (3258, 5120, 11008, True),      # 1.1e11, 1.0e11, 1.4e11, 1.8e11
    (2209, 8128, 14528, True), (2209, 8192, 14528, False), (1024, 2048, 8448, False), (1025, 2048, 8448, True), (3258, 2048, 8128, False),
    (3258, 1016, 8448, False), (3258, 2048, 8448, True)])
def test_partial_sums_of_a_long_k_stay_in_one_round_of_tiles_or_where_they_are_many(lib, M, N, K, here):
    """Beyond one tile to a compute unit the vendor's library is the faster one up to 1.4e11 multiply-adds."""
    assert bool(lib.tq_gemm_here_rather(M, N, K, 3)) is here
    assert not lib.tq_gemm_here_rather(M, N, K, 0)
