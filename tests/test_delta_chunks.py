"""The scratch that the delta rule's chunks ask for: a function of the host, so it needs no GPU."""
import ctypes

import pytest

from turboquant_cpp_amd.csrc import build


@pytest.fixture(scope="module")
def scratch():
    fn = ctypes.CDLL(build.find_library("float32") or build.build("float32")).tq_delta_chunk_scratch
    fn.argtypes, fn.restype = [ctypes.c_int] * 5, ctypes.c_int64
    return fn


@pytest.mark.parametrize("H,D,V", [(1, 16, 16), (16, 128, 128), (32, 128, 128), (64, 256, 256), (3, 144, 48)])
def test_scratch_is_bounded(scratch, H, D, V):
    """Enough for the step's chunks while they are few, and never more than 1 GiB, however long or many the sequences are."""
    chunk = H * (32 * (3 * D + V) + 32 * 32 + D)
    for T, B in ((48, 1), (2048, 1), (69147, 64), (65535 * 48 - 1, 65535), (3_000_000, 1), (2 ** 31 - 1, 8)):
        chunks = T // 32 + min(B, T // 48)
        assert scratch(T, B, H, D, V) == min(chunks, 65535, 2 ** 28 // chunk) * chunk


def test_what_the_chunks_refuse_asks_for_no_scratch(scratch):
    for T, B, H, D, V in ((47, 1, 16, 128, 128), (2 ** 22, 65536, 16, 128, 128), (96, 0, 16, 128, 128), (96, 1, 16, 40, 128),
                          (96, 1, 16, 128, 24), (96, 1, 16, 272, 128)):
        assert scratch(T, B, H, D, V) == 0
