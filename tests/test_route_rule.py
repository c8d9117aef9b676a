"""Choice and order of experts in two launches or in more, as the rule says without a GPU."""
import ctypes

import pytest

from turboquant_cpp_amd.csrc import build


@pytest.fixture(scope="module", params=["bfloat16", "float32"])
def lib(request):
    return ctypes.CDLL(build.find_library(request.param) or build.build(request.param))


# tokens, experts, experts a token, row: both sides of each line
@pytest.mark.parametrize("tokens,experts,top,width,two", [
    (511, 60, 4, 2048, 0), (512, 60, 4, 2048, 1), (1023, 130, 8, 2048, 0), (1024, 130, 8, 2048, 1), (4096, 7, 4, 2048, 0), (4096, 8, 4, 2048, 1),
    (1280, 9, 2, 2048, 1), (1279, 9, 2, 2048, 0), (1024, 10, 2, 2048, 1), (1023, 10, 2, 2048, 0), (1000, 16, 1, 2560, 0), (1000, 16, 1, 2561, 1),
    (1000, 15, 1, 2561, 0), (2049, 32, 1, 4096, 1), (2049, 33, 1, 4096, 0), (2048, 64, 1, 1024, 1), (2048, 65, 1, 1024, 0), (2500, 64, 2, 4608, 1), (2500, 65, 2, 4608, 0),
    (1000, 96, 4, 5120, 1), (1000, 97, 4, 5120, 0), (1000, 97, 4, 4608, 1), (1024, 129, 8, 5120, 1), (1025, 129, 8, 5120, 0), (1025, 128, 8, 5120, 1),
    (3071, 20, 2, 5120, 1), (3072, 20, 2, 5120, 0), (7168, 24, 4, 2560, 1), (7169, 24, 4, 2560, 0), (7169, 24, 4, 2048, 1), (7169, 24, 4, 2561, 1),
    (1407, 193, 8, 1024, 0), (1408, 193, 8, 1024, 1), (1024, 193, 8, 1024, 1), (1407, 192, 8, 1024, 1), (600, 10, 1, 5121, 1), (600, 9, 8, 5121, 0),
    (2100, 15, 4, 5121, 0), (2100, 16, 4, 5121, 1), (16384, 32, 4, 1024, 1), (16384, 33, 4, 1024, 0), (600, 16, 2, 45000, 0)])
def test_both_sides_of_the_rules_lines(lib, tokens, experts, top, width, two):
    assert lib.tq_route_in_two(tokens, experts, 0, top, width) == two
