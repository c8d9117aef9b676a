"""Prompt attention of heads between and beyond the sizes that are compiled without run-time conditions, and of two groups of columns a wave: against
64 bits, around tiles and blocks, behind windows (whose pages before them are gone), with kept first positions and every change of a score."""
import pytest

from test_attention_reads_ahead_gpu import check_prompts, check_two_maps

pytestmark = pytest.mark.gpu


# 208 and 240: compiled for up to 256; 272 to 496: for up to 512, in halves of a step of 32 and whole ones; 192, 256 and 512: their own
@pytest.mark.parametrize("hd", [192, 208, 240, 256, 272, 304, 320, 384, 496, 512])
@pytest.mark.parametrize("lens,old,mod", [
    ([193, 64, 1], [0] * 3, {}), ([65], [60], {"sink": 1}), ([194], [500], {"window": 70}), ([210, 17], [300, 3], {"window": 66, "keep": 65}),
    ([130], [0], {"bias": 1, "cap": 5.0}), ([129], [300], {"window": 130, "sigmoid": 1, "gate": 1})])
def test_heads_of_any_size(hd, lens, old, mod):
    check_prompts(hd, lens, old, mod)


# 64 query heads, 64 kv heads of them two each, and sequences whose blocks of 128 tokens are 512 and more: two groups of 16 columns to a wave
@pytest.mark.parametrize("hd", [64, 128, 32, 96])
@pytest.mark.parametrize("lens,old,mod", [
    ([385, 257, 129], [0] * 3, {}), ([385, 200, 1], [100, 0, 7], {"window": 200}), ([400, 260, 33], [300, 60, 0], {"window": 66, "keep": 65}),
    ([385, 129, 64], [0] * 3, {"bias": 1}), ([385, 300, 31], [0, 50, 0], {"sigmoid": 1, "gate": 1})])
def test_two_groups_of_columns_a_wave(hd, lens, old, mod):
    nh = 64
    assert -(-max(lens) // 128) * nh * len(lens) >= 512
    check_prompts(hd, lens, old, mod, nh=nh)


# keys of 192 with values of 128, in one group a wave and in two
@pytest.mark.parametrize("nh,lens", [(4, [193, 64, 1]), (64, [385, 257, 129])])
@pytest.mark.parametrize("old,mod", [([0] * 3, {}), ([70, 0, 300], {"window": 100}), ([0] * 3, {"sink": 1, "bias": 1})])
def test_values_narrower_than_keys(nh, lens, old, mod):
    check_prompts(192, lens, old, {**mod, "values": 128}, nh=nh)


@pytest.mark.parametrize("hd", [160, 256])
@pytest.mark.parametrize("lens,old", [([193, 64, 1], [0] * 3), ([200], [130])])
def test_two_maps_of_wider_heads(hd, lens, old):
    check_two_maps(hd, lens, old)
