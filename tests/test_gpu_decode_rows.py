"""Decode attention of short pairs, everything of which is requested at once: lengths around the tiles of 16 keys and the four wavefronts that
share them, one, two and three tiles a wavefront, wavefronts without a tile, sequences far shorter than the longest, the longest that
the launch takes and the next, one to sixteen heads a group; values by distance are in the tests of the design that has them."""
import pytest

import test_gpu_decode_whole_pairs as pairs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,KV,hd", [(32, 8, 64), (8, 8, 64), (16, 1, 64), (32, 4, 128), (6, 2, 128), (16, 1, 128)])
@pytest.mark.parametrize("lengths", [[1], [16], [17], [49], [64], [65], [128], [2, 16, 33, 63, 64, 65, 1, 127, 128]])
def test_short_pairs(H, KV, hd, lengths):
    pairs.test_decode_over_whole_pairs(H, KV, hd, lengths, max(lengths) > 48)  # (spans are of four tiles at least)


@pytest.mark.parametrize("lengths", [[129, 1], [176, 160], [192, 3], [193, 3], [177, 16, 192, 5]])
def test_three_tiles_a_wavefront_and_more(lengths):
    pairs.test_decode_over_whole_pairs(32, 8, 64, lengths, True)
