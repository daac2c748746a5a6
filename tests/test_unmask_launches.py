"""Which unmask steps select in the vocabulary pass's own launch: none whose arrivals at a sequence's counter, or whose many short rows, take longer than a second launch."""
import pytest

import mdx


# (blocks, positions, vocabulary, seeded): 9, 8 and 3 splits of 32 positions, 4 and 9 of 64; draws; 2048 rows and more, long and short
@pytest.mark.parametrize("bs, S, vocab, seeded, one", [
    (1, 32, 151936, 0, False), (3, 32, 151936, 0, False), (4, 32, 151936, 0, True), (32, 32, 151936, 0, True), (1, 32, 151936, 1, True),
    (1, 32, 64000, 0, True), (1, 64, 64000, 0, True), (1, 64, 151936, 0, False), (4, 64, 151936, 0, True), (1, 64, 151936, 1, True),
    (64, 32, 151936, 0, True), (65, 32, 151936, 0, False), (32, 32, 1000, 0, True), (33, 32, 1000, 0, False), (33, 32, 1000, 1, False), (64, 32, 4096, 1, True),
    (2, 65, 5000, 0, False), (0, 32, 5000, 0, False), (1, 32, 0, 0, False)])
def test_where_one_launch_pays(bs, S, vocab, seeded, one):
    assert bool(mdx._lib.lib().mdx_unmask_step_single_launch_pays(bs, S, vocab, seeded)) == one
