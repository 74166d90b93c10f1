"""Which decode steps of five to eight sequences go in one launch: not those whose chunks come out longer than the launches of the layers pay for (no GPU: the rule)."""
import random

import pytest

from nano_vllm_x_amd import ops


def _chunk(lengths, rows):
    """Tiles of the longest chunk, as the kernel's lanes find it."""
    total = sum(lengths)
    least, most = max(1, -(-total // 1024)), max(1, -(-total // 512))
    step = (most - least + 62) // 63
    fits = [least + lane * step for lane in range(64) if sum(max(1, -(-n // (64 * (least + lane * step)))) for n in lengths) + rows - len(lengths) <= 16]
    return fits[0]


@pytest.mark.parametrize("lengths,pays", [      # us of the launches and of the one
    ([2000] * 5, False),                        # 1046 and 1114
    ([3000] * 3 + [100] * 5, False),            # 1088 and 1111
    ([1900] * 5 + [10] * 3, False),             # 1046 and 1091
    ([1700] * 5, False),                        # 1033 and 1056
    ([1250] * 8, True),                         # 1040 and 958
    ([1400] * 7, True),                         # 1046 and 989
    ([9900] + [10] * 7, True),                  # 1299 and 1173
    ([4900] * 2 + [10] * 6, True),              # 1140 and 1112
    ([1100] * 5, True),                         # 984 and 920
    ([2400] * 4, True),                         # 1042 and 877
    ([1], True), ([0] * 8, True), ([60000], True)])
def test_where_the_chunks_come_out_too_long(lengths, pays):
    rows = next(r for r in (1, 2, 4, 8) if r >= len(lengths))
    assert ops.DecodeChain.pays(lengths, rows) is pays


def test_the_rule_finds_a_chunk_for_whatever_is_asked():
    rng = random.Random(3)
    for _ in range(2000):
        n = rng.randint(5, 8)
        lengths = [max(0, int(10 ** rng.uniform(0, 5))) for _ in range(n)]
        got = ops.DecodeChain.pays(lengths, 8)
        total = sum(lengths)
        assert got is (total <= 6000 or 662 + 28.7 * _chunk(lengths, 8) <= 878 + 0.0124 * total + 0.0287 * max(lengths))
