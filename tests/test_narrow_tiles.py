"""Tile widths of FP64 register-resident passes in small launches (CPU: plans on the
stand-in runtime): narrower tiles only while they are one workgroup per CU at most.
"""
import re

import pytest

from .standin import plans

# 256-point passes of 65536 points x batch: 256 units a sequence, 16 or 8 or 4 to a tile
CASES = [(4, 4), (5, 8), (8, 8), (9, 16), (10, 16), (14, 16), (16, 16), (40, 16)]


@pytest.fixture(scope="module")
def answers(tmp_path_factory):
    so = plans.build(tmp_path_factory.mktemp("standin"))
    return plans.run(so, [dict(type="Z2Z", n=[65536], batch=b) for b, _ in CASES])


@pytest.mark.parametrize("k", range(len(CASES)))
def test_fp64_tiles_fit_the_cus(answers, k):
    batch, tile = CASES[k]
    for label, *_ in answers[k]["launches"][0]:
        m = re.search(r"k_col<fp64,(\d+),16,16,", label)
        assert m and int(m.group(1)) == tile, (batch, label)
