"""The rule and the plan of the many-query decode over their ranges."""
import shutil

import pytest

import mq_rule

pytestmark = pytest.mark.skipif(not shutil.which("g++"), reason="no g++")


def test_plan_covers_its_work():
    for heads in (1, 3, 8, 64, 96, 513, 4000):
        for nq in (8, 15, 16, 17, 32, 33, 48, 49, 64, 65, 200):
            for n in (1, 15, 16, 17, 127, 128, 129, 1300, 8192, 8300, 32768, 300000):
                p = mq_rule.plan(heads, nq, n)
                assert p["qgroups"] == (nq + 15) // 16 and p["qg"] in (1, 2, 4)
                assert p["qblocks"] * p["qg"] >= p["qgroups"] > (p["qblocks"] - 1) * p["qg"]
                assert p["splits"] >= 1 and p["chunk"] % (16 * (4 // p["qg"])) == 0
                assert p["splits"] * p["chunk"] >= n > (p["splits"] - 1) * p["chunk"]


def test_rule_at_its_measured_points():
    """(heads, queries, tokens, padded): the faster of the two, as measured."""
    for point, mq in (((8, 4, 32768, 128), False), ((8, 8, 32768, 128), True),
                      ((16, 8, 16384, 64), False), ((16, 12, 16384, 64), True),
                      ((2, 12, 32768, 128), True), ((12, 12, 512, 128), False),
                      ((4, 12, 1024, 64), False), ((8, 64, 32768, 128), True)):
        assert mq_rule.takes(*point) == mq, point
    assert not mq_rule.takes(4000, 7, 32768, 128)
