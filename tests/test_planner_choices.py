"""The planner's choices between two kernels' tilings against what was measured of both (profiles/)."""
import csv

import numpy as np
import pytest

from conftest import ROOT
from georefine_amd import _fused


def _measured(name):
    with open(ROOT / "profiles" / name, newline="") as file:
        return list(csv.DictReader(file))


def test_whole_lines_are_taken_where_they_were_measured_faster():
    taken, refused = [], []
    for line in _measured("whole_lines.csv"):
        ratio = float(line["model_lines"]) / float(line["model_walk"])
        gain = [float(line[f"us_walk_{n}"]) / float(line[f"us_lines_{n}"]) - 1 for n in (1, 2, 4)]
        (taken if ratio <= _fused.lines_limit(int(line["rows"]), int(line["cols"])) else refused).append(gain)
    taken, refused = np.array(taken), np.array(refused)
    assert len(taken) > 80 and len(refused) > 30
    # one result written over and over stays in the last-level cache; of two and four in turn less and less does
    assert np.all(taken.mean(axis=0) > 0.06) and taken[:, 2].min() > -0.03 and taken.min() > -0.09
    assert np.all(refused.mean(axis=0) < -0.07)


@pytest.mark.parametrize("rows,cols,limit", [(4096, 6144, 1.25), (4095, 6144, 1.14), (17408, 5120, 1.25), (256, 512, 1.14)])
def test_whole_lines_limit_by_the_size_of_the_result(rows, cols, limit):
    assert _fused.lines_limit(rows, cols) == limit


def test_small_predictive_lookups_are_taken_where_they_were_measured_faster():
    taken, refused = [], []
    for line in _measured("predictive_lookups.csv"):
        one = lambda name: int(line[name])
        tiling = {key: one("small_" + key) for key in ("threads", "lanes_per_row", "n_slabs", "n_tiles")}
        pays = _fused.fewer_lookups_pay(one("seg_len"), one("cols") // one("seg_len"), tiling, one("small_lds"),
                                        float(line["share_16"]) / float(line["share_64"]))
        (taken if pays else refused).append([float(line[f"us64_{m}"]) / float(line[f"us16_{m}"]) - 1 for m in (2, 6, 20, 32, 64, 96, 128)])
    taken, refused = np.array(taken), np.array(refused)
    assert len(taken) > 10 and len(refused) > 100
    assert taken.mean() > 0.04 and taken.mean(axis=1).min() > -0.03 and taken.min() > -0.06
    assert refused.mean() < -0.05
