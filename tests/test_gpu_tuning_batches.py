"""The shipped tuning file on batches: its batch line, measured on 256 replicas of 4 million
beads, is not for a few boxes as large each, which keep the automatic choice; a line without
the range of all beads holds for any batch, and the library reads what dpd_amd.tune finds."""
import json

import numpy as np
import pytest

import dpd_amd as D
from dpd_amd import tune as T
from helpers import chain_state

pytestmark = pytest.mark.gpu
A3 = np.array([[25.0, 30.0, 35.0], [30.0, 10.0, 25.0], [35.0, 25.0, 40.0]])
G3 = np.full((3, 3), 4.5)


def batch(sides):
    e = D.Batch([{"cells": (s, s, s), "a": A3, "gamma": G3, "seed": 3 + q} for q, s in enumerate(sides)])
    for q, s in enumerate(sides):
        n = 3 * s ** 3
        ids, t, x, u, v, (h, tl, fi, se) = chain_state((s, s, s), n // 100, 10, n - 10 * (n // 100), seed=q)
        e.upload_box(q, ids, t, x, v, unpbc=u)
        e.upload_box_topology(q, h, tl, np.full(len(h), 128.0), np.full(len(h), 0.5))
    e.commit()
    return e


@pytest.mark.parametrize("sides", [(15, 14), (14, 15, 16, 17), (14, 15, 16, 17) * 3])
def test_few_boxes_keep_the_automatic_choice(sides):
    e = batch(sides)
    auto = e.schedule
    print(f"{len(sides)} boxes, {e.n} beads: {D.schedule_name(auto)}", flush=True)
    assert 8192 <= e.n // len(sides) < 16384
    assert T.apply(e) is None and e.schedule == auto
    assert T.lookup(len(sides), e.n, 3, True) is None


def test_lines_with_and_without_all_beads(tmp_path):
    e = batch((14, 15, 16))
    lo = 1 << (e.n.bit_length() - 1)
    key = dict(nbox=2, beads_lo=8192, beads_hi=16384, ntypes=3, bonded=1)
    for extra, holds in (({}, True), (dict(total_lo=lo, total_hi=2 * lo), True),
                         (dict(total_lo=2 * lo, total_hi=4 * lo), False), (dict(total_lo=lo // 2, total_hi=lo), False)):
        path = tmp_path / "tune.json"
        path.write_text(json.dumps(dict(key, **extra, schedule=1)) + "\n")
        e.set_schedule(3)
        got = T.apply(e, str(path))
        assert got == T.lookup(3, e.n, 3, True, str(path)) == (1 if holds else None)
        assert e.schedule == (1 if holds else 3)
