"""A force evaluation that ends with an error leaves the engine as it was: without the
thermostat it switches the thermostat's table off for the evaluation alone."""
import numpy as np
import pytest

import dpd_amd as D
from helpers import random_state

pytestmark = pytest.mark.gpu
A2 = np.array([[25.0, 40.0], [40.0, 25.0]])
G2 = np.full((2, 2), 4.5)
ERR_NAN = 4


@pytest.mark.parametrize("boxes", [1, 2])
def test_thermostat_is_back_after_a_failed_evaluation(boxes):
    cells, n = (6, 6, 6), 648
    ids, t, x, v = random_state(cells, n, 2, seed=2)
    bad = v.copy()
    bad[100] = np.nan

    def engine():
        if boxes == 1:
            return D.Engine(cells, A2, G2, seed=4)
        return D.Batch([{"cells": cells, "a": A2, "gamma": G2, "seed": 4 + b} for b in range(boxes)])

    def upload(e, vel):
        if boxes == 1:
            e.upload(ids, t, x, vel)
        else:
            for b in range(boxes):
                e.upload_box(b, ids, t, x, vel)
            e.commit()

    print("failed evaluation", boxes, flush=True)
    e, fresh = engine(), engine()
    upload(e, bad)
    with pytest.raises(D.DpdError) as err:
        e.compute_forces(step=3, thermostat=False)
    assert err.value.code == ERR_NAN
    upload(e, v)
    upload(fresh, v)
    f = e.compute_forces(step=3)[0]
    assert np.array_equal(f, fresh.compute_forces(step=3)[0])
    assert not np.array_equal(f, fresh.compute_forces(step=3, thermostat=False)[0])
    e.step(4)
    fresh.step(4)
    for a, b in zip(e.download(), fresh.download()):
        assert np.array_equal(a, b)
