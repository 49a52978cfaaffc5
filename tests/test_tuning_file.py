"""Keys of the tuning file: a batch's line holds for batches of as many beads in all, within a
power of two, and a line without that range, as files had them before, for any."""
from dpd_amd import tune as T


def test_shape_of_a_batch_has_all_its_beads():
    one = T.shape(1, 12000, 3, True)
    assert one == {"nbox": 1, "beads_lo": 8192, "beads_hi": 16384, "ntypes": 3, "bonded": 1}
    few, many = T.shape(4, 45384, 3, True), T.shape(256, 3960969, 3, True)
    assert (few["beads_lo"], few["total_lo"], few["total_hi"]) == (8192, 32768, 65536)
    assert (many["beads_lo"], many["total_lo"], many["total_hi"]) == (8192, 2097152, 4194304)


def test_shipped_file():
    # 256 replicas, which the batch line was measured on, and four boxes as large
    assert T.lookup(256, 3960969, 3, True) == 2
    assert T.lookup(4, 45384, 3, True) is None
    assert T.lookup(1, 786432, 3, True) == 2


def test_lines_with_and_without_all_beads(tmp_path):
    path = str(tmp_path / "tune.json")
    old = dict(nbox=2, beads_lo=8192, beads_hi=16384, ntypes=3, bonded=1, schedule=5)
    T.save([old], path)
    assert T.lookup(4, 45384, 3, True, path) == T.lookup(256, 3960969, 3, True, path) == 5

    class Engine:
        def autotune_schedules(self, nsteps):
            return 3, {}

    # a new record of a shape replaces the line that held for it
    T_name, T.schedule_name = T.schedule_name, str
    try:
        T.tune(Engine(), 4, 45384, 3, True, path=path)
    finally:
        T.schedule_name = T_name
    assert T.lookup(4, 45384, 3, True, path) == 3
    assert T.lookup(256, 3960969, 3, True, path) is None
