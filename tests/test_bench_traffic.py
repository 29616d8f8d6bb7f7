"""The benchmark's counted HBM bytes belong to the schedule they were counted
under: given for schedules that launch a kernel the same way, left out otherwise."""
from types import SimpleNamespace

import pytest

import bench

WL = SimpleNamespace(name="config2-100Mbp-250bp-40x", k=31, buckets_log=10, second_buckets_log=6,
                     data=SimpleNamespace(size=4_016_000_000))
COUNTED = dict(item_occ=0, unit_bytes=2000, table_pct=200, lds_table_log=11, rec_cap=256, use_graphs=1)


@pytest.mark.parametrize("change,stage,merge", [({}, True, True), (dict(unit_bytes=3000, use_graphs=0), True, True),
                                                (dict(item_occ=1024, table_pct=400), True, True),
                                                (dict(table_pct=100), True, False), (dict(item_occ=2048), True, False),
                                                (dict(lds_table_log=10, rec_cap=128), True, False),
                                                (dict(unit_bytes=1000), False, False), (dict(unit_cap=800), False, False)])
def test_traffic_is_of_the_timed_schedule(change, stage, merge):
    s = dict(COUNTED, **change)
    for kernel, known in (("bucket_stage", stage), ("unit_compact", stage), ("merge", merge)):
        gb, source = bench.measured_traffic(WL, 1.0, kernel, s)
        assert (gb is not None and gb > 0 and bool(source)) if known else (gb is None and source is None)


def test_traffic_is_of_the_workload():
    other = SimpleNamespace(**dict(vars(WL), name="config4-500Mbp-150bp-30x-k63"))
    assert bench.measured_traffic(other, 1.0, "merge", COUNTED) == (None, None)
    assert bench.measured_traffic(WL, 0.5, "merge", COUNTED) == (None, None)
    assert bench.measured_traffic(WL, 1.0, "merge", None)[0] == bench.measured_traffic(WL, 1.0, "merge", COUNTED)[0]
