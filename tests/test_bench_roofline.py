"""The benchmark's carving bandwidth comes from measured traffic, not from the count of camera tests, which the
solid maps leave out for the most part (no GPU needed)."""

import bench

KERNEL = "carve_classify_queue_kernel"


def _levels(tests):
    return [dict(step=0, level=1, kernel="carve_classify_child_kernel", ms=0.02, parents=64, camera_tests=9, children=5),
            dict(step=7, level=8, kernel=KERNEL, ms=0.5, parents=10, camera_tests=tests, children=20),
            dict(step=8, level=9, kernel=KERNEL, ms=1.5, parents=20, camera_tests=tests, children=40)]


def test_bandwidth_is_measured_traffic_over_time(monkeypatch):
    monkeypatch.setattr(bench, "traffic_from_profile", lambda k: {"fetch": 6e8, "write": 2e8, "hash": "x"})
    for tests in (1, 10**9):
        r = bench.roofline_from(_levels(tests))
        assert r["kernel"] == KERNEL and r["launches"] == 2 and r["levels"] == [8, 9]
        assert r["traffic"] == 800000000 and r["achieved"] == 800.0 and r["frac"] == 0.1
        assert r["camera_tests_per_launch"] == tests


def test_unmeasured_traffic_gives_no_bandwidth(monkeypatch):
    for profile in (None, {"stale": "other build"}):
        monkeypatch.setattr(bench, "traffic_from_profile", lambda k: profile)
        r = bench.roofline_from(_levels(10**9))
        assert r["achieved"] is None and r["frac"] is None and r["traffic"] is None
