"""How many waves the preparation kernels keep in flight, against the recorded times of both ways."""
import os

PROFILES = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "profiles")


def _records(name):
    with open(os.path.join(PROFILES, name)) as f:
        return [[float(v) for v in line.split()] for line in f if not line.startswith("#")]


def test_prepare_a(mx):
    """No slower than the kernel before it, and within 1.1 times the better way."""
    records = _records("prep_rows_waves_in_flight.txt")
    assert len(records) > 50
    for rows, K, before, few, many in records:
        us = few if mx.lib().mxfp6_hip_prep_few_waves(int(rows), int(K)) else many
        assert us <= before and us <= 1.1 * min(few, many), (rows, K)
    for K in (64, 1024):  # short rows never, however many
        assert not mx.lib().mxfp6_hip_prep_few_waves(1 << 20, K)
    # few rows: every wave there is
    assert not mx.lib().mxfp6_hip_prep_few_waves(1024, 16128)
    assert mx.lib().mxfp6_hip_prep_few_waves(2048, 16128)


def test_prepare_b(mx):
    """Large B within 1.02 times the better way, however few of a workgroup's columns there are."""
    records = _records("prep_b_waves_in_flight.txt")
    assert len(records) > 15
    for K, N, few, many in records:
        us = few if mx.lib().mxfp6_hip_prep_b_few(int(K), int(N)) else many
        assert us <= 1.02 * min(few, many), (K, N)
    assert not mx.lib().mxfp6_hip_prep_b_few(8192, 2048)  # the last-level cache may hold it
