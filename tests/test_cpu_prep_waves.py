"""How many waves prep_rows_kernel keeps in flight, against the recorded times of both: no slower than the
kernel before it, and within 1.1 times the better one."""
import os

PROFILE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "profiles",
                       "prep_rows_waves_in_flight.txt")


def test_waves_in_flight(mx):
    n = 0
    for line in open(PROFILE):
        if line.startswith("#"):
            continue
        rows, K, before, few, many = map(float, line.split())
        us = few if mx.lib().mxfp6_hip_prep_few_waves(int(rows), int(K)) else many
        assert us <= before and us <= 1.1 * min(few, many), line
        n += 1
    assert n > 50
    for K in (64, 1024):  # short rows never, however many
        assert not mx.lib().mxfp6_hip_prep_few_waves(1 << 20, K)
    # few rows: every wave there is
    assert not mx.lib().mxfp6_hip_prep_few_waves(1024, 16128)
    assert mx.lib().mxfp6_hip_prep_few_waves(2048, 16128)
