"""The benchmark's result line: chain traces are thinned, so that a record that keeps
the last few KB of the output holds the whole line."""
import json

import bench


def test_trace_points():
    assert bench.trace_points(100) == [24, 49, 74, 99]
    assert bench.trace_points(1) == [0] and bench.trace_points(0) == []
    for n in range(1, 300):
        p = bench.trace_points(n)
        assert p[-1] == n - 1 and p[0] >= 0 and len(p) <= 4 and p == sorted(set(p))
    # four chains' three statistics at those steps
    assert len(json.dumps([[[-279225.7165188541] * 4 for _ in p] for _ in range(3)])) < 1200


def test_short_numbers():
    x = dict(a=[1.23456789012345, 3, "t"], b=(dict(c=-279225.7165188541, d=None),), e=True)
    assert bench.short(x) == dict(a=[1.23456789, 3, "t"], b=[dict(c=-279225.717, d=None)], e=True)
