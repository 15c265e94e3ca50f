"""The traffic summary that bench.py reads: bytes per launch are reads plus
writes, and agree with the bytes per site and step on the workload's lattice."""
import json
import os
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_bytes_per_launch():
    sys.path.insert(0, ROOT)
    import bench
    with open(os.path.join(ROOT, 'profiles', 'traffic.json')) as f:
        table = json.load(f)
    assert set(table) == set(bench.WORKLOADS)
    for name, t in table.items():
        sites = 1
        for d in bench.WORKLOADS[name]['dims']:
            sites *= d
        assert abs(t['fetch_bytes'] + t['write_bytes'] - t['bytes_per_launch']) <= 1, name
        want = t['bytes_per_site'] * sites * t.get('steps_per_launch', 1)
        # bytes_per_site has one decimal
        assert abs(t['bytes_per_launch'] - want) <= 0.05 / t['bytes_per_site'] * want, name
