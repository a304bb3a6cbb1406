"""The benchmark's count of M2L launches and of the bytes that they cannot do
without: chunks of right-hand sides merged into one launch in the stored
variant, one launch a chunk in the batched one."""
import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)

import bench


@pytest.mark.parametrize("L,nrhs,mixed,batched,launches", [
    (8, 16, True, False, 1), (8, 16, True, True, 8), (8, 17, True, False, 2),
    (4, 19, True, False, 3), (4, 19, True, True, 6), (2, 19, True, False, 3),
    (5, 40, True, False, 3), (8, 16, False, False, 2), (3, 7, False, False, 3),
    (6, 1, False, False, 1)])
def test_launches_and_bytes(L, nrhs, mixed, batched, launches):
    st = {"m2l_group_entries": 1000, "m2l_groups": 50, "m2f_slots": 300, "m2l_targets": 200,
          "m2l_table_rows": 70}
    total, n = bench.m2l_compulsory_bytes(st, L, nrhs, mixed, batched)
    assert n == launches
    one, n1 = bench.m2l_compulsory_bytes(st, L, 1, mixed, batched)
    none = dict(st, m2f_slots=0, m2l_targets=0)
    table, _ = bench.m2l_compulsory_bytes(none, L, 1, mixed, batched)
    assert n1 == 1 and total == nrhs * (one - table) + launches * table
