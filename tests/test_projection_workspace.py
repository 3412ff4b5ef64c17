"""Workspace queries of the general projection and of the Router on it (no GPU).

A workspace sized for a capacity serves every smaller row count, so the queries must not
shrink as the rows grow.
"""

from __future__ import annotations

import time

import pytest

from crosspool_amd import _native


@pytest.mark.parametrize("n,k,dtype", ((1030, 2053, _native.XP_DTYPE_F32), (2048, 6144, _native.XP_DTYPE_BF16),
                                       (128, 2048, _native.XP_DTYPE_F16), (1, 1, _native.XP_DTYPE_BF16)))
def test_projection_workspace_grows_with_the_rows(n, k, dtype):
    query = _native.library().xp_projection_workspace_bytes
    sizes = [query(rows, n, k, dtype) for rows in range(1, 400)]
    assert sizes == sorted(sizes)
    assert sizes[0] >= (4 * n * 2 if k > 1000 else 0)


@pytest.mark.parametrize("precision", (2, 3))
def test_router_workspace_grows_with_the_rows(precision):
    for hidden, experts in ((2048, 128), (1003, 130), (40, 17)):
        query = _native.library().xp_moe_router_workspace_bytes
        sizes = [query(rows, hidden, experts, precision) for rows in range(1, 400)]
        assert sizes == sorted(sizes)


def test_projection_workspace_refuses_nothing():
    query = _native.library().xp_projection_workspace_bytes
    assert query(0, 8, 8, _native.XP_DTYPE_BF16) == 0 and query(8, 8, 8, 99) == 0


@pytest.mark.parametrize("n,k", ((24576, 4096), (4096, 12288), (128, 2048)))
def test_projection_workspace_of_many_rows_is_quick(n, k):
    # The query walks every 64 rows; pricing the column splits of each, which keep no sums, took
    # up to a second at a million rows (22 to 31 ms without).
    query = _native.library().xp_projection_workspace_bytes
    sizes = [query(rows, n, k, _native.XP_DTYPE_F16) for rows in (64, 130, 1024, 8192, 65536)]
    assert sizes == sorted(sizes)
    times = []
    for _ in range(3):
        started = time.perf_counter()
        assert query(1 << 20, n, k, _native.XP_DTYPE_F16) >= sizes[-1]
        times.append(time.perf_counter() - started)
    assert min(times) < 0.15
