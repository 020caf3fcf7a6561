"""Host grouping of table entries by target point (``vl1_table_groups_host``)
against a stable sort: one entry, all entries of one point, duplicates, unsorted
ids, the largest key; ids out of range are refused."""

import ctypes

import numpy as np
import pytest

from volumential_amd import _capi


def _group(n_cases, n, ids):
    ids = np.ascontiguousarray(ids, dtype=np.int64)
    order, mode = np.empty(ids.size, np.int64), np.empty(ids.size, np.int32)
    start, key = np.empty((2, min(ids.size, n_cases * n) + 1), dtype=np.int64)
    np_ = ctypes.c_int64()
    _capi.check(_capi.lib().vl1_table_groups_host(
        n_cases, n, ids.size, ids.ctypes.data, order.ctypes.data, mode.ctypes.data,
        start.ctypes.data, key.ctypes.data, ctypes.byref(np_)), "vl1_table_groups_host")
    return order, mode, start[:np_.value + 1], key[:np_.value]


@pytest.mark.parametrize("n_cases,n,count", [(1, 1, 1), (33, 4, 200), (139, 27, 5000), (7, 8, 448)])
def test_groups_match_stable_sort(n_cases, n, count):
    ids = np.random.default_rng(n).integers(0, n_cases * n * n, count)
    ids[-1] = n_cases * n * n - 1
    order, mode, start, key = _group(n_cases, n, ids)
    k = ids // (n * n) * n + ids % n
    want = np.argsort(k, kind="stable")
    assert np.array_equal(order, want)
    assert np.array_equal(mode, (ids // n % n)[want])
    u, first = np.unique(k[want], return_index=True)
    assert np.array_equal(key, u) and np.array_equal(start, np.append(first, count))


@pytest.mark.parametrize("bad", [-1, 33 * 16])
def test_groups_refuse_ids_out_of_range(bad):
    with pytest.raises(ValueError):
        _group(33, 4, [3, bad])
