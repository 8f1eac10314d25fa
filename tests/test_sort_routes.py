"""The lists of tests/test_gpu_pair_sort.py reach the branches of the row-major sort that they are there for."""
import numpy as np
import pytest

from tests import sort_routes, test_gpu_pair_sort

ROUTES = {
    "two records": {"one workgroup"},
    "the last count of one workgroup": {"one workgroup"},
    "the first of one level": {"one level"},
    "the last of one level": {"one level"},
    "the first of two levels": {"two levels"},
    "a small join of runs": {"one workgroup"},
    "one level of runs": {"one level", "second cut"},
    "two levels of runs": {"two levels", "second cut"},
    "one level, a crowded row": {"one level", "windows"},
    "two levels, a crowded row": {"two levels", "windows"},
    "a row too crowded for one workgroup": {"one level", "windows"},
    "few records, long keys": {"one level"},
    "many records, long keys": {"two levels"},
    "0.97 million in 130 000 rows": {"one level"},
    "1.04 million in 130 000 rows": {"one level"},
    "1.0 million in 200 000 rows": {"one level"},
    "1.04 million in 250 000 rows": {"one level"},
    "1.1 million in 250 000 rows": {"two levels"},
    "a crowded core": {"one level", "windows"},
}
LISTS = {**test_gpu_pair_sort.CASES, **test_gpu_pair_sort.SPARSE}


def _route(qv, cv):
    qv, cv = np.asarray(qv).astype(np.int64), np.asarray(cv).astype(np.int64)
    assert max(len(qv), len(cv)) > test_gpu_pair_sort.MAX_BIT_ROWS
    return sort_routes.route(sort_routes.pairs_of(qv, cv), len(qv), len(cv))


def test_every_list_has_a_route():
    assert set(ROUTES) == set(LISTS)


@pytest.mark.parametrize("name", list(ROUTES))
def test_route(name):
    assert ROUTES[name] <= _route(*LISTS[name]())


@pytest.mark.parametrize("name", list(sort_routes.CASES))
def test_route_of_crowded_list(name):
    lists, branches = sort_routes.CASES[name]
    qv, cv = lists()
    assert max(qv.max(), cv.max()) < 4000000  # what two FP16 coordinates below 2000 can code
    assert branches <= _route(qv, cv)
