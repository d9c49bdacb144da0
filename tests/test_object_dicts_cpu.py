"""Object lists, whichever way they are converted: the values and the types of converting one by one, and
no fixed cost that a short list would notice (a list of 5 took twice as long through numpy as one by one
when every call built the record's dtype)."""
import time

import numpy as np
import pytest


def _array(pkg, n):
    arr = (pkg.Object * max(n, 1))()
    rng = np.random.default_rng(n)
    for o in arr:
        o.centroid[:] = rng.standard_normal(3).tolist()
        o.weighted_centroid[:] = rng.standard_normal(3).tolist()
        o.max_value, o.mean_value = rng.standard_normal(2).tolist()
        o.num_voxels, o.label = int(rng.integers(1, 1 << 40)), int(rng.integers(0, 1 << 40))
        o.bounds[:] = rng.integers(-5, 5000, 6).tolist()
    return arr


def _types(v):
    return [type(x) for x in v] if isinstance(v, list) else type(v)


@pytest.mark.parametrize("n", [0, 1, 2, 3, 40])
def test_values_and_types(pkg, n):
    arr = _array(pkg, n)
    want, got = [arr[i].as_dict() for i in range(n)], pkg.Object.as_dicts(arr, n)
    assert got == want
    for a, b in zip(want, got):
        assert list(a) == list(b)
        assert [_types(v) for v in a.values()] == [_types(v) for v in b.values()]


def test_short_lists_cost_no_more_than_one_by_one(pkg):
    arr = _array(pkg, 5)

    def best(f):
        times = []
        for _ in range(30):
            t = time.perf_counter()
            for _ in range(50):
                f()
            times.append(time.perf_counter() - t)
        return min(times)

    assert best(lambda: pkg.Object.as_dicts(arr, 5)) < 1.5 * best(lambda: [arr[i].as_dict() for i in range(5)])
