"""kg_neighbor_sets around the edges of the device scan that makes its row
starts (tiles of 512 agents): every list equals the oracle's, the starts are
the lists' prefix sums, and a buffer too small is refused with the total and
the starts known."""
import ctypes

import numpy as np
import pytest

from krabmaga_amd import Field2D, _abi, lib

pytestmark = pytest.mark.gpu

D = 10.0 / 1.5


@pytest.mark.parametrize("n", [1, 511, 512, 513, 5000])
def test_lists_equal_the_oracle(oracle, n):
    side = 300.0
    x, y, hx, hy = oracle.init_uniform(n, side, side, n, 1)
    f = Field2D(side, side, D, True, n)
    f.set_object_locations(np.arange(n, dtype=np.uint32), x, y, hx, hy)
    f.lazy_update()
    of = oracle.Field2D(side, side, D, True)
    for i in range(n):
        of.set_object_location(i, float(x[i]), float(y[i]))
    of.lazy_update()
    storage, row_ptr, ids = f.neighbor_sets(10.0)
    assert row_ptr[0] == 0 and row_ptr[n] == len(ids)
    for k in range(0, n, max(1, n // 300)):
        i = storage[k]
        want = [b[0] for b in of.get_neighbors_within_distance(float(x[i]), float(y[i]), 10.0)]
        assert list(ids[row_ptr[k]:row_ptr[k + 1]]) == want
    again = np.zeros(n + 1, np.uint32)
    total = ctypes.c_size_t()
    rc = lib().kg_neighbor_sets(f._h, 10.0, _abi.u32p(again), _abi.u32p(ids), len(ids) - 1,
                                ctypes.byref(total))
    assert rc == _abi.KG_E_CAPACITY and total.value == len(ids)
    assert np.array_equal(again, row_ptr)
