"""GPU tests of size- and layout-dependent branches of the strategies, each at
the sizes where it can go wrong, against the oracle (bit-exact for integers)."""
import numpy as np
import pytest

import oracle as O
from eiger_amd import gamax as G
from test_groupby_gpu import STRATEGIES, assert_same, run, sorted_by_key

pytestmark = pytest.mark.gpu
A = G.aggregation_id


@pytest.mark.parametrize("n", [1, 4095, 4097, 70_001])
@pytest.mark.parametrize("dtype,shift,low,minimum", [
    (np.int64, 12, 7, -(1 << 40)), (np.int32, 5, 31, -(1 << 20)), (np.uint64, 40, 0, 1 << 63), (np.uint32, 0, 0, 5),
    (np.int64, 62, 1, 0)])
def test_sort_strategy_keys_sharing_low_bits(n, dtype, shift, low, minimum):
    """Keys whose low bits are all alike (ids handed out in blocks): the sort
    covers only the varying bits of key - min; output ascending."""
    rng = np.random.default_rng(n + shift)
    codes = rng.integers(0, 2 if shift == 62 else 3000, n)
    keys = (np.array([minimum], dtype=dtype) + ((codes.astype(dtype) << dtype(shift)) | dtype(low))).astype(dtype)
    vals = rng.integers(-1000, 1000, n).astype(np.int64)
    reqs = [(0, A.SUM), (-1, A.COUNT_ALL)]
    exp = sorted_by_key(O.groupby(keys, [vals], reqs))
    for fn in (G.sort_groupby, G.sort_groupby_gfur):
        assert_same(run(fn, keys, [vals], reqs), exp)
