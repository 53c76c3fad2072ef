"""The radix sort at the sizes where its tiles change (4, 8 and 16 keys a thread, the tile and look-back edges), for
both key widths, on full, partial and constant digits: stable, against the oracle."""
import numpy as np
import pytest

import oracle
from test_gpu_stages import _gpu_sort

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1023, 1025, 8 * 1024 + 1, 131072, 131073, 200001, 524288, 524289, 9 * 4096 * 16 + 5])
@pytest.mark.parametrize("dtype,bits", [(np.uint32, 24), (np.uint32, 13), (np.uint64, 63)])
def test_sort_sizes(n, dtype, bits):
    print(f"sort: {n} keys of {bits} bits", flush=True)
    rng = np.random.default_rng(n + bits)
    vals = np.arange(n, dtype=np.uint32)
    for keys in (rng.integers(0, 1 << bits, n, dtype=np.uint64).astype(dtype), np.full(n, 77, dtype),
                 (rng.integers(0, 5, n, dtype=np.uint64) << np.uint64(bits - 3)).astype(dtype)):
        gk, gv = _gpu_sort(keys, vals, 0, bits)
        ok, ov = oracle.sort_pairs(keys, vals, 0, bits)
        assert np.array_equal(gk, ok) and np.array_equal(gv, ov)
