"""The preparation kernels of GaccO and GPUTx at the sizes where they change
course: tile edges, the switch between tile sizes, rows that span tiles."""
import numpy as np
import pytest

import gpu_cc_tb_amd as g

SHORT_MAX = 1 << 20  # pairs up to which the sort uses its short tile (1,024)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1023, 1025, SHORT_MAX, SHORT_MAX + 1])
@pytest.mark.parametrize("dtype,bits", [(np.uint32, 17), (np.uint64, 33)])
def test_sort_tile_sizes(n, dtype, bits):
    """Either tile size, with key bits that split unevenly over the passes."""
    rng = np.random.default_rng(n + bits)
    keys = rng.integers(0, np.iinfo(dtype).max, n, dtype=dtype, endpoint=True)
    vals = np.arange(n, dtype=np.uint32)
    print(f"[sort-tiles] n={n} bits={bits}", flush=True)
    k, v, _ = g.sort_pairs(keys, vals, key_bits=bits)
    order = np.argsort(keys & dtype((1 << bits) - 1), kind="stable")
    assert np.array_equal(v, order.astype(np.uint32)) and np.array_equal(k, keys[order])
