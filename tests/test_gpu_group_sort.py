"""Values sorted inside groups for MEDIAN / QUANTILE against the CPU oracle:
group sizes on both sides of what one lane, one wave and one workgroup hold,
and one group past that (the counting sort of the whole column)."""
import numpy as np
import pytest

from tests.gbutil import AGG, assert_parity, host_col

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 3, 63, 64, 65, 127, 128, 129, 255, 256, 257, 511, 512, 513, 1000, 1024, 1025, 2047, 2048, 2049,
         4096, 4097, 8191, 8192]


def _values(rng, dtype, n):
    if np.issubdtype(dtype, np.floating):
        x = rng.standard_normal(n).astype(dtype)
        x[rng.integers(0, n, n // 50)] = np.nan
        x[rng.integers(0, n, n // 50)] = -0.0
        x[rng.integers(0, n, n // 100)] = np.inf
        x[rng.integers(0, n, n // 100)] = -np.inf
        return x
    info = np.iinfo(dtype)
    x = rng.integers(-40, 40, n) if info.min < 0 else rng.integers(0, 80, n)  # many equal values
    x = x.astype(dtype)
    x[rng.integers(0, n, n // 50)] = info.max
    x[rng.integers(0, n, n // 50)] = info.min
    return x


@pytest.mark.parametrize("dtype", [np.float64, np.float32, np.int64, np.int32, np.uint8, np.uint64])
@pytest.mark.parametrize("nulls", [0.0, 0.3])
@pytest.mark.parametrize("longest", [8192, 8193])
def test_sizes_around_the_limits(dtype, nulls, longest):
    rng = np.random.default_rng(longest + int(nulls * 10))
    sizes = SIZES + [longest]
    k = rng.permutation(np.repeat(np.arange(len(sizes), dtype=np.int32) * 3, sizes))
    n = len(k)
    valid = rng.random(n) >= nulls if nulls else None
    if nulls:
        valid[k == 3 * SIZES.index(129)] = False  # a group without values
    v = host_col(_values(rng, np.dtype(dtype), n), valid)
    assert_parity([host_col(k)], [(v, [(AGG["MEDIAN"], 1), (AGG["MAX"], 1)])])
