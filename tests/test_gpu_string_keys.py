"""String keys read a word at a time: lengths on both sides of the 4-, 8- and
16-byte steps, every alignment of the characters, and keys that differ in one
byte only, against the CPU oracle and the host's MurmurHash3."""
import numpy as np
import pytest

from oracle import oracle as orc
from tests.gbutil import AGG, assert_parity, host_col

pytestmark = pytest.mark.gpu

LENGTHS = [0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 11, 12, 15, 16, 17, 20, 23, 24, 31, 32, 33, 40, 47]


def _variants():
    """Per length a base string and copies with the first, a middle and the last byte changed."""
    out = []
    for n in LENGTHS:
        base = bytes((37 * i + n) % 256 for i in range(n))
        out.append(base)
        for at in sorted({0, n // 2, n - 1} if n else set()):
            out.append(base[:at] + bytes([base[at] ^ 0x80]) + base[at + 1:])
    return out


@pytest.mark.parametrize("strategy", ["auto", "partitioned", "exact"])
def test_lengths_alignments_and_near_duplicates(strategy):
    from cudf_amd import _lib
    rng = np.random.default_rng(5)
    pool = _variants()
    n = 30_001
    pick = rng.integers(0, len(pool), n)
    key = orc.HostColumn.from_strings([pool[i] for i in pick])
    v = host_col(rng.integers(-50, 50, n))
    _lib.set_strategy({"auto": _lib.STRATEGY_AUTO, "partitioned": _lib.STRATEGY_PARTITIONED,
                       "exact": _lib.STRATEGY_PARTITIONED_EXACT}[strategy])
    try:
        ng = assert_parity([key], [(v, [(AGG["SUM"], 1), (AGG["MIN"], 1), (AGG["COUNT_ALL"], 1)])])
    finally:
        _lib.set_strategy(_lib.STRATEGY_AUTO)
    assert ng == len(set(pool[i] for i in pick))
