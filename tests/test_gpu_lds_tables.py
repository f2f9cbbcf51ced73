"""Workgroup-local tables of the hash group-by against the CPU oracle: slots
taken by the key's value, tables that many workgroups store and merge, and the
split of hot keys from the partitioned path.  Integer results are compared
exactly, floating sums within the parity helper's bound (sums in another order)."""
import numpy as np
import pytest

from tests.gbutil import AGG, C2_AGGS, assert_parity, host_col

pytestmark = pytest.mark.gpu

SENTINEL = np.array([0xFFF1A5A5A5A5A5A5], dtype=np.uint64)  # the tables' empty marker


def _stats():
    from cudf_amd import _lib
    return _lib.last_stats()


@pytest.mark.parametrize("dtype,low,card,n", [
    (np.int8, -128, 256, 300_000),            # negative keys of a narrow type
    (np.bool_, 0, 2, 20_000),
    (np.uint16, 65_000, 536, 70_001),
    (np.int32, -2**31, 1_000, 1_200_000),     # the type's smallest values
    (np.uint32, 2**32 - 700, 700, 600_001),
    (np.int64, 2**63 - 1_500, 1_500, 900_000),  # the type's largest
    (np.uint64, 2**63 - 20, 64, 50_000),      # across the sign bit
    (np.int64, int(SENTINEL.view(np.int64)[0]) - 30, 64, 50_000),  # around the empty marker: probed
])
@pytest.mark.parametrize("policy", [0, 1])
def test_keys_of_a_small_range(dtype, low, card, n, policy):
    rng = np.random.default_rng(n + policy)
    k = (rng.integers(0, card, n).astype(object) + low) if card > 2 else rng.integers(0, 2, n)
    k = np.array(k, dtype=dtype)
    key = host_col(k, rng.random(n) >= 0.02)
    f = host_col(rng.standard_normal(n).astype(np.float32), rng.random(n) >= 0.05)
    i = host_col(rng.integers(-1000, 1000, n))
    assert_parity([key], [(f, [(AGG["SUM"], 1), (AGG["MAX"], 1), (AGG["COUNT_VALID"], 1)]),
                          (i, [(AGG["SUM"], 1), (AGG["MIN"], 1), (AGG["MEAN"], 1), (AGG["COUNT_ALL"], 1)])], policy)
    assert _stats()["lds_preagg"] == 1.0


@pytest.mark.parametrize("n", [40_000, 1_500_000])
def test_keys_outside_the_sampled_range(n):
    """A few rows hold keys far from the others: whether the sample sees them
    or not, they get groups of their own."""
    rng = np.random.default_rng(n)
    k = rng.integers(0, 500, n)
    far = rng.choice(n, 40, replace=False)
    k[far] = 10**12 + rng.integers(0, 20, 40)
    v = host_col(rng.integers(-100, 100, n))
    assert_parity([host_col(k)], [(v, [(AGG["SUM"], 1), (AGG["MIN"], 1), (AGG["COUNT_ALL"], 1)])])


@pytest.mark.parametrize("card", [1, 63, 2_300, 4_000, 4_097])
def test_sparse_keys_and_special_floats(card):
    """Keys without a small range (probed tables, up to and past what LDS
    holds), values with NaN and infinities."""
    rng = np.random.default_rng(card)
    n = 400_003
    k = rng.integers(-2**62, 2**62, card)[rng.integers(0, card, n)]
    x = rng.standard_normal(n)
    x[rng.integers(0, n, 300)] = np.nan
    x[rng.integers(0, n, 30)] = np.inf
    f = host_col(x, rng.random(n) >= 0.1)
    assert_parity([host_col(k)], [(f, [(AGG["MIN"], 1), (AGG["MAX"], 1), (AGG["COUNT_VALID"], 1)]),
                                  (host_col(rng.integers(0, 9, n).astype(np.uint8)), [(AGG["SUM"], 1), (AGG["MAX"], 1)])])


@pytest.mark.parametrize("key_dtype,policy,nulls", [(np.int64, 0, 0.0), (np.int64, 1, 0.05), (np.int32, 1, 0.05),
                                                    (np.float64, 0, 0.05)])
def test_hot_keys_apart_from_the_rest(key_dtype, policy, nulls):
    """A third of the rows on 40 keys, the others on 300,000 more: the hot
    groups and the partitioned path's make one result, with every aggregation
    of both kinds of pass."""
    rng = np.random.default_rng(11)
    n = 1_300_007
    k = rng.integers(0, 300_000, n)
    hot = rng.random(n) < 0.34
    k[hot] = rng.integers(0, 40, int(hot.sum())) * 7
    k = k.astype(key_dtype)
    if key_dtype == np.int64:
        k[rng.integers(0, n, 5_000)] = SENTINEL.view(np.int64)[0]
    key = host_col(k, rng.random(n) >= nulls if nulls else None)
    f = host_col(rng.standard_normal(n) * 10 + 3, rng.random(n) >= nulls if nulls else None)
    i = host_col(rng.integers(0, 10_000, n).astype(np.int32), rng.random(n) >= 0.03)
    assert_parity([key], [(f, C2_AGGS), (i, C2_AGGS)], policy)
    st = _stats()
    assert st["strategy"] == 5 and st["hot_groups"] >= 40 and st["spilled_rows"] > n / 2, st


@pytest.mark.parametrize("n,card,general", [(199_999, 9_000, False), (200_000, 9_000, False), (600_001, 5_000, False),
                                            (1_100_003, 20_000, False), (299_999, 3_000, True), (300_000, 3_000, True)])
def test_path_for_the_rows_and_groups(n, card, general):
    """Both sides of the line between the device-wide table and the
    partitioned path (with few groups its bins are many and nearly empty)."""
    rng = np.random.default_rng(n)
    k = rng.integers(-2**40, 2**40, card)[rng.integers(0, card, n)]
    keys = [host_col(k, rng.random(n) >= 0.01)]
    if general:
        keys.append(host_col((k % 7).astype(np.int16)))
    v = host_col(rng.standard_normal(n), rng.random(n) >= 0.04)
    i = host_col(rng.integers(-9, 9, n).astype(np.int8))
    assert_parity(keys, [(v, C2_AGGS), (i, [(AGG["SUM"], 1), (AGG["MAX"], 1)])])
    assert _stats()["strategy"] == (2 if n >= (300_000 if general else 200_000) else 1)


@pytest.mark.parametrize("card", [1, 20, 700, 3_000])
@pytest.mark.parametrize("spread", [1, 1_000_003])
def test_variance_of_few_groups(card, spread):
    """The variance pass with the means in LDS, slots by value and by probe;
    null keys as a group; NaN, infinities and groups of one value."""
    rng = np.random.default_rng(card + spread)
    n = 90_001
    k = rng.integers(0, card, n) * spread
    k[:3] = [10**15, 10**15 + 1, -10**15]
    x = rng.standard_normal(n) * 1e3 + 1e5
    x[rng.integers(0, n, 5)] = np.nan
    x[rng.integers(0, n, 5)] = -np.inf
    key = host_col(k, rng.random(n) >= 0.02)
    assert_parity([key], [(host_col(x, rng.random(n) >= 0.05), [(AGG["VARIANCE"], 1), (AGG["STD"], 0), (AGG["COUNT_VALID"], 1)]),
                          (host_col(rng.integers(0, 50, n).astype(np.uint16)), [(AGG["VARIANCE"], 1), (AGG["MEAN"], 1)])], 1)


def _spread_over_mean(rng, n, card, kind):
    """Keys and float64 values whose mean is 20 standard deviations."""
    if kind == "hot":
        k = rng.integers(0, card, n)
        hot = rng.random(n) < 0.3
        k[hot] = rng.integers(0, 5, int(hot.sum()))
    else:
        k = rng.integers(0, card, n)
    return k * 1_000_003, rng.standard_normal(n) + 20.0


@pytest.mark.parametrize("kind,n,card", [("one", 300_001, 6_000), ("general", 400_003, 8_000), ("hot", 1_100_003, 20_000)])
def test_variance_subtracts_the_mean(kind, n, card):
    """Calls below a million rows or 65,536 groups, and the keys beside hot
    ones: M2 is the sum of squared deviations from the mean.  With u = 2^-53
    and m rows in a group every squared deviation is within 3u of itself and
    their sum within (m - 1)u, the mean's own error counts quadratically: at
    most (m + 5)u.  (The sum of squares less the squared sum would lose
    m * x^2 / sigma^2 = 400 m of the same units.)"""
    from cudf_amd import GroupBy, GroupByRequest, Table
    from cudf_amd.aggregation import Aggregation
    from tests.gbutil import to_device
    rng = np.random.default_rng(card)
    k, x = _spread_over_mean(rng, n, card, kind)
    keys = [host_col(k)] + ([host_col((k % 5).astype(np.int32))] if kind == "general" else [])
    out, res = GroupBy(Table([to_device(c) for c in keys])).aggregate(
        [GroupByRequest(to_device(host_col(x)), [Aggregation(AGG["VARIANCE"], 1), Aggregation(AGG["COUNT_VALID"])])])
    got_keys = out.columns()[0].to_numpy()[0]
    got = res[0].columns()[0].to_numpy()[0][np.argsort(got_keys)]
    order = np.argsort(k, kind="stable")
    uniq, first, count = np.unique(k[order], return_index=True, return_counts=True)
    xs = x[order].astype(np.longdouble)  # 64 bits of mantissa
    dev = xs - np.repeat(np.add.reduceat(xs, first) / count, count)
    many = count > 1
    want = np.add.reduceat(dev * dev, first)[many] / (count[many] - 1)
    err = np.abs((got[many] - want) / want).astype(np.float64)
    bound = (count[many] + 5) * 2.0**-53
    assert np.all(err <= bound), (err / bound).max()


def test_variance_when_the_hot_key_comes_last():
    """Zipf(2) keys: more groups than the estimate sized the LDS tables for,
    and the key of most rows in the last slots of the device-wide table.  Its
    rows must not queue up on one address (37 ms when they do, 0.1 ms else)."""
    from cudf_amd import _lib
    from oracle import oracle as orc
    rng = np.random.default_rng(3)
    n, card = 5_000_003, 2_500_000
    w = np.arange(1, card + 1, dtype=np.float64) ** -2.0
    rank = np.minimum(np.searchsorted(np.cumsum(w) / w.sum(), rng.random(n)), card - 1)
    candidates = np.arange(1, 200_000, dtype=np.int64) << 40
    slot = orc.hash_rows([host_col(candidates)]).astype(np.int64) & (2**14 - 1)
    ids = rng.permutation(card).astype(np.int64) * 1_000_003
    ids[0] = candidates[slot >= 2**14 - 4][0]
    v = host_col(rng.standard_normal(n))
    _lib.set_phase_timing(True)
    try:
        assert_parity([host_col(ids[rank])], [(v, [(AGG["VARIANCE"], 1), (AGG["MEAN"], 1)])])
        st = _stats()
    finally:
        _lib.set_phase_timing(False)
    assert st["lds_preagg"] == 1.0 and st["groups"] > 2.6 * st["est_groups"], st
    assert st["t_second_pass_ms"] < 4.0, st


@pytest.mark.parametrize("n,card,spread,lds", [
    (4_097, 170, 2**40, 1), (4_097, 1_500, 1, 0), (4_096, 20, 1, 0),   # up to 512 slots from the smallest estimated call on
    (41_000, 1_024, 1, 0), (41_500, 1_024, 1, 1),                      # 1,024 slots by value
    (90_000, 3_000, 2**40, 0), (900_000, 3_000, 2**40, 1),             # 9,000 by probe
    (20_000, 10, 1_000, 1),                                            # a wide range of few keys: by probe
])
@pytest.mark.parametrize("kinds", [["SUM", "MIN"], ["MEAN", "VARIANCE"]])
def test_rows_that_pay_for_tables(n, card, spread, lds, kinds):
    """Both sides of the line between LDS tables and the device-wide table."""
    rng = np.random.default_rng(n + card)
    k = np.concatenate([np.arange(card), rng.integers(0, card, n - card)])[rng.permutation(n)] * spread
    v = host_col(rng.integers(-1000, 1000, n))
    assert assert_parity([host_col(k)], [(v, [(AGG[a], 1) for a in kinds])]) == card
    if kinds[0] == "SUM" or card < 3_000:  # the variance tables hold fewer groups
        assert _stats()["lds_preagg"] == lds, _stats()


@pytest.mark.parametrize("n,card,keys,share,lds,strategy", [
    (60_000, 6_000, 1, 0.02, 0, 1),      # 1,200 rows of one key: an ordinary call
    (300_000, 20_000, 20, 0.05, 0, 2),   # 750 rows each
    (300_000, 25_000, 1, 0.01, 0, 2),
    (300_000, 25_000, 1, 0.02, 1, 1),    # 6,000 rows: hot, tables half filled
    (150_000, 50_000, 3, 0.3, 1, 1),
])
def test_hot_keys_by_their_rows(n, card, keys, share, lds, strategy):
    """A key is hot by its rows as well as by its share of them."""
    rng = np.random.default_rng(n + card)
    k = rng.integers(0, card, n)
    hot = rng.random(n) < share
    k[hot] = rng.integers(0, keys, int(hot.sum()))
    key = host_col(k * 1_000_003, rng.random(n) >= 0.005)
    f = host_col(rng.standard_normal(n) + 3, rng.random(n) >= 0.04)
    i = host_col(rng.integers(0, 10_000, n).astype(np.int32))
    assert_parity([key], [(f, C2_AGGS), (i, C2_AGGS)], 1)
    assert (_stats()["lds_preagg"], _stats()["strategy"]) == (lds, strategy), _stats()


@pytest.mark.parametrize("kind,n,card", [("one", 300_001, 6_000), ("general", 400_003, 3_000), ("hot", 1_100_003, 20_000)])
def test_memory_for_the_groups_only(kind, n, card, monkeypatch):
    """A memory resource with room for the groups found but not for what the
    partitioned path may find: the call takes the device-wide table, and every
    buffer of the attempt is given back."""
    from cudf_amd import groupby
    made = []

    class Limited(groupby.TorchMemoryResource):
        def __init__(self):
            super().__init__()
            self.refused = 0
            made.append(self)

        def _allocate(self, ctx, nbytes, stream):
            if nbytes > 12 * card + 64:
                self.refused += 1
                return None
            return super()._allocate(ctx, nbytes, stream)

    monkeypatch.setattr(groupby, "TorchMemoryResource", Limited)
    rng = np.random.default_rng(card)
    k, x = _spread_over_mean(rng, n, card, kind)
    key = host_col(k, rng.random(n) >= 0.01)
    keys = [key] + ([host_col((k % 5).astype(np.int32))] if kind == "general" else [])
    v = host_col(x, rng.random(n) >= 0.05)
    i = host_col(rng.integers(-100, 100, n).astype(np.int32))
    assert_parity(keys, [(v, [(AGG["SUM"], 1), (AGG["MAX"], 1), (AGG["VARIANCE"], 1)]),
                         (i, [(AGG["SUM"], 1), (AGG["MIN"], 1), (AGG["COUNT_ALL"], 1)])], 1)
    assert _stats()["strategy"] == 1
    assert made[0].refused > 0 and not made[0].live


@pytest.mark.parametrize("n,card,kinds,strategy", [
    (590_000, 9_000, ["SUM", "MIN", "MAX"], 1), (610_000, 9_000, ["SUM", "MIN", "MAX"], 2),
    (390_000, 9_000, ["SUM", "MIN", "MAX", "COUNT_ALL"], 1), (410_000, 9_000, ["SUM", "MIN", "MAX", "COUNT_ALL"], 2),
    (700_000, 9_000, ["SUM", "MAX"], 1), (310_000, 900, ["SUM"], 2),
])
def test_path_of_general_keys_by_accumulators(n, card, kinds, strategy):
    rng = np.random.default_rng(n)
    k = rng.integers(0, card, n)
    v = host_col(rng.integers(-1000, 1000, n))
    assert_parity([host_col((k % 89).astype(np.int16)), host_col(k)], [(v, [(AGG[a], 1) for a in kinds])])
    assert _stats()["strategy"] == strategy, _stats()
