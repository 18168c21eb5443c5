"""GPU parity of the radix argsort (am_argsort / am_argsort_ex / am_argsort_ex2) and am_take against the
CPU oracle, bit-exact, on the sizes and key shapes of the reference's own suites
(Tests/ArrowMetalTests/RadixSortScaleTests.swift:28-201, SortOptionsTests.swift, SortTests.swift)."""
import json
import os
import time

import numpy as np
import pytest

import arrowmetal_amd as am
import oracle_py as O

pytestmark = pytest.mark.gpu

GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")

# RadixSortScaleTests.swift:28-29: lane, chunk, block and pass-skip boundaries.
SIZES = [0, 1, 2, 31, 32, 33, 63, 64, 65, 255, 256, 257, 511, 512, 513, 4095, 4096, 4097, 65536,
         (1 << 18) - 1, 1 << 18, (1 << 18) + 1]


def gpu_argsort(vals, valid=None, desc=False, place=0, order=0):
    a = am.MetalArray.from_numpy(vals, valid)
    r = a.argsort(bool(desc), am.NULL_PLACEMENTS[place], am.FLOAT_ORDERS[order])
    assert r.format == "I"
    out, v = r.to_numpy()
    assert v is None
    return out


def check(vals, valid=None, desc=False, place=0, order=0, label=""):
    got = gpu_argsort(vals, valid, desc, place, order)
    want = O.argsort(vals, valid, desc, place, order)
    if not np.array_equal(got, want):
        bad = int(np.nonzero(got != want)[0][0])
        raise AssertionError(f"{label} n={len(vals)} desc={desc} place={place} order={order}: "
                             f"first difference at {bad}: got {got[bad]} want {want[bad]}")


@pytest.mark.parametrize("n", SIZES)
def test_int64_full_range_sizes(n):
    vals = O.splitmix64(0xA11CE501 + n, n).view(np.int64)
    for desc in (False, True):
        check(vals, None, desc, label="i64")


@pytest.mark.parametrize("n", [1, 33, 4097, 70001, (1 << 18) + 1])
def test_float64_orders_and_placements(n):
    rng = np.random.default_rng(n)
    f = rng.uniform(-1e3, 1e3, n).round(0)
    sp = np.array([np.nan, -np.nan, np.inf, -np.inf, -0.0, 0.0, 5e-324, -5e-324], dtype=np.float64)
    m = rng.random(n) < 0.1
    f[m] = sp[rng.integers(0, len(sp), int(m.sum()))]
    b = f.view(np.uint64)
    b[rng.random(n) < 0.01] = np.uint64(0x7FF0000000000001)     # signalling NaN payload
    valid = rng.random(n) >= 0.05
    for desc in (0, 1):
        for place in (0, 1):
            for order in (0, 1, 2):
                check(f, valid, desc, place, order, "f64")


def test_reference_vectors():
    with open(os.path.join(GOLDEN, "reference_vectors.json")) as fh:
        v = json.load(fh)
    s = v["sort_specials"]
    vals = np.array(s["values"], dtype=np.uint64).view(np.float64)
    valid = np.array(s["valid"], dtype=bool)
    assert gpu_argsort(vals, valid).tolist() == s["ascending"]
    assert gpu_argsort(vals, valid, desc=True).tolist() == s["descending"]
    t = v["sort_total_specials"]
    vals = np.array(t["values"], dtype=np.uint64).view(np.float64)
    valid = np.array(t["valid"], dtype=bool)
    assert gpu_argsort(vals, valid, desc=True).tolist() == t["desc_ieee"]
    assert gpu_argsort(vals, valid, desc=True, order=1).tolist() == t["desc_total"]


def test_pyarrow_fixtures():
    fx = np.load(os.path.join(GOLDEN, "sort_fixtures.npz"))
    for n in [0, 1, 2, 33, 257, 4097, 20001]:
        f = fx[f"f64_{n}_bits"].view(np.float64)
        valid = fx[f"f64_{n}_valid"]
        ints = fx[f"i64_{n}_vals"]
        for desc in (0, 1):
            for pl, place in ((0, "at_end"), (1, "at_start")):
                np.testing.assert_array_equal(gpu_argsort(f, valid, desc, pl, 0), fx[f"f64_{n}_ieee_{desc}_{place}"])
                np.testing.assert_array_equal(gpu_argsort(f, valid, desc, pl, 1), fx[f"f64_{n}_total_{desc}_{place}"])
                np.testing.assert_array_equal(gpu_argsort(ints, valid, desc, pl), fx[f"i64_{n}_{desc}_{place}"])


@pytest.mark.parametrize("n", [4097, (1 << 18) + 1, 1 << 20])
def test_key_shapes(n):
    rng = np.random.default_rng(7)
    # All keys equal (every pass skipped; the single pass is a stable compaction).
    check(np.full(n, 42, dtype=np.int64), None, label="all-equal")
    check(np.full(n, 42, dtype=np.int64), rng.random(n) > 0.5, True, 1, label="all-equal-nulls")
    # Constant high digits, then constant low digits (pass skipping both ways).
    check(rng.integers(0, 256, n).astype(np.int64), None, label="low-byte-only")
    check((rng.integers(0, 256, n).astype(np.int64) << 40) | 0x55, None, True, label="one-mid-byte")
    # Monotone input, both directions.
    check(np.arange(n, dtype=np.int64), None, label="ascending-input")
    check(np.arange(n, 0, -1, dtype=np.int64), None, label="descending-input")
    # Nulls at 1/1000, 1/4, 1/2, and all null.
    vals = rng.integers(-1000, 1000, n).astype(np.int64)
    for frac in (0.001, 0.25, 0.5, 1.0):
        valid = rng.random(n) >= frac
        for place in (0, 1):
            check(vals, valid, False, place, label=f"nulls {frac}")
            check(vals, valid, True, place, label=f"nulls {frac}")


@pytest.mark.parametrize("seed", range(6))
def test_full_range_columns_are_not_taken_for_skewed(seed):
    """Below 2^24 rows, where a top digit may hold 1 / 64 of the rows, chance alone fills none of the sample."""
    x = O.splitmix64(seed + 1, (1 << 24) - 5).astype(np.uint32).view(np.int32)
    a = am.MetalArray.from_numpy(x)
    am.prof_reset()
    am.prof_enable(True)
    got = a.argsort().to_numpy()[0]
    am.prof_enable(False)
    names = set(am.prof_report())
    am.prof_reset()
    assert "sort_msd_first" in names, sorted(names)
    if seed == 0:
        np.testing.assert_array_equal(got, O.argsort(x, None))


@pytest.mark.parametrize("n", [1 << 16, 300_001, 2_000_003])
@pytest.mark.parametrize("case,sweeps", [("small", 1), ("rare", 1), ("sampled_wide", 2), ("all_null", 1), ("one_value", 1),
                                         ("hot", 1)])
def test_analysis_of_32_bit_columns(case, sweeps, n):
    """Columns that the LSD passes sort are counted for them in the first analysis, by a sample of 4 neighbours
    at 16 places; a sample that misses the wide values, or sees nothing else, still leaves a sorted column."""
    rng = np.random.default_rng(n)
    x = rng.integers(-30_000, 30_000, n).astype(np.int32) if case == "hot" else rng.integers(0, 5000, n).astype(np.int32)
    wide = O.splitmix64(9, n).astype(np.uint32).view(np.int32)
    valid = rng.random(n) > 0.1
    places = ((n - 4) * np.arange(16) // 15)[:, None] + np.arange(4)
    if case == "rare": x[places[:-1, 0] + 50] = wide[:15]
    elif case == "sampled_wide": x[places.ravel()] = wide[places.ravel()]
    elif case == "all_null": valid[:] = False
    elif case == "one_value": x[:] = -77
    elif case == "hot": x = np.where(rng.random(n) < 0.97, x & 0xFFFF, wide).astype(np.int32)
    if case == "hot": sweeps = 1 if n > 300_001 else None       # up to 2^18 rows on a digit the hybrid sort takes it
    if case == "sampled_wide" and n <= 1 << 18: sweeps = None
    for va, desc, place in ((valid, 1, 0), (None, 0, 1)):
        am.prof_reset()
        am.prof_enable(True)
        got = gpu_argsort(x, va, desc, place, 0)
        am.prof_enable(False)
        ran = am.prof_report()
        if sweeps is not None:
            assert ran["sort_upsweep"][0] == sweeps and "sort_msd_first" not in ran, sorted(ran.items())
        np.testing.assert_array_equal(got, O.argsort(x, va, desc, place, 0))


@pytest.mark.parametrize("dtype", [np.int32, np.uint32, np.float32, np.int8, np.int16, np.uint8, np.uint16, np.uint64])
def test_other_key_widths(dtype):
    rng = np.random.default_rng(3)
    n = 70001
    if np.dtype(dtype).kind == "f":
        vals = rng.uniform(-100, 100, n).astype(dtype)
        vals[::37] = np.nan
        vals[::41] = -0.0
    else:
        info = np.iinfo(dtype)
        vals = rng.integers(info.min, info.max, n, dtype=dtype, endpoint=True)
    valid = rng.random(n) > 0.1
    for desc in (0, 1):
        for place in (0, 1):
            for order in ((0, 1, 2) if np.dtype(dtype).kind == "f" else (0,)):
                check(vals, valid, desc, place, order, str(np.dtype(dtype)))


def test_offset_slice_import():
    rng = np.random.default_rng(1)
    vals = rng.integers(-50, 50, 10000).astype(np.int64)
    valid = rng.random(10000) > 0.2
    for off in (0, 3, 64, 1001):
        a = am.MetalArray.from_numpy(vals, valid, offset=off)
        got, v = a.argsort(True, "at_start").to_numpy()
        want = O.argsort(vals[off:], valid[off:], True, 1)
        np.testing.assert_array_equal(got, want)


def test_repeat_determinism():
    vals = O.splitmix64(99, 300001).view(np.int64) >> 40      # many duplicate keys
    first = gpu_argsort(vals)
    for _ in range(3):
        np.testing.assert_array_equal(gpu_argsort(vals), first)


def test_bad_float_order_is_an_error():
    a = am.MetalArray.from_numpy(np.arange(4, dtype=np.float64))
    with pytest.raises(am.ArrowMetalError, match="unknown float_order 7"):
        a.argsort(False, "at_end", 7)


def test_batch_matches_unbatched():
    vals = O.splitmix64(5, 100000).view(np.int64)
    a = am.MetalArray.from_numpy(vals)
    want = a.argsort().to_numpy()[0]
    with am.batch():
        r1 = a.argsort()
        r2 = a.argsort(True)
    np.testing.assert_array_equal(r1.to_numpy()[0], want)
    np.testing.assert_array_equal(r2.to_numpy()[0], O.argsort(vals, None, True))


@pytest.mark.parametrize("n", [1, 63, 64, 65, 255, 256, 257, 4097, 16383, 16384, 16385, 40001])
def test_small_inputs_of_every_width(n):
    """Up to 16,384 rows the argsort ranks by counting (one launch), above it takes the passes: the edges
    of a workgroup's 64 rows and of the padding, for every key width, with many ties, the largest and the
    smallest key (a value whose mapped key is all ones beside NaN and null rows), nulls at both ends."""
    rng = np.random.default_rng(n)
    valid = rng.random(n) >= 0.3
    for dt in (np.int64, np.uint64, np.int32, np.uint32, np.int16, np.uint8, np.float64, np.float32):
        if np.issubdtype(dt, np.integer):
            lo, hi = np.iinfo(dt).min, np.iinfo(dt).max
            vals = np.where(rng.random(n) < 0.5, rng.choice(np.array([lo, 0, hi], dtype=dt), n),
                            rng.integers(lo, hi, n, dtype=dt, endpoint=True))
        else:
            vals = rng.choice(np.array([np.nan, -np.nan, np.inf, -np.inf, -0.0, 0.0, 1.5], dtype=dt), n)
        vals = vals.astype(dt)
        for desc, place, order in ((0, 0, 0), (1, 1, 0), (1, 0, 1), (0, 1, 2)):
            check(vals, valid, desc, place, order, str(dt))
        check(vals, None, 0, 0, 0, str(dt))
        check(vals, np.zeros(n, bool), 1, 0, 0, str(dt))


@pytest.mark.parametrize("dtype,n,shape,path", [
    (np.int32, (1 << 16) - 1, "wide", "lsd"), (np.int32, 1 << 16, "wide", "msd"), (np.uint32, 300_001, "wide", "msd"),
    (np.int32, 3_000_001, "wide", "msd"), (np.int32, 3_000_001, "small", "lsd"), (np.int32, 2_000_003, "skewed", "lsd"),
    (np.uint32, 1_500_007, "runs", "msd"), (np.int32, 200_003, "two_digits", "msd"), (np.float32, (1 << 24) + 3, "wide", "msd"),
    (np.float32, 1_000_003, "wide", "lsd"), (np.int64, 16_385, "wide", "msd"), (np.int64, 20_001, "small", "lsd"),
    (np.uint64, 40_000, "one_key", "lsd")])
def test_hybrid_sort_of_each_key_type(dtype, n, shape, path):
    """Where each key type takes the hybrid sort: 32-bit keys with and without a level, long equal runs (the
    LSD queue and copies), a top-digit bucket too large for it, a constant top digit (the LSD passes over the
    digits that vary), nulls at both ends, both directions."""
    rng = np.random.default_rng(n)
    dt = np.dtype(dtype)
    if dt.kind == "f":
        vals = (rng.random(n) * 2e6 - 1e6).astype(dt)
        vals[::1001] = np.nan
        vals[::997] = -0.0
    else:
        vals = O.splitmix64(n, n).view(np.uint64).astype(np.uint64)
        vals = (vals >> np.uint64(64 - 8 * dt.itemsize)).astype(f"u{dt.itemsize}").view(dt) if dt.itemsize == 4 else vals.view(dt)
        if shape == "small": vals = (vals & dt.type(0xFFF)).astype(dt)
        elif shape == "one_key": vals = np.full(n, 77, dt)
        elif shape == "skewed": vals = np.where(rng.random(n) < 0.9, vals & dt.type(0xFFFFF), vals).astype(dt)
        elif shape == "runs": vals = np.where(rng.random(n) < 0.5, vals[rng.integers(0, 3000, n)], vals).astype(dt)
        elif shape == "two_digits": vals = (vals & dt.type(0x7F0000FF)).astype(dt)
    valid = rng.random(n) >= 0.03
    for va, desc, place in ((valid, 1, 0), (None, 0, 0), (valid, 0, 1)):
        am.prof_reset()
        am.prof_enable(True)
        got = gpu_argsort(vals, va, desc, place, 0)
        am.prof_enable(False)
        names = set(am.prof_report())
        assert ("sort_msd_first" in names) == (path == "msd"), names
        np.testing.assert_array_equal(got, O.argsort(vals, va, desc, place, 0))


@pytest.mark.parametrize("dtype", [np.int32, np.uint64])
@pytest.mark.parametrize("shape", ["runs", "top_digit_only"])
def test_runs_of_equal_keys_at_the_edges_of_a_copy(dtype, shape):
    """Runs of equal keys leave the sort as copies of 4,096 rows each: runs of about that many rows and of
    several times as many, among keys that are all different, and keys that differ in their top digit alone."""
    rng = np.random.default_rng(3)
    bits = 8 * np.dtype(dtype).itemsize
    lens = [4095, 4096, 4097, 8191, 8192, 8193, 50_000, 1, 2]
    keys = O.splitmix64(11, len(lens)) >> np.uint64(64 - bits)
    if shape == "top_digit_only":
        keys = np.arange(1, len(lens) + 1, dtype=np.uint64) << np.uint64(bits - 5)
        x = np.repeat(keys, lens)
    else:
        x = np.concatenate([np.repeat(keys, lens), O.splitmix64(12, 60_000) >> np.uint64(64 - bits)])
    x = rng.permutation(x).astype(f"u{bits // 8}").view(dtype)
    valid = rng.random(len(x)) > 0.01
    for va, desc, place in ((None, False, 0), (valid, True, 1)):
        a = am.MetalArray.from_numpy(x, va)
        want = O.argsort(x, va, desc, place, 0)
        got, names = sort_with_kernels(x, va, desc, place, 0)
        assert "sort_msd_local" in names, sorted(names)
        np.testing.assert_array_equal(got, want)
        ok = np.ones(len(x), bool) if va is None else va
        vals, gv = a.sort(desc, am.NULL_PLACEMENTS[place]).to_numpy()
        gv = np.ones(len(x), bool) if gv is None else gv
        np.testing.assert_array_equal(gv, ok[want])
        np.testing.assert_array_equal(vals[gv], x[want][gv])
        np.testing.assert_array_equal(am.unique_rows([a]).to_numpy()[0], O.unique_rows([x], [va]))


@pytest.mark.parametrize("call", ["argsort", "sort", "unique"])
def test_a_hot_value_costs_no_more_than_the_rest(call):
    """30% of 32M int32 rows on one value: about the time of the column without it (a lone workgroup copying
    the value's rows would take ten times as long)."""
    n = 32_000_000
    rng = np.random.default_rng(1)
    x = rng.integers(-2**31, 2**31 - 1, n, dtype=np.int32)
    hot = np.where(rng.random(n) < 0.3, np.int32(12345), x)
    times = []
    for col in (x, hot):
        a = am.MetalArray.from_numpy(col)
        run = (lambda: am.unique_rows([a])) if call == "unique" else getattr(a, call)
        run()
        t = []
        for _ in range(5):
            t0 = time.perf_counter()
            run()
            t.append(time.perf_counter() - t0)
        times.append(min(t))
    print(call, [f"{t * 1e6:.0f} us" for t in times], flush=True)
    assert times[1] < 3 * times[0]


# ---------------------------------------------------------------- take


def test_take_matches_oracle():
    rng = np.random.default_rng(4)
    n = 100003
    vals = rng.uniform(-1e6, 1e6, n)
    valid = rng.random(n) > 0.1
    a = am.MetalArray.from_numpy(vals, valid)
    for it in (np.int32, np.int64, np.uint32):
        idx = rng.integers(0, n, 77777).astype(it)
        ivalid = rng.random(77777) > 0.05
        got, gv = a.take(am.MetalArray.from_numpy(idx, ivalid)).to_numpy()
        want, wv = O.take(vals, idx, valid, ivalid)
        np.testing.assert_array_equal(gv, wv)
        np.testing.assert_array_equal(got.view(np.uint64)[wv], want.view(np.uint64)[wv])
    got, gv = a.take(np.arange(n, dtype=np.uint32)[::-1].copy()).to_numpy()
    np.testing.assert_array_equal(got.view(np.uint64)[gv], vals[::-1].view(np.uint64)[gv])


@pytest.mark.parametrize("n", [1, 63, 64, 65, 255, 256, 1023, 1024, 1025, 70001])
def test_take_null_counts(n):
    """The null count and bitmap at the edges of a wave's rows and of a workgroup's (256 rows x 4): nulls in
    the values, in the indices, in both, and a result without any."""
    rng = np.random.default_rng(n)
    vals = rng.integers(-100, 100, 501).astype(np.int16)
    valid = rng.random(501) > 0.3
    idx = rng.integers(0, 501, n).astype(np.int32)
    ivalid = rng.random(n) > 0.5
    for va, iva in ((valid, None), (None, ivalid), (valid, ivalid), (None, None)):
        r = am.MetalArray.from_numpy(vals, va).take(am.MetalArray.from_numpy(idx, iva))
        want, wv = O.take(vals, idx, va, iva)
        got, gv = r.to_numpy()
        gv = np.ones(n, bool) if gv is None else gv
        assert r.null_count == n - int(wv.sum())
        np.testing.assert_array_equal(gv, wv)
        np.testing.assert_array_equal(got[wv], want[wv])
    empty = am.MetalArray.from_numpy(np.zeros(0, np.int64))
    assert empty.take(am.MetalArray.from_numpy(idx, np.zeros(n, bool))).null_count == n


@pytest.mark.parametrize("dtype,itype,n,length", [
    (np.float32, np.int32, 3 << 22, 1 << 22),                    # whole tiles, the smallest source
    (np.int32, np.uint32, (3 << 22) + 1, 2 * ((3 << 22) + 1)),   # a tile of one row, the largest source
    (np.float64, np.int64, (3 << 22) + 16_383, 1 << 21),
    (np.int64, np.uint32, (3 << 23) + 5, (1 << 25) + 7),
    (np.float32, np.int64, (3 << 22) - 1, 1 << 23),              # the plain gather on either side of the rule
    (np.float32, np.int32, 3 << 22, (3 << 23) + 1),
])
def test_take_by_slices(dtype, itype, n, length):
    """Large gathers: random indices by source slice, neighbours and windows directly, a bad index in the last row."""
    rng = np.random.default_rng(n)
    vals = np.arange(length, dtype=np.uint32).astype(dtype) if dtype != np.float32 \
        else np.arange(length, dtype=np.uint32).view(np.float32)   # every bit pattern is one of its own
    a = am.MetalArray.from_numpy(vals)
    bits = np.uint32 if vals.itemsize == 4 else np.uint64
    idx = rng.integers(0, length, n).astype(itype)
    seq = (np.arange(n, dtype=np.int64) % length).astype(itype)
    for ix in (idx, seq, np.minimum(seq // 4096 * 4096 + idx % 4096, length - 1).astype(itype)):
        got, gv = a.take(am.MetalArray.from_numpy(ix)).to_numpy()
        assert gv is None or gv.all()
        assert np.array_equal(got.view(bits), vals.view(bits)[ix])
    idx[-1] = length
    with pytest.raises(am.ArrowMetalError, match=rf"take: index out of range \(array length {length}\)"):
        a.take(am.MetalArray.from_numpy(idx))


def test_take_out_of_range():
    a = am.MetalArray.from_numpy(np.arange(10, dtype=np.int64))
    with pytest.raises(am.ArrowMetalError, match=r"take: index out of range \(array length 10\)"):
        a.take(np.array([1, 10], dtype=np.int64))
    with pytest.raises(am.ArrowMetalError, match="out of range"):
        a.take(np.array([-1], dtype=np.int32))


def test_order_by_gather_config_shape():
    """ORDER BY: argsort descending nulls last, then gather a float64 payload (20 B/row)."""
    n = 1_000_003
    keys = (O.splitmix64(0xB0B, n) >> np.uint64(1)).view(np.int64) - (1 << 62)
    valid = (O.splitmix64(0xC0C, n) >> np.uint64(11)).astype(np.float64) / 2.0**53 < 0.98
    payload = (O.splitmix64(0xD0D, n) >> np.uint64(11)).astype(np.float64) / 2.0**53 * 2e6 - 1e6
    k = am.MetalArray.from_numpy(keys, valid)
    p = am.MetalArray.from_numpy(payload)
    idx = k.argsort(True, "at_end")
    got = p.take(idx).to_numpy()[0]
    want_idx = O.argsort(keys, valid, True, 0)
    np.testing.assert_array_equal(idx.to_numpy()[0], want_idx)
    np.testing.assert_array_equal(got, payload[want_idx])


@pytest.mark.parametrize("order", [0, 1])
@pytest.mark.parametrize("width", [8, 4])
def test_large_tiles_first_pass_and_nulls(order, width):
    """9M rows, NaN and null bins included, against the oracle. 64-bit keys take the hybrid sort;
    32-bit float keys keep the LSD passes below 2^24 rows, whose scatter passes take 20 keys per thread above 8.4M rows and
    whose first pass takes 16: both tile shapes and their look-back chains."""
    n = 9_000_001
    print(f"large sort n={n} order={order} width={width}", flush=True)
    bits = O.splitmix64(0x1A2B + order, n)
    valid = (O.splitmix64(0x3C4D, n) >> np.uint64(11)).astype(np.float64) / 2.0**53 < 0.97
    if order == 0:
        vals = (bits >> np.uint64(1)).view(np.int64) - (1 << 62)
        if width == 4:
            vals = (vals >> 32).astype(np.int32)
    else:
        vals = ((bits >> np.uint64(11)).astype(np.float64) / 2.0**53 - 0.5) * 1e6
        vals[(bits & np.uint64(1023)) == 7] = np.nan
        vals[(bits & np.uint64(1023)) == 9] = -0.0
        if width == 4:
            vals = vals.astype(np.float32)
    for desc, place in ((True, 0), (False, 1)):
        check(vals, valid, desc, place, order, label="large")


def sort_with_kernels(vals, valid=None, desc=False, place=0, order=0):
    """The GPU argsort with kernel timing on: (indices, names of the kernels it launched)."""
    am.prof_reset()
    am.prof_enable(True)
    try:
        got = gpu_argsort(vals, valid, desc, place, order)
    finally:
        am.prof_enable(False)
    names = set(am.prof_report())
    am.prof_reset()
    return got, names


def msd_case(case, n):
    bits = O.splitmix64(0x7E57 + len(case), n)
    if case == "uniform":
        return bits.view(np.int64), None, "hybrid"
    if case == "low_digits_constant":   # only the top two digits vary: the local sort has no pass
        return ((bits & np.uint64(0xFFFF000000000000)) | np.uint64(0x1234)).view(np.int64), None, "hybrid"
    if case == "correlated_top":        # second digit equals the top one: every top bucket is carried a level
        top = bits >> np.uint64(56)
        k = (top << np.uint64(56)) | (top << np.uint64(48)) | (bits & np.uint64((1 << 48) - 1))
        return k.view(np.int64), None, "hybrid"
    if case == "duplicates":            # one key on 0.5% of the rows: a bucket that goes down every level
        k = bits.copy()
        k[(bits % np.uint64(200)) == 3] = np.uint64(0x0123456789ABCDEF)
        return k.view(np.int64), None, "hybrid"
    if case == "few_distinct":          # 3,000 distinct keys: buckets of equal keys, carried, then copied
        return O.splitmix64(0xD15, 3000)[(bits >> np.uint64(5)) % np.uint64(3000)].view(np.int64), None, "hybrid"
    if case == "narrow_floats":         # float64 in [1, 2) and [-2, -1): two top digits, the levels go deeper
        v = 1.0 + (bits >> np.uint64(12)).astype(np.float64) / 2.0**52
        v[(bits & np.uint64(1)) == 1] *= -1.0
        return v, None, "hybrid"
    if case == "repeats":               # 1/16 of the rows on 2,000 keys (~140 each): runs the bucket LSD queue
        k = bits.copy()
        pick = (bits >> np.uint64(7)) % np.uint64(16) == 0
        k[pick] = O.splitmix64(0x5EED, 2000)[(bits[pick] >> np.uint64(20)) % np.uint64(2000)]
        return k.view(np.int64), None, "hybrid"
    if case == "wide_buckets":          # top 16 bits from 1,500 values: ~3,000-row buckets, 16 keys per thread
        tops = np.unique(O.splitmix64(0x70B5, 1600) >> np.uint64(48))[:1500] << np.uint64(48)
        k = tops[(bits >> np.uint64(3)) % np.uint64(len(tops))] | (bits & np.uint64(0x0000FFFFFFFFFFFF))
        return k.view(np.int64), None, "hybrid"
    if case == "half_range":            # the ORDER BY keys: [-2^62, 2^62), 128 top digits, ~1,500-row buckets
        return ((bits >> np.uint64(1)).view(np.int64) - (1 << 62)), None, "hybrid"
    if case == "float_bits":            # random bit patterns: every exponent, NaNs, infinities, -0.0
        v = bits.view(np.float64).copy()
        # Equal keys must fit one LDS bucket (4096 rows): about 450 rows of -0.0, and a quarter of
        # the 1-in-2048 NaN patterns kept (nan_largest orders every NaN as one key).
        v[(bits % np.uint64(9973)) == 5] = -0.0
        drop = np.isnan(v) & ((bits >> np.uint64(3)) % np.uint64(4) != 0)
        v[drop] = (bits[drop] >> np.uint64(11)).astype(np.float64)
        valid = (bits >> np.uint64(20)) % np.uint64(33) != 0
        return v, valid, "hybrid"
    if case == "skewed":                # top digit nearly constant: the estimate sends it to the LSD passes
        return (bits >> np.uint64(10)).view(np.int64), None, "lsd"
    raise ValueError(case)


@pytest.mark.parametrize("case", ["uniform", "low_digits_constant", "correlated_top", "duplicates",
                                  "few_distinct", "narrow_floats", "repeats", "wide_buckets", "half_range",
                                  "float_bits", "skewed"])
def test_msd_hybrid_and_fallback(case):
    """64-bit keys above 4M rows whose top digit varies take the hybrid sort: a stable partition by the
    top digit, then level by level a segmented partition of every bucket above 4096 rows by the next
    digit (buckets whose rows share the digit carried without moving), then an LDS sort of each
    bucket by its remaining digits (LSD passes in LDS for buckets with many equal keys, a copy for
    buckets of equal keys). A constant top digit keeps the LSD passes. Each case checks the path it
    took and the order against the oracle."""
    n = 4_500_000
    vals, valid, path = msd_case(case, n)
    combos = [(False, 0, 0), (True, 1, 0)] + ([(False, 1, 1), (True, 0, 2)] if vals.dtype == np.float64 else [])
    for desc, place, order in combos:
        print(f"msd case={case} n={n} desc={desc} place={place} order={order}", flush=True)
        got, names = sort_with_kernels(vals, valid, desc, place, order)
        want = O.argsort(vals, valid, desc, place, order)
        if not np.array_equal(got, want):
            bad = int(np.nonzero(got != want)[0][0])
            raise AssertionError(f"{case} desc={desc} place={place} order={order}: first difference at {bad}: "
                                 f"got {got[bad]} want {want[bad]}")
        bucket_sort = "sort_msd_local" in names or "sort_msd_group" in names
        took = ("hybrid" if bucket_sort else "fallback" if "sort_msd_first" in names else "lsd")
        assert took == path, f"{case}: took the {took} path, kernels {sorted(names)}"


def test_msd_list_overflow_falls_back(monkeypatch):
    """A hybrid sort whose bucket-sort list runs out of room (forced here by capping the list at 64
    entries) drops the bucket sort and finishes with the LSD passes, whose order is the same."""
    monkeypatch.setenv("ARROWMETAL_MSD_LIST_CAP", "64")
    vals, valid, _ = msd_case("uniform", 4_500_000)
    for desc, place, order in ((False, 0, 0), (True, 1, 0)):
        print(f"msd list overflow desc={desc} place={place}", flush=True)
        got, names = sort_with_kernels(vals, valid, desc, place, order)
        want = O.argsort(vals, valid, desc, place, order)
        assert np.array_equal(got, want), f"desc={desc}: first difference at {int(np.nonzero(got != want)[0][0])}"
        assert "sort_msd_first" in names and "sort_msd_local" not in names and "sort_msd_group" not in names, \
            sorted(names)


@pytest.mark.parametrize("n", [1 << 18, 300_007, 1_000_000, (1 << 22) - 1])
@pytest.mark.parametrize("case", ["uniform", "float_bits", "half_range", "duplicates"])
def test_msd_hybrid_small_inputs(n, case):
    """From 2^18 rows, 64-bit keys take the hybrid sort with 4K-row units (16K from 2^22 rows): units
    that end inside a tile, top-digit buckets that go straight to the bucket sort, and the levels
    when a bucket is larger."""
    vals, valid, _ = msd_case(case, n)
    for desc, place, order in ((False, 0, 0), (True, 1, 1)):
        print(f"small msd case={case} n={n} desc={desc} place={place} order={order}", flush=True)
        got, names = sort_with_kernels(vals, valid, desc, place, order)
        want = O.argsort(vals, valid, desc, place, order)
        if not np.array_equal(got, want):
            bad = int(np.nonzero(got != want)[0][0])
            raise AssertionError(f"{case} n={n}: first difference at {bad}: got {got[bad]} want {want[bad]}")
        assert "sort_msd_local" in names or "sort_msd_group" in names, f"{case} n={n}: kernels {sorted(names)}"
