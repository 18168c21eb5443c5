"""Calls whose allocations of device memory fail, one after another: every call gives its result by a form
that needs less scratch, or the out-of-memory error, and the calls after it are not affected."""
import threading

import numpy as np
import pytest
import torch

import arrowmetal_amd as am
import oracle_py as O

pytestmark = pytest.mark.gpu


def failing(call, check, k):
    """One call whose k-th allocation fails: (whether it failed, whether the call gave its result)."""
    am.fail_alloc(k)
    try:
        got = call()
        done = True
    except am.ArrowMetalError as e:
        assert "out of device memory" in str(e), e
        done = False
    finally:
        hit = am.fail_alloc(0) == 0
    if done:
        check(got)
    return hit, done


def test_a_thread_whose_table_could_not_be_had():
    """A thread's look-back table is allocated by its first sort: when that fails, its next one has it."""
    x = O.splitmix64(5, 60_001).astype(np.uint32).view(np.float32)
    want = O.argsort(x, None)
    a = am.MetalArray.from_numpy(x)
    outcomes = []

    def work(k):
        try:
            check = lambda r: np.testing.assert_array_equal(r.to_numpy()[0], want)
            outcomes.append(failing(a.argsort, check, k))
            check(a.argsort())
        except BaseException as e:   # reported by the test
            outcomes.append(e)

    for k in range(1, 30):
        t = threading.Thread(target=work, args=(k,))
        t.start()
        t.join()
        assert isinstance(outcomes[-1], tuple), outcomes[-1]
        if not outcomes[-1][0]:
            break
    assert not outcomes[-1][0] and len(outcomes) > 6, outcomes


def test_unique_rows_hold_the_kept_rows_only():
    n = 10_000_000
    rng = np.random.default_rng(4)
    a = am.MetalArray.from_numpy(rng.integers(-2**62, 2**62, 1000)[rng.integers(0, 1000, n)])
    held = [am.unique_rows([a])]
    before = torch.cuda.mem_get_info()[0]
    held += [am.unique_rows([a]) for _ in range(40)]
    assert all(len(r) == 1000 for r in held)
    assert before - torch.cuda.mem_get_info()[0] < 200 << 20


def wide_pair(n):
    rng = np.random.default_rng(7)
    return [rng.integers(-2**40, 2**40, n)[rng.integers(0, n, n)], rng.integers(0, 7, n).astype(np.int16)]


def unique_two():
    cols = wide_pair(200_003)
    want = O.unique_rows(cols, [None, None])
    arrays = [am.MetalArray.from_numpy(c) for c in cols]
    return lambda: am.unique_rows(arrays), lambda r: np.testing.assert_array_equal(r.to_numpy()[0], want)


def group_two():
    cols = wide_pair(200_003)
    ids, K, _ = O.group_keys(cols, [None, None])
    arrays = [am.MetalArray.from_numpy(c) for c in cols]

    def check(g):
        assert g.group_count == K
        np.testing.assert_array_equal(g.ids().to_numpy()[0], ids)
    return lambda: am.group_by(arrays), check


def take_random():
    n = 3 << 22
    x = O.splitmix64(3, n)
    at = np.random.default_rng(3).integers(0, n, n).astype(np.uint32)
    a, ix = am.MetalArray.from_numpy(x), am.MetalArray.from_numpy(at)
    return lambda: a.take(ix), lambda r: np.testing.assert_array_equal(r.to_numpy()[0], x[at])


def table():
    n = 100_003
    rng = np.random.default_rng(9)
    t = {"k": rng.standard_normal(n), "a": rng.integers(0, 9, n), "b": rng.integers(0, 99, n).astype(np.int16)}
    at = O.argsort(t["k"], None)
    src = am.PlanSource("t", {c: am.MetalArray.from_numpy(v) for c, v in t.items()})
    plan = {"op": "sort", "by": [["k", False]], "input": {"op": "scan", "source": "t"}}

    def check(got):
        for c, v in t.items():
            np.testing.assert_array_equal(got[c].to_numpy()[0], v[at])
    return lambda: am.plan_run(plan, [src]), check


def sorted_values():
    x = O.splitmix64(3, 100_003).astype(np.uint32).view(np.int32)
    valid = np.random.default_rng(2).random(len(x)) > 0.1
    a = am.MetalArray.from_numpy(x, valid)
    want = x[O.argsort(x, valid)]

    def check(r):
        got, gv = r.to_numpy()
        m = int(valid.sum())
        assert gv[:m].all() and not gv[m:].any()
        np.testing.assert_array_equal(got[:m], want[:m])
    return a.sort, check


def argsort_i32():
    x = O.splitmix64(4, 100_003).astype(np.uint32).view(np.int32)
    a = am.MetalArray.from_numpy(x)
    want = O.argsort(x, None)
    return a.argsort, lambda r: np.testing.assert_array_equal(r.to_numpy()[0], want)


# call, and how many of its allocations it can do without (their scratch has a form that needs less).
@pytest.mark.parametrize("make,spared", [(sorted_values, 12), (argsort_i32, 5),
                                         (unique_two, 14), (group_two, 1), (take_random, 5), (table, 1)])
def test_calls_with_a_form_that_needs_less_scratch(make, spared):
    call, check = make()
    check(call())
    outcomes = []
    for k in range(1, 200):
        outcomes.append(failing(call, check, k))
        check(call())
        if not outcomes[-1][0]:
            break
    assert not outcomes[-1][0], "more allocations than expected"
    assert sum(done for hit, done in outcomes if hit) >= spared, outcomes
