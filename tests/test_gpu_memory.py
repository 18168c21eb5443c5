"""Calls whose allocations of device memory fail, one after another: every call gives its result by a form
that needs less scratch, or the out-of-memory error, and the calls after it are not affected."""
import threading

import numpy as np
import pytest

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
