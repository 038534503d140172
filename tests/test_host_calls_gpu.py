"""Host calls share one kept buffer per potential: calls of any size and choice of
outputs after each other, after an error, and from two threads at once give what a
fresh potential gives."""

import threading

import numpy as np
import pytest

from timemachine_amd.lib import custom_ops

pytestmark = pytest.mark.gpu


def _bond(n):
    idxs = np.stack([np.arange(n - 1), np.arange(1, n)], 1).astype(np.int32)
    return custom_ops.HarmonicBond_f32(idxs)


def _inputs(rng, n):
    x = rng.normal(size=(n, 3))
    params = np.stack([rng.uniform(100, 200, n - 1), rng.uniform(0.1, 0.2, n - 1)], 1)
    return x, params, np.eye(3) * 10.0


@pytest.mark.parametrize("n,others", [(2, (2, 3)), (65, (70, 300, 65)), (1000, (5000, 1000, 1000))])
def test_calls_after_each_other_and_from_threads(gpu, n, others):
    rng = np.random.default_rng(n)
    pot = _bond(n)
    cases = [_inputs(rng, n)] + [(np.concatenate([rng.normal(size=(m, 3))]), *_inputs(rng, n)[1:]) for m in others
                                 if m >= n]
    want = [_bond(n).execute_fixed_raw(*c, 0.3) for c in cases]
    for c, w in zip(cases, want):
        for g, e in zip(pot.execute_fixed_raw(*c, 0.3), w):
            np.testing.assert_array_equal(g, e)
    only = pot.execute_selective(*cases[0], 0.3, False, False, False, True)
    assert only[0] is None and only[3] == pot.execute(*cases[0], 0.3)[3]
    failed = []

    def work(k):
        for _ in range(20):
            got = pot.execute_fixed_raw(*cases[k], 0.3)
            failed.extend(1 for g, e in zip(got, want[k]) if not np.array_equal(g, e))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert not failed


def test_call_after_an_error(gpu):
    rng = np.random.default_rng(0)
    n = 200
    x, p = rng.uniform(0, 4, (n, 3)), np.stack([rng.normal(size=n), np.full(n, 0.1), np.full(n, 0.5)], 1)
    zero = np.zeros(n, np.int32)
    pot = custom_ops.NonbondedAllPairs_f32(None, zero, zero, 2.0, 1.2)
    want = custom_ops.NonbondedAllPairs_f32(None, zero, zero, 2.0, 1.2).execute_fixed_raw(x, p, np.eye(3) * 4, 0.0)
    for _ in range(2):
        with pytest.raises(RuntimeError):
            pot.execute(x, p, np.eye(3) * 1.5, 0.0)
        for g, e in zip(pot.execute_fixed_raw(x, p, np.eye(3) * 4, 0.0), want):
            np.testing.assert_array_equal(g, e)
