"""Calls share what a potential keeps (host buffer, neighborlist, tile sums): calls of
any size and choice of outputs after each other, after an error, and from two threads
at once give what a fresh potential gives."""

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
    _in_threads([lambda k=k: pot.execute_fixed_raw(*cases[k], 0.3) for k in range(2)], want[:2])


def _in_threads(calls, want, repeats=20):
    """Every call in a thread of its own, over and over: each result is its own."""
    failed = []

    def work(call, expect):
        for _ in range(repeats):
            failed.extend(1 for g, e in zip(call(), expect) if not np.array_equal(g, e))

    threads = [threading.Thread(target=work, args=a) for a in zip(calls, want)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert not failed


def _charges(rng, n, interpolated):
    g = int(np.ceil(n ** (1 / 3)))
    sites = np.stack(np.meshgrid(*[np.arange(g)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
    x = (sites + rng.uniform(0.2, 0.8, (n, 3))) * (3.0 / g)
    p = np.stack([rng.normal(size=n), np.full(n, 0.1), rng.uniform(0.3, 0.9, n)], 1)
    return x, np.concatenate([p, 0.9 * p]) if interpolated else p, np.eye(3) * 3.0


@pytest.mark.parametrize("interpolated", [False, True])
@pytest.mark.parametrize("n,same", [(700, True), (700, False)])
def test_threads_in_one_nonbonded_potential(gpu, n, same, interpolated):
    """The neighborlist and the tiles' sums belong to the potential: calls from two
    threads use them one after the other, alone or as a part that two sums share."""
    rng = np.random.default_rng(n + same)
    plane, offset = np.zeros(n, np.int32), (rng.random(n) < 0.05).astype(np.int32)
    kind = custom_ops.NonbondedAllPairs_f32_interpolated if interpolated else custom_ops.NonbondedAllPairs_f32

    def new():
        return kind(None, plane, offset, 2.0, 1.2)

    a = _charges(rng, n, interpolated)
    b = a if same else _charges(rng, n, interpolated)
    want = [new().execute_fixed_raw(*c, 0.4) for c in (a, b)]
    pot = new()
    _in_threads([lambda c=c: pot.execute_fixed_raw(*c, 0.4) for c in (a, b)], want)
    sums = [custom_ops.SummedPotential([pot], [a[1].size]), custom_ops.FanoutSummedPotential([pot])]
    _in_threads([lambda c=c, s=s: s.execute_fixed_raw(*c, 0.4) for c, s in zip((a, b), sums)], want)
    frames = np.stack([b[0]] * 2), b[1][None], np.stack([b[2]] * 2), np.array([0.4, 0.7]), True, True, True, True
    want_batch = new().execute_selective_batch(*frames)
    _in_threads([lambda: pot.execute_fixed_raw(*a, 0.4), lambda: pot.execute_selective_batch(*frames)],
                [want[0], want_batch], 8)


def test_call_after_an_error(gpu):
    """After a call refused on the host (box), one refused once its inputs were under
    way (parameter count), and one of a sum refused after its first part's launches."""
    rng = np.random.default_rng(0)
    n = 200
    x, p, box = _charges(rng, n, False)
    bond = _bond(n)
    bx, bp, bbox = _inputs(rng, n)
    pot = custom_ops.NonbondedAllPairs_f32(None, np.zeros(n, np.int32), np.zeros(n, np.int32), 2.0, 1.2)
    both = custom_ops.SummedPotential([pot, bond], [p.size, bp.size])
    wrong = custom_ops.SummedPotential([pot, bond], [p.size, bp.size - 1])
    fresh = custom_ops.NonbondedAllPairs_f32(None, np.zeros(n, np.int32), np.zeros(n, np.int32), 2.0, 1.2)
    want = fresh.execute_fixed_raw(x, p, box, 0.0)
    want_bond = _bond(n).execute_fixed_raw(bx, bp, bbox, 0.3)
    flat = np.concatenate([p.ravel(), bp.ravel()])
    want_both = custom_ops.SummedPotential([fresh, _bond(n)], [p.size, bp.size]).execute_fixed_raw(x, flat, box, 0.0)

    def same(got, expect):
        for g, e in zip(got, expect):
            np.testing.assert_array_equal(g, e)

    for _ in range(2):
        with pytest.raises(RuntimeError, match="half of the box width"):
            pot.execute(x, p, np.eye(3) * 1.5, 0.0)
        same(pot.execute_fixed_raw(x, p, box, 0.0), want)
        with pytest.raises(RuntimeError, match="expected P =="):
            bond.execute(bx, bp.ravel()[:-1], bbox, 0.3)
        same(bond.execute_fixed_raw(bx, bp, bbox, 0.3), want_bond)
        with pytest.raises(RuntimeError, match="expected P =="):
            wrong.execute(x, flat[:-1], box, 0.0)
        same(both.execute_fixed_raw(x, flat, box, 0.0), want_both)
        same(pot.execute_fixed_raw(x, p, box, 0.0), want)
