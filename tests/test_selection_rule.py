"""The one-wave selection's rule, as it is restated in selection_rule.py, against the oracle's selection over the probabilities: what it accepts is the
selection, and what it must not accept it leaves alone."""
import numpy as np
import pytest

import selection_rule as rule


def test_accepted_rows_are_the_selection(oracle):
    """Rows whose logits around the k-th crowd within and around the differences that the rule asks for, of several magnitudes."""
    rng = np.random.default_rng(20261205)
    accepted = refused = 0
    for trial in range(4000):
        n, k = ((64, 6), (128, 10), (512, 10), (264, 15))[trial % 4]
        l = (rng.normal(-6.0, 0.5, n) * 2.0 ** rng.uniform(-4, 1)).astype(np.float32)
        where = rng.permutation(n)
        l[where[:k - 1]] = (4.0 + np.arange(k - 1)).astype(np.float32)
        at = np.float32(rng.choice([-1.0, 1.0]) * 2.0 ** rng.uniform(-5, 1.5))
        crowd = where[k - 1:k + 3]
        l[crowd] = (at + rng.uniform(-1, 1, crowd.size) * 2.0 ** rng.uniform(-22, -14)).astype(np.float32)
        ok, ids = rule.select(l, k)
        if ok:
            accepted += 1
            assert np.array_equal(ids, oracle.route(l, k)[0]), (trial, l[crowd])
        refused += not ok
    assert accepted > 800 and refused > 800


def test_a_logit_of_the_same_probability_and_a_lower_id_is_not_forgotten(oracle):
    l, k = np.linspace(-3.0, -0.5, 64).astype(np.float32), 6
    l[[3, 9, 17, 33, 50]] = np.array([4.0, 3.5, 3.0, 2.5, 2.0], np.float32)
    l[[40, 30]] = [np.float32(float.fromhex(v)) for v in ("0x1.3d74p-1", "0x1.3d73fep-1")]
    want, _ = oracle.route(l, k)
    p = oracle.softmax_row(l)
    assert p[40] == p[30] and want[-1] == 30
    ok, ids = rule.select(l, k, gap=np.float32(0), gap_last=np.float32(0))
    assert ok and ids[-1] == 40            # negative control: by the order of the logits alone it is the wrong one
    assert not rule.select(l, k)[0]


def test_rows_that_are_left_to_the_rungs():
    base = np.linspace(-2.0, 2.0, 64).astype(np.float32)
    assert rule.select(base, 6)[0]
    for value in (np.nan, -np.float32(np.nan), np.inf, base[-1]):   # (the last: a tie of the largest)
        row = base.copy()
        row[5] = value
        assert not rule.select(row, 6)[0], value
    row = np.full(64, -np.inf, np.float32)
    row[:7] = base[:7]
    assert rule.select(row, 6)[0] and not rule.select(row, 7)[0]     # six and a seventh that is finite; seven and none
    row = base.copy()
    row[:6] += np.float32(200)
    assert not rule.select(row, 7)[0]                                # the seventh is below what has a normal exponential
    assert rule.select(base[:8], 8)[0]                               # every expert


@pytest.mark.parametrize("n,k", [(512, 10), (512, 15), (512, 11), (256, 8), (128, 10), (64, 10)])
def test_crowded_rows_are_accepted_up_to_lists_of_64(oracle, n, k):
    seen = set()
    for seed in range(20):
        for length, row in rule.crowded_rows(n, k, seed):
            ok, ids = rule.select(row, k)
            seen.add((length > 32, length > 64))
            if ok:
                assert length <= 64 and np.array_equal(ids, oracle.route(row, k)[0])
            elif length <= 64:
                l = np.sort(row)[::-1][:k + 1]
                assert (l[:-1] - l[1:]).min() < 2.0 ** -16        # a near tie, nothing else
    assert (True, False) in seen and (n < 512 or (True, True) in seen)


def test_random_rows_are_accepted_almost_always():
    rng = np.random.default_rng(7)
    lengths = [rule.list_length(r, 10) for r in rng.normal(0, 1, (12000, 512)).astype(np.float32)]
    assert 0 < sum(l > 32 for l in lengths) < 36 and max(lengths) <= 64
