"""The fused layer publishes the routed ids before the softmax denominator is known: it accepts its candidates when
their exponentials e are separated by the margin below, and claims that the probabilities p = fl(e * inv) - one inv
per row, 1 / sum with 1 <= sum <= 1024, as in the reference (src/qwen38_moe.cuh:711-749) - are then strictly
ordered as well.  This checks the claim in float32 arithmetic on the tightest pairs the test lets through."""
import numpy as np

MARGIN = np.float32(1.000001)     # the constant of the device code
FLOOR = np.float32(2.0 ** -100)


def _tightest_pairs(rng, n):
    # e_b anywhere a softmax numerator can be (down to subnormals), e_a the smallest float the test accepts above it
    expo = rng.uniform(-149.0, 0.0, n)
    e_b = np.exp2(expo).astype(np.float32) * rng.uniform(1.0, 2.0, n).astype(np.float32)
    e_b = np.minimum(e_b, np.float32(1.0))
    below = (e_b * MARGIN).astype(np.float32)
    e_a = np.nextafter(np.maximum(below, np.nextafter(FLOOR, np.float32(0.0))), np.float32(np.inf))
    keep = e_a <= np.float32(1.0)
    return e_a[keep], e_b[keep]


def test_margin_on_exponentials_orders_the_probabilities():
    rng = np.random.default_rng(20261014)
    e_a, e_b = _tightest_pairs(rng, 2_000_000)
    assert np.all(e_a >= FLOOR) and np.all(e_a > (e_b * MARGIN).astype(np.float32))
    sums = np.concatenate([rng.uniform(1.0, 1024.0, e_a.size - 4), [1.0, 1024.0, 1.0 + 2.0 ** -40, 1023.999999]])
    inv = (1.0 / sums).astype(np.float32)   # static_cast<float>(1.0 / sum) of a double sum
    p_a = (e_a * inv).astype(np.float32)
    p_b = (e_b * inv).astype(np.float32)
    assert np.all(p_a > p_b)
    assert np.all(p_a >= np.float32(2.0 ** -111))   # far above the subnormal range, where products lose bits


def test_without_the_margin_the_order_can_collapse():
    # negative control: adjacent exponentials do round to the same probability for some denominators
    rng = np.random.default_rng(7)
    e_b = rng.uniform(0.5, 1.0, 200_000).astype(np.float32)
    e_a = np.nextafter(e_b, np.float32(np.inf))
    inv = (1.0 / rng.uniform(1.0, 1024.0, e_b.size)).astype(np.float32)
    assert np.any((e_a * inv).astype(np.float32) == (e_b * inv).astype(np.float32))


# ---- the one-wave selection: keys of 23 bits ------------------------------------------------------------------------
def step_a(oracle, logits, k, cell_top=True):
    """The device's first step restated for one row: (accepted, ids).  Keys are the logits' bits in float order with the
    low nine replaced by 511 - expert; cell_top: the (k+1)-th exponential is that of the top of its key's cell."""
    b = logits.view(np.uint32)
    order = np.where(b >> 31, ~b, b ^ np.uint32(0x80000000)).astype(np.uint32)
    key = (order & np.uint32(0xFFFFFE00)) | (511 - np.arange(logits.size)).astype(np.uint32)
    taken = np.argsort(key)[::-1][:k + 1]
    l = logits[taken].copy()
    if cell_top:
        top = key[taken[k]] | np.uint32(0x1FF)
        l[k] = np.array([top ^ np.uint32(0x80000000) if top >> 31 else ~top], np.uint32).view(np.float32)[0]
    e = oracle.exp_ggml((l - logits.max()).astype(np.float32))
    margin = np.full(k, 1.000001, np.float32)
    margin[k - 1] = 1.000004
    grid = key[taken] >> 9
    ok = np.all(grid[:-1] > grid[1:]) and np.all(e[:-1] >= FLOOR) and np.all(e[:-1] > (e[1:] * margin).astype(np.float32))
    return bool(ok), taken[:k]


def near_tie_row(n=64):
    """Five clear winners; then the first float of a cell (id 40), the last of the cell below (id 30: the same
    probability, and the lower id) and a float low in that cell (id 20: a higher key than id 30's).  Top-6 takes id 30."""
    l = np.linspace(-3.0, -0.5, n).astype(np.float32)
    l[[3, 9, 17, 33, 50]] = np.array([4.0, 3.5, 3.0, 2.5, 2.0], np.float32)
    l[[40, 30, 20]] = [np.float32(float.fromhex(v)) for v in ("0x1.3d74p-1", "0x1.3d73fep-1", "0x1.3d700ap-1")]
    return l


def test_a_logit_left_out_of_the_last_cell_is_not_forgotten(oracle):
    l, k = near_tie_row(), 6
    want, _ = oracle.route(l, k)
    p = oracle.softmax_row(l)
    assert p[40] == p[30] and want[-1] == 30
    accepted, ids = step_a(oracle, l, k, cell_top=False)
    assert accepted and ids[-1] == 40     # negative control: by the (k+1)-th logit itself the row passes with the wrong id
    accepted, ids = step_a(oracle, l, k)
    assert not accepted                   # the row takes the rungs over the probabilities


def test_accepted_rows_are_the_selection(oracle):
    """Rows whose k-th and later logits crowd around the end of a cell, of either sign and several magnitudes."""
    rng = np.random.default_rng(20261202)
    accepted = 0
    for trial in range(3000):
        n, k = (64, 6) if trial % 2 else (128, 10)
        l = rng.normal(-6.0, 0.5, n).astype(np.float32)
        where = rng.permutation(n)
        l[where[:k - 1]] = (4.0 + np.arange(k - 1)).astype(np.float32)
        edge = np.array([np.float32(rng.choice([-1.0, 1.0]) * 2.0 ** rng.uniform(-5, 1.5))]).view(np.uint32)[0] & np.uint32(0xFFFFFE00)
        crowd = where[k - 1:k + 3]
        reach = int(rng.choice([4, 64, 600, 3000]))   # units in the last place around the end of the cell
        l[crowd] = (edge + rng.integers(-reach, reach, crowd.size)).astype(np.uint32).view(np.float32)
        ok, ids = step_a(oracle, l, k)
        if ok:
            accepted += 1
            assert np.array_equal(ids, oracle.route(l, k)[0]), (trial, l[crowd])
    assert accepted > 300


# ---- the one-wave selection: differences of the logits --------------------------------------------------------------
def test_differences_of_the_logits_order_the_probabilities(oracle):
    """The one-wave selection accepts on d = fl(l - l_0) alone: a fall of 2^-19 from one selected logit to the next, of 2^-17 to the
    first that is not, nothing selected below -69.  The tightest such pairs, through the reference's exponential: separated by
    the margins above, and by anything that is left, up to the first that is not selected, too."""
    rng = np.random.default_rng(20261204)
    d_a = -np.concatenate([rng.uniform(0.0, 69.0, 300_000), 2.0 ** rng.uniform(-18, 6, 300_000)]).astype(np.float32)
    d_a = d_a[d_a >= np.float32(-69.0)]
    for gap, margin in ((np.float32(2.0 ** -19), MARGIN), (np.float32(2.0 ** -17), np.float32(1.000004))):
        d_b = (d_a - gap).astype(np.float32)
        d_b = np.where((d_a - d_b).astype(np.float32) >= gap, d_b, np.nextafter(d_b, np.float32(-np.inf)))
        assert np.all((d_a - d_b).astype(np.float32) >= gap)
        e_a, e_b = oracle.exp_ggml(d_a), oracle.exp_ggml(d_b)
        assert np.all(e_a >= FLOOR) and np.all(e_a > (e_b * margin).astype(np.float32))
        below = oracle.exp_ggml((d_b * (1 + rng.uniform(0, 2.0 ** -18, d_b.size))).astype(np.float32))
        assert np.all(e_a > (below * MARGIN).astype(np.float32))
