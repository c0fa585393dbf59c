"""What the streaming triangular kernel with two accumulator sets relies on, by the fp32 law of its coordinates and coefficients: the source
rows of output row r + 2 lie behind those of row r, but for one at most that both have, which is neither the window's first nor its
last row, the first tap of row r + 2 and not the first of row r. Rows with a coefficient of 0 count for neither."""
import numpy as np
import pytest

f = np.float32


def _first_and_last(sh, dh, y0):
    """Source rows of the first and last coefficient other than 0 of every output row, clamped to the window, and which taps they are."""
    ry = f(f(sh) / f(dh))
    raw = (np.arange(dh).astype(f) * ry + f(f(f(ry - f(1)) * f(0.5)) - ry)).astype(f) + f(y0)
    loc = np.ceil(raw)
    k = np.arange(int(np.ceil(f(2) * ry))).astype(f)
    c = f(1) - np.abs((((loc - raw).astype(f) - ry)[:, None] + k) * f(f(1) / ry))
    rows = np.clip(loc[:, None].astype(np.float64) + k, y0, y0 + sh - 1)
    return np.where(c > 0, rows, np.inf).min(1), np.where(c > 0, rows, -np.inf).max(1), np.where(c > 0, k, np.inf).min(1), np.where(c > 0, k, -np.inf).max(1)


def _shared(sh, dh, y0):
    first, last, first_tap, last_tap = _first_and_last(sh, dh, y0)
    assert (first <= last).all(), (sh, dh, y0)
    a, b = first[2:], last[:-2]
    assert (a >= b).all(), "%d rows to %d at %d: more than one source row in rows two apart" % (sh, dh, y0)
    meet = b[a == b]
    assert ((meet > y0) & (meet < y0 + sh - 1)).all(), "%d rows to %d at %d: the window's end in rows two apart" % (sh, dh, y0)
    assert (first_tap[2:][a == b] == 0).all() and (last_tap[:-2][a == b] > 0).all(), (sh, dh, y0)
    return len(meet)


def test_small_windows_whole():
    assert sum(_shared(sh, dh, y0) for sh in range(3, 90) for dh in range(3, sh) for y0 in (0, 1, 37)) > 0


@pytest.mark.parametrize("seed", range(4))
def test_windows_anywhere_below_two_to_the_twentieth(seed):
    rng = np.random.default_rng(seed)
    met = 0
    for _ in range(1500):
        sh = int(np.exp(rng.uniform(np.log(4), np.log(6000))))
        dh = int(rng.integers(max(3, sh // 8), sh)) if sh > 4 else 3
        if rng.random() < 0.4:  # ratios of small whole numbers, whose rows meet again and again
            q = int(rng.integers(2, 14))
            dh = max(q, sh // q // 2 * q)
            sh = dh // q * int(rng.integers(q + 1, 4 * q))
        y0 = int(rng.choice([0, rng.integers(0, 5000), (1 << 20) - sh]))
        met += _shared(sh, dh, y0)
    assert met > 0


def test_a_ratio_just_above_one():
    for dh in (3, 4, 100, 1000, 100000, (1 << 20) - 2):
        _shared(dh + 1, dh, 0)


@pytest.mark.parametrize("sh,dh", [(550, 350), (704, 448), (484, 308), (352, 224), (476, 140), (640, 384)])
def test_ordinary_sizes_whose_rows_meet_often(sh, dh):
    assert _shared(sh, dh, 0) > 2
