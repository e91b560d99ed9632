"""The choice of splits over a range of batch sizes (cuspx_amd/autotune.py) and
the committed table: lanes per leaf never widen as batches grow, lanes per
request change where a stair of the verify kernel's time ends."""
import os

from cuspx_amd import autotune as T

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LEAF = (16, 4, 1)
VERIFY = (1, 128, 64, 32, 16)


def test_settle_takes_the_least_sum_without_going_back():
    t = [{16: 1.0, 4: 2.0, 1: 3.0}, {16: 1.2, 4: 1.0, 1: 1.2}, {16: 2.0, 4: 1.1, 1: 1.0},
         {16: 3.0, 4: 0.98, 1: 1.0}, {16: 3.0, 4: 1.5, 1: 1.0}]
    # the fourth batch's 2% at 4 lanes does not pay for the third's 10%
    assert T.settle(t, LEAF) == [16, 4, 1, 1, 1]
    # and does if the third's difference is smaller
    t[2] = {16: 2.0, 4: 1.006, 1: 1.0}
    assert T.settle(t, LEAF) == [16, 4, 4, 4, 1]


def test_settle_goes_back_where_that_is_allowed_and_pays():
    t = [{64: 1.0, 16: 1.2}, {64: 1.2, 16: 1.0}, {64: 1.0, 16: 1.004}, {64: 1.0, 16: 1.3},
         {64: 1.1, 16: 1.0}]
    assert T.settle(t, (64, 16), back=True) == [64, 16, 16, 64, 16]
    assert T.settle(t, (64, 16)) == [64, 64, 64, 64, 16]


def test_settle_takes_the_later_split_within_half_a_percent():
    assert T.settle([{16: 1.0, 4: 1.004, 1: 1.0049}], LEAF) == [1]
    assert T.settle([{16: 1.0, 4: 1.004, 1: 1.006}], LEAF) == [4]


def test_settle_with_a_split_that_ends():
    """Speculative verification exists up to 256 requests only."""
    t = [{1: 1.0, 128: 2.0, 64: 2.0, 32: 2.0, 16: 2.0}, {128: 1.0, 64: 1.2, 32: 2.0, 16: 3.0},
         {128: 2.0, 64: 1.0, 32: 1.002, 16: 1.1}, {128: 4.0, 64: 1.5, 32: 1.1, 16: 1.0}]
    assert T.settle(t, VERIFY, back=True) == [1, 128, 32, 16]


def test_verification_is_timed_where_its_stairs_end():
    """A launch of G lanes per request fills the CUs at multiples of 65536 / G
    requests (the finest: 512)."""
    b = T.BATCHES_VERIFY
    assert list(b) == sorted(set(b)) and 256 in b
    for G in (16, 32, 64, 128):
        assert all(n in b for n in range(65536 // G, 16385, 65536 // G)), G


def _table():
    rows = {}
    with open(os.path.join(ROOT, "cuspx_amd", "tuning.txt")) as f:
        for line in f:
            if not line.startswith("#"):
                name, op, units, lanes = line.split()
                rows.setdefault((name, op), []).append((int(units), int(lanes)))
    return rows


def test_table_lines():
    rows = _table()
    assert len(rows) == 36
    for (name, op), r in rows.items():
        assert r[0][0] == 0 and r == sorted(r), (name, op)
        assert all(x[1] != y[1] for x, y in zip(r, r[1:])), (name, op)
        if op == "verify":  # a line begins behind a size that was timed
            assert all(units - 1 in T.BATCHES_VERIFY for units, _ in r[1:]), (name, r)
            assert all(lanes in VERIFY for _, lanes in r), (name, r)
        else:               # lanes per leaf never widen as batches grow
            at = [LEAF.index(lanes) for _, lanes in r]
            assert at == sorted(set(at)), (name, op, r)
