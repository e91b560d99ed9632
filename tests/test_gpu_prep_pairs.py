"""SHAKE256 message hashing on both sides of the line (7168 requests) between a
row of 32 lanes and a lane pair per request: the same requests sign alike on
both, and as the oracle does; messages end at every place of a block."""
import random

import numpy as np
import pytest

import cuspx_amd as C
from oracle import oracle as O

pytestmark = pytest.mark.gpu

ROWS = 7168


@pytest.mark.parametrize("name", ["shake256-128f", "shake256-192f", "shake256-256f"])
def test_both_sides_of_the_rows(name):
    pid = C.param_id(name)
    p = C.params(pid)
    n, keys = ROWS + 1, 7
    rng = random.Random(pid)
    pk, sk = C.batch_keygen(pid, np.frombuffer(rng.randbytes(3 * p.n * keys), np.uint8))
    at = np.arange(n) % keys
    msgs = [rng.randbytes(i % 409 if i % 50 else 409 + i % 1000) for i in range(n)]
    opt = np.frombuffer(rng.randbytes(p.n * n), np.uint8).reshape(n, p.n)
    print("%s: %d and %d requests" % (name, n, ROWS), flush=True)
    pairs = C.batch_sign(pid, sk[at], msgs, opt)
    rows = C.batch_sign(pid, sk[at][1:], msgs[1:], opt[1:])
    assert (pairs[1:] == rows).all()
    assert (C.batch_verify(pid, pk[at], pairs, msgs) == 0).all()
    assert (C.batch_verify(pid, pk[at][1:], rows, msgs[1:]) == 0).all()
    for i in (0, 5, n - 1):
        assert bytes(pairs[i]) == O.signature_with_optrand(pid, msgs[i], bytes(sk[at[i]]),
                                                           opt[i].tobytes()), i
    msgs[n - 1] += b"\0"
    assert ((C.batch_verify(pid, pk[at], pairs, msgs) != 0) == (np.arange(n) == n - 1)).all()
