"""FORS trees of 2^14 leaves (192s, 256s) split over four workgroups in small
batches: the last split batch, the first whole one and the smallest batches
sign the same requests alike, and as the oracle does."""
import random

import numpy as np
import pytest

import cuspx_amd as C
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ["sha2-192s", "sha2-256s", "shake256-192s", "shake256-256s"])
def test_split_and_whole_trees(name):
    pid = C.param_id(name)
    p = C.params(pid)
    last = 4096 // (4 * 4 * p.k)  # the largest split batch: 4 workgroups of 4 waves per tree
    n = last + 1
    rng = random.Random(pid)
    pk, sk = C.batch_keygen(pid, np.frombuffer(rng.randbytes(3 * p.n * n), np.uint8))
    msgs = [rng.randbytes(rng.choice((0, 32, 77))) for _ in range(n)]
    opt = np.frombuffer(rng.randbytes(p.n * n), np.uint8).reshape(n, p.n)
    whole = C.batch_sign(pid, sk, msgs, opt)
    assert (C.batch_verify(pid, pk, whole, msgs) == 0).all()
    for i in (0, last):
        assert bytes(whole[i]) == O.signature_with_optrand(pid, msgs[i], bytes(sk[i]),
                                                           opt[i].tobytes()), i
    for m in (1, 2, 3, 5, last):
        print("%s: %d requests" % (name, m), flush=True)
        assert (C.batch_sign(pid, sk[-m:], msgs[-m:], opt[-m:]) == whole[-m:]).all(), m
