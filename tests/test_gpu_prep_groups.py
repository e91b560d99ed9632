"""SHA-256 message hashing on groups of 8 lanes: the groups of one wave with
different message lengths around a block's ends and the long path's start, and
a last wave that is not full, against the oracle."""
import random

import numpy as np
import pytest

import cuspx_amd as C
from oracle import oracle as O

pytestmark = pytest.mark.gpu

LENGTHS = [0, 1, 3, 4, 31, 32, 39, 40, 47, 48, 55, 56, 63, 64, 65, 103, 104, 119, 120, 127, 128,
           511, 512, 513, 1000]


@pytest.mark.parametrize("name", ["sha2-128f", "sha2-192f", "sha2-256f"])
def test_message_lengths_in_one_wave(name):
    pid = C.param_id(name)
    p = C.params(pid)
    rng = random.Random(pid)
    n = len(LENGTHS)
    pk, sk = C.batch_keygen(pid, np.frombuffer(rng.randbytes(3 * p.n * n), np.uint8))
    msgs = [rng.randbytes(m) for m in LENGTHS]
    opt = np.frombuffer(rng.randbytes(p.n * n), np.uint8).reshape(n, p.n)
    sig = np.array(C.batch_sign(pid, sk, msgs, opt))
    for i in range(n):
        if name == "sha2-128f" or i % 6 == 0:
            assert bytes(sig[i]) == O.signature_with_optrand(pid, msgs[i], bytes(sk[i]),
                                                             opt[i].tobytes()), LENGTHS[i]
    assert (C.batch_verify(pid, pk, sig, msgs) == 0).all()
    msgs[-1] = msgs[-1][:-1] + bytes([msgs[-1][-1] ^ 1])
    assert ((C.batch_verify(pid, pk, sig, msgs) != 0) == (np.arange(n) == n - 1)).all()
