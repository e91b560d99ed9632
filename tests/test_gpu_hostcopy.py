"""Host-buffer calls on both sides of the 2 MiB line between the copying kernel
and the copy engine (122 and 123 SHA2-128f signatures): the same requests give
the same keys, signatures and verdicts, and the oracle's."""
import random

import numpy as np
import pytest

import cuspx_amd as C
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,n", [("sha2-128f", 122), ("shake256-256f", 42), ("sha2-128f", 1)])
def test_both_sides_of_the_kernel_copy(name, n):
    pid = C.param_id(name)
    p = C.params(pid)
    assert n == 1 or n * p.sig_bytes <= 2 << 20 < (n + 1) * p.sig_bytes
    rng = random.Random(n + pid)
    seeds = np.frombuffer(rng.randbytes(3 * p.n * (n + 1)), np.uint8)
    pk, sk = C.batch_keygen(pid, seeds)
    pk1, sk1 = C.batch_keygen(pid, seeds[:3 * p.n * n])
    assert (pk1 == pk[:n]).all() and (sk1 == sk[:n]).all()
    msgs = [rng.randbytes(rng.choice((0, 1, 33, 300))) for _ in range(n + 1)]
    opt = np.frombuffer(rng.randbytes(p.n * (n + 1)), np.uint8).reshape(n + 1, p.n)
    few = C.batch_sign(pid, sk[:n], msgs[:n], opt[:n])
    all_ = np.array(C.batch_sign(pid, sk, msgs, opt))
    assert (few == all_[:n]).all()
    for i in (0, n):
        assert bytes(all_[i]) == O.signature_with_optrand(pid, msgs[i], bytes(sk[i]),
                                                          opt[i].tobytes()), i
    all_[n, -1] ^= 1
    want = np.arange(n + 1) == n
    assert ((C.batch_verify(pid, pk, all_, msgs) != 0) == want).all()
    assert (C.batch_verify(pid, pk[:n], all_[:n], msgs[:n]) == 0).all()
