"""Verification's hypertree kernel in each of its forms: chain steps on a lane,
on a lane pair (groups of 64 lanes or more) and in
two-phase rounds (SHA-256, more workgroups than CUs), with a last workgroup
that is not full.  Every request's verdict is known: signatures are the
oracle's (the first of each set is compared with it), some with one bit
flipped in a FORS part, a chain value, an authentication path or the last
layer."""
import random

import numpy as np
import pytest

import cuspx_amd as C
from oracle import oracle as O

pytestmark = pytest.mark.gpu

ROUTES = [(64, 65), (64, 1025), (32, 2049), (16, 17), (16, 4113)]


@pytest.mark.parametrize("name", ["sha2-128f", "sha2-192f", "sha2-256f", "shake256-128f",
                                  "shake256-192s", "shake256-256f"])
def test_every_chain_form_gives_the_known_verdicts(name):
    pid = C.param_id(name)
    p = C.params(pid)
    rng = random.Random(pid)
    base = 5
    pk, sk = C.batch_keygen(pid, np.frombuffer(rng.randbytes(3 * p.n * base), np.uint8))
    msgs = [rng.randbytes(rng.choice((0, 32, 77))) for _ in range(base)]
    opt = np.frombuffer(rng.randbytes(p.n * base), np.uint8).reshape(base, p.n)
    sig = np.asarray(C.batch_sign(pid, sk, msgs, opt))
    assert bytes(sig[0]) == O.signature_with_optrand(pid, msgs[0], bytes(sk[0]), opt[0].tobytes())
    layer = p.len * p.n + p.full_h // p.d * p.n
    first = p.n + p.k * (p.a + 1) * p.n          # layer 0's signature
    spots = [p.n + 3, first + 1, first + p.len * p.n, first + layer + p.n * p.len - 1,
             p.sig_bytes - 1, p.sig_bytes - layer]
    for G, n in ROUTES + ([(128, 3), (128, 513)] if p.len > 64 else []):
        at = np.arange(n) % base
        sigs = sig[at].copy()
        want = np.zeros(n, bool)
        for i in {0, n - 1, n - 2} | {rng.randrange(n) for _ in range(9)}:
            if i != 0 or n % 2:
                sigs[i, spots[i % len(spots)]] ^= 1 << rng.randrange(8)
                want[i] = True
        print("%s: G %d, %d requests" % (name, G, n), flush=True)
        C.set_split(pid, 1, G)
        try:
            got = C.batch_verify(pid, pk[at], sigs, [msgs[i] for i in at])
        finally:
            C.set_split(pid, 1, 0)
        assert ((np.asarray(got) != 0) == want).all(), (G, n)
