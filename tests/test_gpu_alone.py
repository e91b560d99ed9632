"""SHA-256 launches on both sides of one wave per SIMD (1024 waves), where the
hash rounds change their form: key generation, signing and verification of the
same requests agree, and the oracle's."""
import random

import numpy as np
import pytest

import cuspx_amd as C
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ["sha2-128f", "sha2-192f", "sha2-256f", "sha2-128s"])
def test_both_sides_of_a_wave_per_simd(name):
    pid = C.param_id(name)
    p = C.params(pid)
    th = p.full_h // p.d
    rng = random.Random(pid)

    def waves(trees):
        return -(-(trees << th) // 64) * p.len

    keys = next(n for n in range(1, 4096) if waves(n) > 1024)     # first past the line
    signs = next(n for n in range(1, 64) if waves(n * p.d) > 1024)
    seeds = np.frombuffer(rng.randbytes(3 * p.n * keys), np.uint8)
    pk, sk = C.batch_keygen(pid, seeds)
    pk1, sk1 = C.batch_keygen(pid, seeds[:3 * p.n * (keys - 1)])
    assert (pk1 == pk[:-1]).all() and (sk1 == sk[:-1]).all()
    at = np.arange(signs) % keys
    msgs = [rng.randbytes(33) for _ in range(signs)]
    opt = np.frombuffer(rng.randbytes(p.n * signs), np.uint8).reshape(signs, p.n)
    sig = C.batch_sign(pid, sk[at], msgs, opt)
    one = C.batch_sign(pid, sk[at][:1], msgs[:1], opt[:1])
    assert (one[0] == sig[0]).all()
    assert bytes(one[0]) == O.signature_with_optrand(pid, msgs[0], bytes(sk[0]), opt[0].tobytes())
    for n in (1, 512 * 64 // p.k, 512 * 64 // p.k + 1):           # k_vfors' line, k_vspec at 1
        r = np.arange(n) % signs
        s = np.array(sig)[r]
        s[n - 1, p.n + 5] ^= 1                                    # in the first FORS tree
        got = C.batch_verify(pid, pk[at][r], s, [msgs[i] for i in r])
        assert ((np.asarray(got) != 0) == (np.arange(n) == n - 1)).all(), n
