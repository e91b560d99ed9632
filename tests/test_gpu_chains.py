"""Signing on both sides of the line between the fused launch (k_sign_fused:
FORS tiles and chains together) and k_fors + k_chains: the last batch of the
one and the first of the other give the same signatures for the same requests,
and the first and last request's are the oracle's.  Batches of these sizes
also end inside a wave of chains (leaves not a multiple of 64)."""
import random

import numpy as np
import pytest

import cuspx_amd as C
from oracle import oracle as O

pytestmark = pytest.mark.gpu

# the largest batch of the fused launch (8192 chain waves)
FUSED = {"sha2-128f": 85, "sha2-128s": 4, "sha2-192f": 58, "sha2-192s": 2, "sha2-256f": 28,
         "sha2-256s": 3, "shake256-128f": 85, "shake256-128s": 4, "shake256-192f": 58,
         "shake256-192s": 2, "shake256-256f": 28, "shake256-256s": 3}


@pytest.mark.parametrize("name", sorted(FUSED))
def test_both_sides_of_the_fused_launch(name):
    pid = C.param_id(name)
    p = C.params(pid)
    n = FUSED[name] + 1
    rng = random.Random(n + pid)
    pk, sk = C.batch_keygen(pid, np.frombuffer(rng.randbytes(3 * p.n * n), np.uint8))
    msgs = [rng.randbytes(rng.choice((0, 32, 77))) for _ in range(n)]
    opt = np.frombuffer(rng.randbytes(p.n * n), np.uint8).reshape(n, p.n)
    print("%s: %d and %d requests" % (name, n - 1, n), flush=True)
    C.profile_reset()
    C.profile_enable(True)
    try:
        few = C.batch_sign(pid, sk[:n - 1], msgs[:n - 1], opt[:n - 1])
        assert "k_sign_fused" in C.profile_read() and "k_chains" not in C.profile_read()
        C.profile_reset()
        all_ = C.batch_sign(pid, sk, msgs, opt)
        assert "k_chains" in C.profile_read() and "k_sign_fused" not in C.profile_read()
    finally:
        C.profile_enable(False)
    assert (few == all_[:n - 1]).all()
    for i in (0, n - 1):
        assert bytes(all_[i]) == O.signature_with_optrand(pid, msgs[i], bytes(sk[i]),
                                                          opt[i].tobytes()), i
    assert (C.batch_verify(pid, pk, all_, msgs) == 0).all()


@pytest.mark.parametrize("name", sorted(FUSED))
def test_both_sides_of_the_narrow_fors_tiles(name):
    """The last batch whose FORS tiles are the narrowest (3584 chain waves) and
    the first of the set's own width, inside the fused launch."""
    pid = C.param_id(name)
    p = C.params(pid)
    leaves = p.d << (p.full_h // p.d)
    n = 1
    while -(-(n + 1) * leaves // 64) * p.len <= 3584:
        n += 1
    rng = random.Random(n + pid)
    pk, sk = C.batch_keygen(pid, np.frombuffer(rng.randbytes(3 * p.n * (n + 1)), np.uint8))
    msgs = [rng.randbytes(rng.choice((0, 32, 77))) for _ in range(n + 1)]
    opt = np.frombuffer(rng.randbytes(p.n * (n + 1)), np.uint8).reshape(n + 1, p.n)
    print("%s: %d and %d requests" % (name, n, n + 1), flush=True)
    few = C.batch_sign(pid, sk[:n], msgs[:n], opt[:n])
    all_ = C.batch_sign(pid, sk, msgs, opt)
    assert (few == all_[:n]).all()
    assert bytes(few[0]) == O.signature_with_optrand(pid, msgs[0], bytes(sk[0]), opt[0].tobytes())
    assert (C.batch_verify(pid, pk, all_, msgs) == 0).all()
