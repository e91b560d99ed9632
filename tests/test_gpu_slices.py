"""Batches whose WOTS chains are 2^32 lanes and more, which one launch cannot
hold (SHA2-128s: 34240 signatures, 239675 keys), and the subtrees' launch cut as
well (16 lanes per leaf, split subtrees): every signature verifies and samples
are the oracle's; the keys are those of the two halves."""
import random

import numpy as np
import pytest

import cuspx_amd as C
from oracle import oracle as O

pytestmark = pytest.mark.gpu

NAME = "sha2-128s"


@pytest.mark.parametrize("n,split", [(34261, 0), (39007, 16)])
def test_signing_past_one_launch(n, split):
    pid = C.param_id(NAME)
    p = C.params(pid)
    keys = 5
    rng = random.Random(n)
    pk, sk = C.batch_keygen(pid, np.frombuffer(rng.randbytes(3 * p.n * keys), np.uint8))
    at = np.arange(n) % keys
    msg = np.frombuffer(rng.randbytes(32 * n), np.uint8)
    opt = np.frombuffer(rng.randbytes(p.n * n), np.uint8)
    D = C.DeviceBuffer
    d_sk, d_pk, d_msg, d_opt = (D.from_array(x) for x in (sk[at], pk[at], msg, opt))
    d_moff = D.from_array(np.arange(n, dtype=np.uint64) * 32)
    d_mlen = D.from_array(np.full(n, 32, np.uint32))
    d_sig, d_st = D(n * p.sig_bytes), D(4 * n)
    ws = D(C.workspace_bytes(pid, n, C.OP_SIGN))
    st = C.Stream()
    print("%s: %d signatures, %.1f GB of workspace" % (NAME, n, ws.nbytes / 1e9), flush=True)
    C.set_split(pid, C.OP_SIGN, split)
    try:
        C.sign_device(pid, n, d_sk.ptr, p.sk_bytes, d_msg.ptr, d_moff.ptr, d_mlen.ptr, d_opt.ptr,
                      d_sig.ptr, p.sig_bytes, ws.ptr, st.handle)
    finally:
        C.set_split(pid, C.OP_SIGN, 0)
    C.verify_device(pid, n, d_pk.ptr, p.pk_bytes, d_sig.ptr, p.sig_bytes, d_msg.ptr, d_moff.ptr,
                    d_mlen.ptr, d_st.ptr, ws.ptr, st.handle)
    st.sync()
    assert np.count_nonzero(d_st.download(np.int32, n)) == 0
    sig = d_sig.download().reshape(n, p.sig_bytes)
    for i in (0, n // 2, n - 1):
        assert sig[i].tobytes() == O.signature_with_optrand(
            pid, msg[32 * i:32 * i + 32].tobytes(), sk[at[i]].tobytes(),
            opt[p.n * i:p.n * (i + 1)].tobytes()), i


@pytest.mark.parametrize("n,split", [(239701, 0), (262147, 16)])
def test_keygen_past_one_launch(n, split):
    pid = C.param_id(NAME)
    p = C.params(pid)
    seeds = np.frombuffer(random.Random(n).randbytes(3 * p.n * n), np.uint8)
    D = C.DeviceBuffer
    d_seed, ws = D.from_array(seeds), D(C.workspace_bytes(pid, n, C.OP_KEYGEN))
    st = C.Stream()

    def keys(a, b):
        d_pk, d_sk = D((b - a) * p.pk_bytes), D((b - a) * p.sk_bytes)
        C.set_split(pid, C.OP_KEYGEN, split)
        try:
            C.keygen_device(pid, b - a, d_seed.ptr + 3 * p.n * a, 3 * p.n, d_pk.ptr, d_sk.ptr,
                            ws.ptr, st.handle)
        finally:
            C.set_split(pid, C.OP_KEYGEN, 0)
        st.sync()
        return d_pk.download(), d_sk.download()

    print("%s: %d keys, %.1f GB of workspace" % (NAME, n, ws.nbytes / 1e9), flush=True)
    pk, sk = keys(0, n)
    m = n // 2
    halves = keys(0, m), keys(m, n)
    assert (pk == np.concatenate([h[0] for h in halves])).all()
    assert (sk == np.concatenate([h[1] for h in halves])).all()
    opk, osk = O.seed_keypair(pid, seeds[-3 * p.n:].tobytes())
    assert pk[-p.pk_bytes:].tobytes() == opk and sk[-p.sk_bytes:].tobytes() == osk
