"""SHA-256 message hashing with more long messages (512 bytes and more, the
two-wave form) than workgroups for them, among short ones, through the device
calls (where the library does not know the lengths) and the host calls: every
signature verifies, samples are the oracle's, forged messages are found."""
import random

import numpy as np
import pytest

import cuspx_amd as C
from oracle import oracle as O

pytestmark = pytest.mark.gpu

LENGTHS = [600, 0, 512, 1500, 511, 700, 33]


@pytest.mark.parametrize("name,n", [("sha2-128f", 1100), ("sha2-256f", 901), ("sha2-128f", 1),
                                    ("sha2-192f", 9)])
def test_long_messages_among_short_ones(name, n):
    pid = C.param_id(name)
    p = C.params(pid)
    rng = random.Random(n + pid)
    keys = min(n, 3)
    pk, sk = C.batch_keygen(pid, np.frombuffer(rng.randbytes(3 * p.n * keys), np.uint8))
    at = np.arange(n) % keys
    msgs = [rng.randbytes(LENGTHS[i % len(LENGTHS)]) for i in range(n)]
    opt = np.frombuffer(rng.randbytes(p.n * n), np.uint8).reshape(n, p.n)
    mlen = np.array([len(m) for m in msgs], np.uint32)
    step = (mlen.astype(np.uint64) + np.uint64(19)) // np.uint64(16) * np.uint64(16)
    off = np.concatenate([[0], np.cumsum(step)]).astype(np.uint64)
    flat = np.zeros(int(off[-1]), np.uint8)
    for o, m in zip(off, msgs):
        flat[int(o):int(o) + len(m)] = np.frombuffer(m, np.uint8)
    D = C.DeviceBuffer
    d_sk, d_pk, d_msg, d_opt = (D.from_array(x) for x in (sk[at], pk[at], flat, opt))
    d_off, d_len = D.from_array(off[:-1].copy()), D.from_array(mlen)
    d_sig, d_st = D(n * p.sig_bytes), D(4 * n)
    ws = D(max(C.workspace_bytes(pid, n, op) for op in (C.OP_SIGN, C.OP_VERIFY)))
    st = C.Stream()
    print("%s: %d requests" % (name, n), flush=True)
    C.sign_device(pid, n, d_sk.ptr, p.sk_bytes, d_msg.ptr, d_off.ptr, d_len.ptr, d_opt.ptr,
                  d_sig.ptr, p.sig_bytes, ws.ptr, st.handle)

    def verify():
        C.verify_device(pid, n, d_pk.ptr, p.pk_bytes, d_sig.ptr, p.sig_bytes, d_msg.ptr,
                        d_off.ptr, d_len.ptr, d_st.ptr, ws.ptr, st.handle)
        st.sync()
        return d_st.download(np.int32, n) != 0

    assert not verify().any()
    sig = d_sig.download().reshape(n, p.sig_bytes)
    assert (np.asarray(C.batch_sign(pid, sk[at], msgs, opt)) == sig).all()
    for i in {0, n // 2, n - 1}:
        assert sig[i].tobytes() == O.signature_with_optrand(pid, msgs[i], sk[at[i]].tobytes(),
                                                            opt[i].tobytes()), i
    forged = np.zeros(n, bool)
    for i in {0, n // 3, n - 1}:
        if mlen[i]:
            flat[int(off[i]) + int(mlen[i]) - 1] ^= 1
            forged[i] = True
    d_msg.upload(flat)
    assert (verify() == forged).all()
