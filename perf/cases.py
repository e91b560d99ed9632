"""Timed cases of the engine: signing, verification and key generation as a
program that uses the library calls them.

``listed()`` names the cases, ``draw(rng)`` gives further ones of the same
ranges, ``prepare`` builds what such a program has in hand (keys, messages,
signatures, buffers, a workspace, a graph or a server), ``run`` is one pass
through the public entry points and ``work`` what that pass cannot do without.
All outputs are bytes and status words, so any two builds have to agree on
them exactly.

Sets, batch sizes and message lengths are those of the benchmark
configurations (``cuspx_amd/workloads.py``), of the tests and of the tuning
grid, with odd sizes between them.
"""
import math

import numpy as np
import torch

import cuspx_amd as C

SETS = tuple(C.PARAM_NAMES)
FAST = tuple(s for s in SETS if s.endswith("f"))

# 32-bit operations of one SHA-256 compression (64 rounds of 14, 48 schedule
# words of 10) and of one Keccak-f[1600] permutation (24 rounds of 174)
OPS_SHA256 = 64 * 14 + 48 * 10
OPS_KECCAK = 24 * 174


def listed():
    return [
        # the smallest call: one message signed through the host-buffer entry
        # point, as a program does that signs now and then
        {"name": "host-sign-1-sha2-128f", "op": "sign", "via": "host", "set": "sha2-128f",
         "num": 1, "lo": 33, "hi": 33},
        # one signed message opened through the api.h call (the drop-in use),
        # at the largest of the fast sets
        {"name": "open-1-shake256-256f", "op": "open", "via": "api", "set": "shake256-256f",
         "num": 1, "lo": 33, "hi": 33},
        # a handful of requests with messages of 16 B to 64 KiB: what a signing
        # service has queued at one moment
        {"name": "sign-7-shake256-256f", "op": "sign", "via": "device", "set": "shake256-256f",
         "num": 7, "lo": 16, "hi": 65536},
        # a small batch of short messages at the default set
        {"name": "sign-61-sha2-128f", "op": "sign", "via": "device", "set": "sha2-128f",
         "num": 61, "lo": 32, "hi": 32},
        # small signatures, slow signing: the middle one of the s-set batches
        {"name": "sign-64-sha2-128s", "op": "sign", "via": "device", "set": "sha2-128s",
         "num": 64, "lo": 32, "hi": 32},
        # verification of a middle-sized batch of messages of mixed length,
        # some of them forged
        {"name": "verify-300-sha2-192f", "op": "verify", "via": "device", "set": "sha2-192f",
         "num": 300, "lo": 1, "hi": 4096},
        # signing a middle-sized batch at the highest security level
        {"name": "sign-500-sha2-256f", "op": "sign", "via": "device", "set": "sha2-256f",
         "num": 500, "lo": 1, "hi": 4096},
        # provisioning: many key pairs at once
        {"name": "keygen-1000-shake256-128f", "op": "keygen", "via": "device",
         "set": "shake256-128f", "num": 1000, "lo": 0, "hi": 0},
        # bulk signing and bulk verification of 32-byte digests (the headline
        # configuration)
        {"name": "sign-4096-sha2-128f", "op": "sign", "via": "device", "set": "sha2-128f",
         "num": 4096, "lo": 32, "hi": 32},
        {"name": "verify-4096-sha2-128f", "op": "verify", "via": "device", "set": "sha2-128f",
         "num": 4096, "lo": 32, "hi": 32},
        # the largest: one graph launch that signs a batch of two sets
        {"name": "mixed-8192-shake256", "op": "mixed", "via": "graph", "set": "shake256-128f",
         "set2": "shake256-192f", "num": 8192, "lo": 1, "hi": 4096},
        # a burst of requests to the server, 80% sign and 20% verify, over the
        # three serving sets
        {"name": "serve-256", "op": "serve", "via": "server", "set": "", "num": 256, "lo": 16,
         "hi": 65536},
    ]


def draw(rng):
    most = _cost(next(c for c in listed() if c["op"] == "mixed"))
    while True:
        kind = rng.choice(("sign", "sign", "sign", "verify", "verify", "keygen", "open", "mixed",
                           "serve"))
        if kind == "serve":
            c = {"op": "serve", "via": "server", "set": "", "num": _log(rng, 32, 512)}
        elif kind == "mixed":
            a = rng.choice(FAST)
            b = rng.choice([s for s in FAST if s[:4] == a[:4] and s != a])
            c = {"op": "mixed", "via": "graph", "set": a, "set2": b, "num": _log(rng, 32, 8192)}
        elif kind == "open":
            c = {"op": "open", "via": "api", "set": rng.choice(SETS), "num": 1}
        else:
            c = {"op": kind, "via": rng.choice(("device", "device", "host")),
                 "set": rng.choice(SETS), "num": _log(rng, 2 if kind == "verify" else 1, 4096)}
        c["lo"], c["hi"] = rng.choice(((32, 32), (1, 4096), (16, 65536)))
        if c["op"] == "open":
            c["lo"] = c["hi"] = _log(rng, 1, 65536)
        if c["op"] == "keygen":
            c["lo"] = c["hi"] = 0
        if c["num"] > 1024:
            c["hi"] = min(c["hi"], 4096)
        if _cost(c) <= most:
            return c


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


# ----------------------------------------------------------------- work

SERVE_SETS = ("sha2-128f", "sha2-128s", "shake256-256f")
SERVE_KEYS = 16  # per set

_SHAPE = {  # n, full height, layers, FORS height, FORS trees
    "128s": (16, 63, 7, 12, 14), "128f": (16, 66, 22, 6, 33),
    "192s": (24, 63, 7, 14, 17), "192f": (24, 66, 22, 8, 33),
    "256s": (32, 64, 8, 14, 22), "256f": (32, 68, 17, 9, 35),
}


def _hashes(name, op):
    """Compressions / permutations of one request without its message hashes.
    The chains of the layers' signatures are part of the leaves' chains."""
    n, h, d, a, k = _SHAPE[name[-4:]]
    sha2, th, ln = name.startswith("sha2"), h // d, 2 * n + 3
    blocks = (lambda b: (22 + b + 9 + 63) // 64) if sha2 else (lambda b: (n + 32 + b) // 136 + 1)
    leaf = ln * 16 + blocks(ln * n)
    tree = (1 << th) * leaf + ((1 << th) - 1) * blocks(2 * n)
    if op == "keygen":
        return tree
    if op == "sign":
        return d * tree + k * ((2 << a) + ((1 << a) - 1) * blocks(2 * n)) + blocks(k * n)
    climb = d * (ln * 7.5 + blocks(ln * n) + th * blocks(2 * n))
    return climb + k * (1 + a * blocks(2 * n)) + blocks(k * n)


def _ops(name, op):
    return _hashes(name, op) * (OPS_SHA256 if name.startswith("sha2") else OPS_KECCAK)


def _mean_len(c):
    lo, hi = c["lo"], c["hi"]
    return lo if hi <= lo else (hi - lo) / math.log(hi / lo)


def _parts(c):
    """(set, op, count) of the requests of one pass."""
    if c["op"] == "mixed":
        return [(c["set"], "sign", c["num"] // 2), (c["set2"], "sign", c["num"] - c["num"] // 2)]
    if c["op"] == "serve":
        return [(s, o, c["num"] * f / len(SERVE_SETS)) for s in SERVE_SETS
                for o, f in (("sign", 0.8), ("verify", 0.2))]
    return [(c["set"], "verify" if c["op"] == "open" else c["op"], c["num"])]


def _cost(c):
    return sum(_ops(s, o) * m for s, o, m in _parts(c))


def work(c):
    total, ops = 0.0, 0.0
    for s, o, m in _parts(c):
        n, h, d, a, k = _SHAPE[s[-4:]]
        sig = n * (1 + k * (a + 1) + d * (2 * n + 3) + h)
        msg, rate = _mean_len(c), 64 if s.startswith("sha2") else 136
        per = {"sign": 4 * n + n + sig, "verify": 2 * n + sig + 4, "keygen": 3 * n + 6 * n}[o]
        total += m * (per + msg)
        passes = {"sign": 2, "verify": 1, "keygen": 0}[o]
        ops += m * (_ops(s, o) +
                    passes * msg / rate * (OPS_SHA256 if rate == 64 else OPS_KECCAK))
    return {"bytes": total, "flops": ops}


# -------------------------------------------------------------- prepare

def _lengths(rng, c, num):
    if c["hi"] <= c["lo"]:
        return np.full(num, c["lo"], np.int64)
    x = np.exp(rng.uniform(math.log(c["lo"]), math.log(c["hi"]), num))
    return np.clip(np.rint(x), c["lo"], c["hi"]).astype(np.int64)


def _cuda(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _bytes(rng, *shape):
    return rng.integers(0, 256, shape, np.uint8)


class _Batch:
    """Keys and messages of one batch of one set, in host and device memory."""

    def __init__(self, rng, c, name, num):
        self.name, self.num, self.pid = name, num, C.param_id(name)
        self.p = p = C.params(self.pid)
        self.seeds = _bytes(rng, num, 3 * p.n)
        self.opt = _bytes(rng, num, p.n)
        self.len = _lengths(rng, c, num)
        step = (self.len + 15) // 16 * 16
        self.off = np.concatenate([[0], np.cumsum(step[:-1])])
        self.flat = _bytes(rng, int(step.sum()) + 16)
        self.d_seeds = _cuda(self.seeds)
        self.d_pk = torch.zeros(num, p.pk_bytes, dtype=torch.uint8, device="cuda")
        self.d_sk = torch.zeros(num, p.sk_bytes, dtype=torch.uint8, device="cuda")
        self.d_opt, self.d_msg = _cuda(self.opt), _cuda(self.flat)
        self.d_off, self.d_len = _cuda(self.off.astype(np.uint64).view(np.int64)), _cuda(
            self.len.astype(np.int32))

    def ws(self, op):
        return torch.zeros(C.workspace_bytes(self.pid, self.num, op), dtype=torch.uint8,
                           device="cuda")

    def msgs(self):
        return [self.flat[o:o + n].tobytes() for o, n in zip(self.off, self.len)]

    def keygen(self, ws, stream=None):
        C.keygen_device(self.pid, self.num, self.d_seeds.data_ptr(), 3 * self.p.n,
                        self.d_pk.data_ptr(), self.d_sk.data_ptr(), ws.data_ptr(), stream)

    def sign(self, sig, ws, stream=None):
        C.sign_device(self.pid, self.num, self.d_sk.data_ptr(), self.p.sk_bytes,
                      self.d_msg.data_ptr(), self.d_off.data_ptr(), self.d_len.data_ptr(),
                      self.d_opt.data_ptr(), sig.data_ptr(), self.p.sig_bytes, ws.data_ptr(),
                      stream)

    def verify(self, sig, status, ws, stream=None):
        C.verify_device(self.pid, self.num, self.d_pk.data_ptr(), self.p.pk_bytes, sig.data_ptr(),
                        self.p.sig_bytes, self.d_msg.data_ptr(), self.d_off.data_ptr(),
                        self.d_len.data_ptr(), status.data_ptr(), ws.data_ptr(), stream)

    def new_sig(self):
        return torch.zeros(self.num, self.p.sig_bytes, dtype=torch.uint8, device="cuda")

    def keys(self):
        ws = self.ws(C.OP_KEYGEN)
        self.keygen(ws)
        torch.cuda.synchronize()

    def signed(self):
        sig, ws = self.new_sig(), self.ws(C.OP_SIGN)
        self.sign(sig, ws)
        torch.cuda.synchronize()
        return sig

    def forge(self, rng, sig):
        """One byte changed in about a fifth of the signatures, anywhere in them."""
        rows = np.flatnonzero(rng.random(self.num) < 0.2)
        cols = rng.integers(0, self.p.sig_bytes, rows.size)
        if rows.size:
            sig[_cuda(rows), _cuda(cols)] ^= 0x40


class _Server:
    """A server with its resident keys, closed with the state that holds it."""

    def __init__(self):
        self.srv = C.Server(hbm_budget_bytes=8 << 30, slots=4, batch_window_us=1000)

    def __del__(self):
        try:
            self.srv.close()
        except Exception:
            pass


_streams = []


def _stream():
    """The stream that the program launches everything on."""
    if not _streams:
        _streams.append(C.Stream())
    return _streams[0]


def prepare(case, seed):
    rng = np.random.default_rng([seed, case["num"]])
    op, via, num = case["op"], case["via"], case["num"]
    st = {"case": case}
    if op == "serve":
        return _prepare_serve(st, rng, case)
    if op == "mixed":
        st["parts"] = [_Batch(rng, case, name, m) for name, m in
                       ((case["set"], num // 2), (case["set2"], num - num // 2))]
        for b in st["parts"]:
            b.keys()
        st["ws"] = [b.ws(C.OP_SIGN) for b in st["parts"]]
        st["sigs"] = [b.new_sig() for b in st["parts"]]
        st["stream"] = _stream()
        st["graph"] = C.graph_sign_mixed(
            [C.SignGroup(b.pid, b.num, b.d_sk.data_ptr(), b.p.sk_bytes, b.d_msg.data_ptr(),
                         b.d_off.data_ptr(), b.d_len.data_ptr(), b.d_opt.data_ptr(),
                         sig.data_ptr(), b.p.sig_bytes, ws.data_ptr())
             for b, ws, sig in zip(st["parts"], st["ws"], st["sigs"])])
        return st
    b = st["b"] = _Batch(rng, case, case["set"], num)
    st["stream"] = _stream()
    if op != "keygen":
        b.keys()
    if op in ("verify", "open"):
        sig = b.signed()
        if op == "verify":
            b.forge(rng, sig)
    if via == "device":
        st["ws"] = b.ws({"sign": C.OP_SIGN, "verify": C.OP_VERIFY, "keygen": C.OP_KEYGEN}[op])
        if op == "sign":
            st["sig"] = b.new_sig()
        elif op == "verify":
            st["sig"] = sig
            st["status"] = torch.full((num,), -7, dtype=torch.int32, device="cuda")
    else:
        st["sk"], st["pk"] = b.d_sk.cpu().numpy(), b.d_pk.cpu().numpy()
        st["msgs"] = b.msgs()
        if op in ("verify", "open"):
            st["sigs"] = sig.cpu().numpy()
        if op == "open":
            C.set_default_param(b.pid)
            st["sm"] = st["sigs"][0].tobytes() + st["msgs"][0]
            st["pk1"] = st["pk"][0].tobytes()
    return st


def _prepare_serve(st, rng, case):
    num = case["num"]
    st["server"] = _Server()
    srv = st["server"].srv
    st["reqs"] = []
    signs, checks = int(round(num * 0.8)), num - int(round(num * 0.8))
    which = np.arange(num) % len(SERVE_SETS)
    for s, name in enumerate(SERVE_SETS):
        ns, nv = int((which[:signs] == s).sum()), int((which[signs:] == s).sum())
        keys = _Batch(rng, dict(case, lo=1, hi=1), name, SERVE_KEYS)
        keys.keys()
        sk, pk = keys.d_sk.cpu().numpy(), keys.d_pk.cpu().numpy()
        kid = [srv.add_key(keys.pid, sk[i].tobytes(), pk[i].tobytes()) for i in range(SERVE_KEYS)]
        for count, check in ((ns, False), (nv, True)):
            if not count:
                continue
            b = _Batch(rng, case, name, count)
            key = rng.integers(0, SERVE_KEYS, count)
            if check:
                b.d_sk, b.d_pk = _cuda(sk[key]), _cuda(pk[key])
                sig = b.signed()
                b.forge(rng, sig)
                sig = sig.cpu().numpy()
            for i, m in enumerate(b.msgs()):
                st["reqs"].append((check, kid[key[i]], m,
                                   sig[i].tobytes() if check else b.opt[i].tobytes()))
    assert signs + checks == len(st["reqs"])
    st["reqs"] = [st["reqs"][i] for i in rng.permutation(num)]
    return st


# ------------------------------------------------------------------ run

def run(st):
    case = st["case"]
    op, via = case["op"], case["via"]
    if op == "serve":
        srv = st["server"].srv
        tickets = [srv.submit_verify(k, m, x) if check else srv.submit_sign(k, m, x)
                   for check, k, m, x in st["reqs"]]
        status, sigs = [], []
        for t, (check, k, _, _) in zip(tickets, st["reqs"]):
            rc, sig = srv.wait(t, key=k)
            status.append(rc)
            if not check:
                sigs.append(sig)
        return {"status": np.array(status, np.int32), "sigs": np.frombuffer(b"".join(sigs), np.uint8)}
    if op == "mixed":
        st["graph"].launch(st["stream"])
        return st["sigs"]
    b = st["b"]
    if via == "api":
        rc, m = C.crypto_sign_open(st["sm"], st["pk1"])
        return {"rc": rc, "m": np.frombuffer(m, np.uint8)}
    if via == "host":
        if op == "sign":
            return C.batch_sign(b.pid, st["sk"], st["msgs"], b.opt)
        if op == "verify":
            return C.batch_verify(b.pid, st["pk"], st["sigs"], st["msgs"])
        return list(C.batch_keygen(b.pid, b.seeds))
    h = st["stream"].handle
    if op == "sign":
        b.sign(st["sig"], st["ws"], h)
        return st["sig"]
    if op == "verify":
        b.verify(st["sig"], st["status"], st["ws"], h)
        return st["status"]
    b.keygen(st["ws"], h)
    return [b.d_pk, b.d_sk]
