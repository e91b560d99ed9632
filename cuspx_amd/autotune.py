"""Autotuner for the work splits of the hypertree and verify kernels.

k_ht computes T_len of a WOTS leaf on one lane (S = 1), a lane pair (2, 4) or
16 lanes (8, 16): a small batch waits for T_len, which more lanes shorten; a
large one runs fastest at S = 1. k_vht runs 256 / G requests per workgroup
(G = 16 to 128 lanes per request on average): wider groups put a lane pair on
each chain and shorten each layer's chain phase down to the longest chain,
narrower ones keep more requests busy per lane; G = 1 is speculative
verification (every chain from every start first, batches up to 256). The
crossovers depend on the set and on the batch, so they are measured: for every
set, operation and batch size this times device-resident launches at each
split the set allows, chooses for all batch sizes together (settle) and writes
the choices as

    <set> <sign|keygen|verify> <min_units> <lanes>

lines (a sign launch covers batch*d subtrees, keygen and verify launches
cover batch), the table libcuspx reads from tuning.txt beside itself or from
$CUSPX_TUNING.

    python -m cuspx_amd.autotune [--sets sha2-128f,...] [--out cuspx_amd/tuning.txt]
"""
import argparse
import os
import sys
import time

import numpy as np

import cuspx_amd as C

OPS = {"sign": 0, "keygen": 2, "verify": 1}
# powers of two: a winner holds from its batch up to the next grid point, so a
# 4x grid left e.g. 2048 requests on the split timed best at 1024
BATCHES_FAST = tuple(1 << i for i in range(13))   # 1 .. 4096
BATCHES_SMALL = tuple(1 << i for i in range(11))  # 1 .. 1024
# a table's last line holds for every larger batch, so verification and key
# generation are timed to where every split fills the chip: with 4096 as the
# last size SHAKE256-128f verification stayed at 32 lanes, which at 16384
# requests take 14.5 ms against 9.3 at 16
BATCHES_KEYGEN = tuple(1 << i for i in range(15))  # 1 .. 16384
# k_vht's time is a staircase: 256 workgroups of 256 / G requests fill the CUs
# once, so a stair of any G ends at a multiple of 512 requests, and the best G
# changes from stair to stair (SHAKE256-256s, 16 / 64 lanes: 4096 requests 2.93 /
# 3.58 ms, 5000 5.77 / 4.49).  A size stands for the requests down to the size
# before it, and is timed half-way as well: a launch that ends with full CUs can
# be ahead of every smaller one of its stair (SHA2-128f at 32 lanes, 6000 requests
# 2.27 ms, 6144 1.85).  Speculative verification grows with every request.
BATCHES_VERIFY = ((1, 2, 4, 8, 16, 32, 64, 96) + tuple(range(104, 257, 8)) + (384,) +
                  tuple(512 * i for i in range(1, 33)) + (18432, 20480, 24576, 32768))


def _time(fn, stream, reps):
    fn()
    stream.sync()
    e0, e1 = C.Event(), C.Event()
    best = float("inf")
    for _ in range(reps):
        e0.record(stream)
        fn()
        e1.record(stream)
        stream.sync()
        best = min(best, e0.elapsed_ms(e1))
    return best


CHANGE = 0.005


def settle(times, order, back=False):
    """The split of each batch size, from times[i] = {split: time} for batches in
    ascending order: the least sum of the times over each batch's best, counting
    half a percent (repeats of one launch differ by that much) for each change
    and differences below it as none.  Unless `back`, a larger batch never takes
    a split that comes earlier in `order` (the widest first).  Of equal sums
    later splits are taken.  (Winners taken batch by batch alternate where two
    splits are equal, and a line made of noise then holds up to the next one.)"""
    best = None  # split of the last batch -> (cost, choices so far)
    for t in times:
        low = min(t.values())
        row = {}
        for i, S in enumerate(order):
            if S not in t:
                continue
            cost, path = 0.0, ()
            if best is not None:
                come = [(c + CHANGE * (Q != S), -order.index(Q), p) for Q, (c, p) in best.items()
                        if back or order.index(Q) <= i]
                if not come:
                    continue
                cost, _, path = min(come, key=lambda x: x[:2])
            row[S] = (cost + max(t[S] / low - 1 - CHANGE, 0.0), path + (S,))
        best = row
    return list(min(best.items(), key=lambda x: (x[1][0], -order.index(x[0])))[1][1])


def tune_set(name, batches, reps, log):
    pid = C.param_id(name)
    p = C.params(pid)
    B = max(batches)
    rng = np.random.default_rng(pid)
    D = C.DeviceBuffer
    stream = C.Stream()
    sh = stream.handle
    d_seed = D.from_array(rng.integers(0, 256, B * 3 * p.n, dtype=np.uint8))
    d_opt = D.from_array(rng.integers(0, 256, B * p.n, dtype=np.uint8))
    d_msg = D.from_array(rng.integers(0, 256, B * 32, dtype=np.uint8))
    d_moff = D.from_array(np.arange(B, dtype=np.uint64) * 32)
    d_mlen = D.from_array(np.full(B, 32, np.uint32))
    d_pk, d_sk, d_sig = D(B * p.pk_bytes), D(B * p.sk_bytes), D(B * p.sig_bytes)
    V = max(BATCHES_VERIFY + BATCHES_KEYGEN)
    ws = D(max(C.workspace_bytes(pid, B if op == 0 else V, op) for op in (0, 1, 2)))
    C.keygen_device(pid, B, d_seed.ptr, 3 * p.n, d_pk.ptr, d_sk.ptr, ws.ptr, sh)
    C.sign_device(pid, B, d_sk.ptr, p.sk_bytes, d_msg.ptr, d_moff.ptr, d_mlen.ptr, d_opt.ptr,
                  d_sig.ptr, p.sig_bytes, ws.ptr, sh)
    stream.sync()

    def rows_of(buf, item):  # verification's V requests repeat the signed ones
        a = buf.download().reshape(B, -1)
        return D.from_array(a[np.arange(V) % B, :item])

    v_pk, v_sig, v_msg = rows_of(d_pk, p.pk_bytes), rows_of(d_sig, p.sig_bytes), rows_of(d_msg, 32)
    v_moff = D.from_array(np.arange(V, dtype=np.uint64) * 32)
    v_mlen, d_st = D.from_array(np.full(V, 32, np.uint32)), D(4 * V)
    k_seed = D.from_array(rng.integers(0, 256, V * 3 * p.n, dtype=np.uint8))
    k_pk, k_sk = D(V * p.pk_bytes), D(V * p.sk_bytes)
    hi = 128 if p.len > 64 else 64
    order = {0: (16, 4, 1), 2: (16, 4, 1),  # 2 and 8 run as 4 and 16
             1: (1,) + tuple(G for G in (128, 64, 32, 16) if G <= hi)}
    rows = []
    for op_name, op in OPS.items():
        grid, timed, first = (batches, BATCHES_VERIFY, BATCHES_KEYGEN)[op], [], 0
        for b in grid:
            sizes = {b, (first + b) // 2 or b} if op == 1 else {b}
            first = b + 1

            def run(b):
                if op == 0:
                    C.sign_device(pid, b, d_sk.ptr, p.sk_bytes, d_msg.ptr, d_moff.ptr,
                                  d_mlen.ptr, d_opt.ptr, d_sig.ptr, p.sig_bytes, ws.ptr, sh)
                elif op == 1:
                    C.verify_device(pid, b, v_pk.ptr, p.pk_bytes, v_sig.ptr, p.sig_bytes,
                                    v_msg.ptr, v_moff.ptr, v_mlen.ptr, d_st.ptr, ws.ptr, sh)
                else:
                    C.keygen_device(pid, b, k_seed.ptr, 3 * p.n, k_pk.ptr, k_sk.ptr, ws.ptr, sh)
            times, seen = {}, set()
            for S in order[op]:
                C.set_split(pid, op, S)
                eff = C.get_split(pid, op, b)
                if eff in seen:
                    continue
                seen.add(eff)
                times[eff] = sum(_time(lambda: run(n), stream, reps) for n in sizes) / len(sizes)
            C.set_split(pid, op, 0)
            if op == 1:
                st = d_st.download(np.int32, b)
                if np.count_nonzero(st):
                    raise RuntimeError("%s: verify rejected a valid signature" % name)
            timed.append(times)
        first = 0
        for b, times, S in zip(grid, timed, settle(timed, order[op], back=op == 1)):
            rows.append((name, op_name, first if op == 1 else b * p.d if op == 0 else b, S))
            first = b + 1
            now = C.get_split(pid, op, b)
            log("%-14s %-6s batch %5d  %s  -> S=%d (now S=%d, %.3f vs %.3f ms)" % (
                name, op_name, b, " ".join("S%d %.3f" % kv for kv in sorted(times.items())), S,
                now, times[S], times.get(now, float("nan"))))
    for buf in (d_seed, d_opt, d_msg, d_moff, d_mlen, d_pk, d_sk, d_sig, d_st, ws, v_pk, v_sig,
                v_msg, v_moff, v_mlen, k_seed, k_pk, k_sk):
        buf.free()
    return rows


def compact(rows):
    """Keep only the lines where a set's choice changes as the batch grows."""
    out, last = [], {}
    for name, op, trees, S in sorted(rows, key=lambda r: (r[0], r[1], r[2])):
        key = (name, op)
        if last.get(key) != S:
            out.append((name, op, 0 if key not in last else trees, S))
            last[key] = S
    return out


def main(argv=None):
    ap = argparse.ArgumentParser()
    ap.add_argument("--sets", default="all")
    ap.add_argument("--reps", type=int, default=6)
    ap.add_argument("--out", default=os.path.join(os.path.dirname(os.path.abspath(__file__)),
                                                  "tuning.txt"))
    a = ap.parse_args(argv)
    names = [C.params(i).name.decode() for i in range(12)] if a.sets == "all" else \
        a.sets.split(",")
    log = lambda s: print(s, flush=True)
    rows, t0 = [], time.perf_counter()
    for name in names:
        small = name.endswith("s") and ("192" in name or "256" in name)
        rows += tune_set(name, BATCHES_SMALL if small else BATCHES_FAST, a.reps, log)
    with open(a.out, "w") as f:
        f.write("# k_ht lanes per leaf (sign, keygen; min_units = subtrees) and k_vht lanes per\n"
                "# request (verify; min_units = requests): <set> <op> <min_units> <lanes>\n")
        f.write("# measured by python -m cuspx_amd.autotune on %s (%.0f s)\n"
                % (C.device_info()["name"], time.perf_counter() - t0))
        for r in compact(rows):
            f.write("%s %s %d %d\n" % r)
    log("wrote %s" % a.out)
    return 0


if __name__ == "__main__":
    sys.exit(main())
