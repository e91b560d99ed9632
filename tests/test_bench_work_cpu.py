"""The work that bench.py's roofline divides by at the headline batch
(chain_work: what k_chains runs), pinned to the hash blocks the oracle counts
while it makes a WOTS public key (wots.cu:27-62: a PRF and 15 F per chain)."""
import os
import sys

import pytest

from oracle import oracle as O

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)
import bench  # noqa: E402


@pytest.mark.parametrize("pid", range(12))
def test_chain_work_matches_the_oracles_block_counts(pid):
    p = O.params(pid)
    O.reset_counts()
    O.wots_gen_pk(pid, bytes(range(p.n)), bytes(range(1, p.n + 1)), O.make_addr(pid))
    sha, keccak = O.counts()
    leaf = sha if p.hash == 0 else keccak
    leaves = p.d << (p.full_h // p.d)
    assert bench.chain_work(p, 1) == leaves * leaf
    assert bench.chain_work(p, 4096) == 4096 * bench.chain_work(p, 1)


def test_headline_work_per_launch():
    """SHA2-128f, 4096 requests: the work_per_launch figure of the bench line
    (the chains of one k_chains launch, or of its slices together)."""
    assert bench.chain_work(O.params(O.param_id("sha2-128f")), 4096) == 403701760
