"""The packed NW kernels' scratch next to the generic kernel's, under a memory
limit that holds the call without the former."""
import numpy as np
import pytest

import crispy_amd as ca

pytestmark = pytest.mark.gpu


def _reads(lens, seed):
    rng = np.random.default_rng(seed)
    base = rng.integers(0, 4, max(lens))
    out = []
    for L in lens:
        s = base[:L].copy()
        hit = rng.random(L) < 0.05
        s[hit] = rng.integers(0, 4, int(hit.sum()))
        out.append(np.frombuffer(b"ACGT", np.uint8)[s].tobytes())
    return ca.Reads.from_list(out)


@pytest.mark.parametrize("slack", [0, 390 << 20, 640 << 20])
def test_packed_and_generic_pairs_share_a_limit(slack):
    """Full alignments of ACGT reads of 560-1,500 bp: the shorter pairs run
    packed (their scratch takes 400-690 MB of a limit that leaves it that),
    those past the widest band in the generic kernel."""
    lens = np.random.default_rng(3).integers(560, 640, 60)
    lens[::4] = np.random.default_rng(4).integers(800, 1501, 15)
    reads = _reads(lens, 1)
    pairs = np.random.default_rng(2).integers(0, reads.n, (3000, 2)).astype(np.int32)
    with ca.Context(0) as c:
        c._check(c._L.crispy_ctx_set_scratch_limit(c._h, 0))
        c.upload_reads(ca.NW, reads)
        want = c.nw_dists(pairs, 1)
        need = c.device_bytes()
    with ca.Context(0) as c:
        c.mem_limit(need + slack)
        c.upload_reads(ca.NW, reads)
        for _ in range(2):
            print("slack", slack, flush=True)
            assert np.array_equal(c.nw_dists(pairs, 1), want)
            assert c.device_bytes() <= need + slack
