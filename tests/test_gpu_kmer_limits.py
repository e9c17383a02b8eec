"""Large k = 6 runs (from 4 x 10^8 pairs up, which take candidates) where
memory holds the counts in the tile only: the same pairs and distances, in a
context with a limit and in a server with a budget."""
import numpy as np
import pytest

import crispy_amd as ca

pytestmark = pytest.mark.gpu

N, THR, BAND = 29000, 0.25, 10


@pytest.fixture(scope="module")
def reads():
    rng = np.random.default_rng(1)
    lens = rng.integers(60, 91, N)
    codes = rng.integers(0, 4, (1500, 90))[rng.integers(0, 1500, N)]
    hit = rng.random(codes.shape) < 0.02
    codes[hit] = rng.integers(0, 4, int(hit.sum()))
    flat = np.frombuffer(b"ACGT", np.uint8)[codes][np.arange(90)[None, :] < lens[:, None]]
    return ca.Reads(flat.tobytes(), np.concatenate([[0], np.cumsum(lens)]))


def _job(ctx, reads):
    for slot in (ca.KMER, ca.NW):
        ctx.upload_reads(slot, reads)
    ctx.kmer_run(6, THR)
    k = ctx.kmer_fetch()
    ctx.nw_run_on_kmer(BAND, THR)
    return (*k, *ctx.nw_fetch())


def _same(a, b):
    return all(np.array_equal(x, y) for x, y in zip(a, b))


@pytest.fixture(scope="module")
def in_tile(reads):
    """The job with counts in the tile and no directions, and what it holds."""
    with ca.Context(0) as c:
        c.kmer_exact_pass(0)
        c._check(c._L.crispy_ctx_set_scratch_limit(c._h, 0))
        got = _job(c, reads)
        assert len(got[1]) > 10000 and len(got[3]) > 1000
        return got, c.device_bytes()


def test_limit_that_holds_the_counts_in_the_tile(reads, in_tile):
    want, need = in_tile
    with ca.Context(0) as c:
        c.mem_limit(need)
        for _ in range(3):
            print("limit", need, flush=True)
            assert _same(_job(c, reads), want)
            assert c.device_bytes() <= need
        c.mem_limit(0)  # candidates again
        assert _same(_job(c, reads), want)
        assert c.kmer_tile_bits() == 1280


def test_candidates_make_room_for_the_pairs(reads, in_tile):
    """A limit that holds the k-mer run's candidates, then not the NW stage's
    buffers beside them."""
    want, need = in_tile
    with ca.Context(0) as c:
        c.upload_reads(ca.KMER, reads)
        c.kmer_run(6, THR)
        assert c.kmer_tile_bits() == 1280
    with ca.Context(0) as c:
        c.mem_limit(need + (24 << 20))
        for _ in range(2):
            print("limit", need + (24 << 20), flush=True)
            assert _same(_job(c, reads), want)


def test_budget_that_holds_the_counts_in_the_tile(reads, in_tile):
    want, _ = in_tile
    n, nb, nbases = reads.n, (reads.n + 127) // 128, len(reads.bases)
    guess = min(1 << 22, nb * (nb + 1) // 2 * 128 * 128)
    budget = 2 * (nbases + nbases // 4 + 48 * n) + n * (4 * 128 + 48) + 6 * nbases + 12 * guess + 72 * 256 * n + (8 << 20)
    with ca.Server(0, 1, budget) as srv:
        for _ in range(2):
            jid = srv.submit(reads, 6, THR, BAND, THR)
            assert _same(srv.fetch(jid), want[2:])
        assert srv.status()["peak_reserved_bytes"] <= budget
