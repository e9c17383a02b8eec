"""The hashed candidate sweep against exact counts in the tile, every pair and
distance bit for bit: read counts around a wave's, a tile's, a row pair's and a
super-tile's edge, counts at which a block sweeps 1, 2 and 16 column tiles, tile
ranges that cut sweeps, and both bucket counts it takes."""
import numpy as np
import pytest

import crispy_amd as ca

pytestmark = pytest.mark.gpu

# reads, shortest, longest, buckets, tile ranges as fractions of all slots
CASES = [
    (2, 30, 60, 1280, [0, 1]),
    (63, 30, 300, 1536, [0, 1]),
    (65, 30, 300, 1280, [0, 1]),
    (128, 300, 900, 1280, [0, 1]),
    (129, 30, 300, 1280, [0, 1]),
    (257, 30, 300, 1536, [0, 0.01, 0.5, 1]),
    (2048, 30, 120, 1280, [0, 0.1, 1]),
    (2049, 30, 120, 1536, [0, 0.3, 0.31, 1]),
    (4301, 30, 80, 1280, [0, 0.003, 0.501, 1]),
    (23011, 20, 40, 1280, [0, 0.4003, 1]),
    (66003, 20, 30, 1280, [0, 1]),
]


@pytest.mark.parametrize("n,lo,hi,buckets,cuts", CASES)
def test_sweep_equals_counts_in_the_tile(n, lo, hi, buckets, cuts):
    print("sweep", n, lo, hi, buckets, flush=True)
    rng = np.random.default_rng(n)
    lens = rng.integers(lo, hi + 1, n)
    base = rng.integers(0, 4, (max(1, n // 40), hi))
    codes = base[rng.integers(0, len(base), n)]
    hit = rng.random(codes.shape) < 0.03
    codes[hit] = rng.integers(0, 4, int(hit.sum()))
    flat = np.frombuffer(b"ACGT", np.uint8)[codes][np.arange(hi)[None, :] < lens[:, None]]
    reads = ca.Reads(flat.tobytes(), np.concatenate([[0], np.cumsum(lens)]))
    with ca.Context(0) as ctx:
        ctx.upload_reads(ca.KMER, reads)
        slots = ca.api.load_library().crispy_kmer_num_tiles(n)
        ctx.kmer_exact_pass(0)
        ctx.kmer_run(6, 0.4)
        want_p, want_d = ctx.kmer_fetch()
        assert n < 40 or len(want_d) > 0
        ctx.kmer_exact_pass(1)
        ctx.kmer_hash_buckets(buckets)
        got = []
        for t0, t1 in zip(cuts[:-1], cuts[1:]):
            for _ in range(2):  # launched, then replayed from the captured graph
                ctx.kmer_run(6, 0.4, tiles=(int(t0 * slots), int(t1 * slots)))
            got.append(ctx.kmer_fetch())
        p = np.concatenate([x[0] for x in got])
        d = np.concatenate([x[1] for x in got])
        order = np.lexsort((p[:, 1], p[:, 0]))
        assert np.array_equal(p[order], want_p)
        assert np.array_equal(d[order].view(np.uint32), want_d.view(np.uint32))
