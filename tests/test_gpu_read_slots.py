"""Uploads of reads with other bytes than ACGT when memory is short, and
uploads that fail or hold only such reads: the distances stay those of a context without a limit, and
no call finds reads that are not whole in a slot."""
import time

import numpy as np
import pytest

import crispy_amd as ca

pytestmark = pytest.mark.gpu

BAND = 10


def _reads(n, seed, other=b"", lo=150, hi=400):
    """n reads of one backbone; `other` bytes in every third of them."""
    rng, at = np.random.default_rng(seed), np.random.default_rng(seed + 1000)  # the same lengths whatever `other` is
    base = rng.integers(0, 4, hi)
    out = []
    for k in range(n):
        s = base.copy()
        hit = rng.random(hi) < 0.05
        s[hit] = rng.integers(0, 4, int(hit.sum()))
        a = np.frombuffer(b"ACGT", np.uint8)[s][:rng.integers(lo, hi + 1)].copy()
        if other and k % 3 == 0:
            a[at.integers(0, a.size, 5)] = np.frombuffer(other, np.uint8)[at.integers(0, len(other), 5)]
        out.append(a.tobytes())
    return ca.Reads.from_list(out)


def _pairs(n, count, seed=9):
    return np.random.default_rng(seed).integers(0, n, (count, 2)).astype(np.int32)


def _free(reads, pairs):
    with ca.Context(0) as c:
        c.upload_reads(ca.NW, reads)
        uploaded = c.device_bytes()
        return c.nw_dists(pairs, BAND), uploaded, c.device_bytes()


def test_upload_without_room_for_the_upper_code_bits():
    """A limit that holds the reads but not the packed kernels' extra code bits."""
    plain, ambiguous = _reads(3000, 1), _reads(3000, 1, b"N")
    assert plain.n == ambiguous.n and np.array_equal(plain.offsets, ambiguous.offsets)
    pairs = _pairs(plain.n, 4000)
    want, _, _ = _free(ambiguous, pairs)
    _, held, _ = _free(plain, pairs)
    with ca.Context(0) as c:
        c.mem_limit(held)
        c.upload_reads(ca.NW, ambiguous)
        assert c.device_bytes() <= held
        c.mem_limit(0)
        assert np.array_equal(c.nw_dists(pairs, BAND), want)
        c.upload_reads(ca.NW, ambiguous)  # with room now
        assert np.array_equal(c.nw_dists(pairs, BAND), want)


def test_upper_code_bits_make_room_for_later_buffers():
    """A limit that holds a whole call without the code bits (their need
    measured with thirteen distinct other bytes, which have none) holds it for
    reads whose code bits fit at the upload."""
    ambiguous, many = _reads(3000, 2, b"N"), _reads(3000, 2, b"BDEFHIJKLMNOP")
    pairs = _pairs(ambiguous.n, 20000)
    want, uploaded, _ = _free(ambiguous, pairs)
    with ca.Context(0) as c:
        c.upload_reads(ca.NW, many)
        assert c.device_bytes() < uploaded
        c._check(c._L.crispy_ctx_set_scratch_limit(c._h, 0))
        c.nw_dists(pairs, BAND)
        need = c.device_bytes()
    assert need > uploaded
    with ca.Context(0) as c:
        c.mem_limit(need)
        for _ in range(3):
            c.upload_reads(ca.NW, ambiguous)
            assert np.array_equal(c.nw_dists(pairs, BAND), want)
            assert c.device_bytes() <= need


def test_failed_upload_leaves_an_empty_slot():
    first, second = _reads(500, 3), _reads(4000, 4)
    pairs = _pairs(first.n, 1000)
    want, _, _ = _free(first, pairs)
    with ca.Context(0) as c:
        for slot in (ca.KMER, ca.NW):
            c.upload_reads(slot, first)
        count = c.kmer_run(6, 0.4)
        assert count > 0
        kept = c.kmer_fetch()
        c.mem_limit(c.device_bytes())
        for slot in (ca.KMER, ca.NW):
            with pytest.raises(ca.CrispyError) as e:
                c.upload_reads(slot, second)
            assert e.value.code == -3
            with pytest.raises(ca.CrispyError):
                c.nw_dists(_pairs(second.n, 1000) if slot == ca.KMER else pairs, BAND)
        with pytest.raises(ca.CrispyError):
            c.nw_run_on_kmer(BAND, 0.4)
        again = c.kmer_fetch()  # the finished result is still there
        assert all(np.array_equal(a, b) for a, b in zip(kept, again))
        c.mem_limit(0)
        c.upload_reads(ca.NW, first)
        assert np.array_equal(c.nw_dists(pairs, BAND), want)


def test_refused_upload_leaves_the_slot_as_it_was():
    first = _reads(300, 5)
    pairs = _pairs(first.n, 1000)
    want, _, _ = _free(first, pairs)
    with ca.Context(0) as c:
        c.upload_reads(ca.NW, first)
        bad = ca.Reads.from_list([b"ACGT" * 10, b"ACGT" * 600])
        with pytest.raises(ca.CrispyError) as e:
            c.upload_reads(ca.NW, bad)
        assert e.value.code == -1
        assert np.array_equal(c.nw_dists(pairs, BAND), want)


@pytest.mark.parametrize("slot", [ca.KMER, ca.NW])
def test_lowercase_reads_upload_like_others(slot):
    """Every base another byte than ACGT: one global atomic per base made this
    upload 250 times as long as that of ACGT reads; 3 leaves room for noise."""
    n, L = 20000, 600
    codes = np.random.default_rng(6).integers(0, 4, n * L)
    times = {}
    for letters in (b"ACGT", b"acgt"):
        reads = ca.Reads(np.frombuffer(letters, np.uint8)[codes].tobytes(), np.arange(n + 1, dtype=np.int64) * L)
        with ca.Context(0) as c:
            best = 1e9
            for _ in range(6):
                t0 = time.perf_counter()
                c.upload_reads(slot, reads)
                c.sync()
                best = min(best, time.perf_counter() - t0)
        times[letters] = best
        print(letters, best, flush=True)
    assert times[b"acgt"] < 3 * times[b"ACGT"]
