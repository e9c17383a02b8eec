"""The packed 16-bit NW kernels against the unpacked ones (no direction scratch
allowed) over every pair, and against the CPU oracle over a sample, bit for
bit: every slice width, several lanes per pair, both frames, positions past the
band, full alignments, other bytes, the 16-bit range's end and short scratch."""
import ctypes

import numpy as np
import pytest

import crispy_amd as ca
from oracle import oracle as O

pytestmark = pytest.mark.gpu

# n, shortest, longest, band, pairs, other bytes, scratch limits (-1: the default)
CASES = {
    "every width, one lane per pair": (700, 1, 79, 2, 300000, b"", [-1]),
    "few pairs, narrow slices": (200, 60, 400, 10, 150, b"", [-1]),
    "one pair": (2, 299, 300, 10, 1, b"", [-1]),
    "several lanes per pair": (200, 100, 320, 2, 20000, b"", [1 << 20, 20 << 20, -1]),
    "full alignments": (120, 1, 300, 1, 3000, b"", [-1]),
    "full alignments past the widest band": (40, 560, 760, 1, 300, b"", [-1]),
    "16-bit range": (60, 1300, 1900, 10, 1500, b"", [8 << 20, -1]),
    "half-precision range": (80, 650, 800, 6, 2000, b"", [-1]),
    "one other byte": (150, 150, 330, 7, 8000, b"N", [-1]),
    "twelve other bytes": (150, 20, 120, 2, 30000, b"NRYKMSWBDHVn", [-1]),
    "thirteen other bytes": (100, 20, 120, 2, 500, b"NRYKMSWBDHVnx", [-1]),
    "other bytes, full alignments": (60, 30, 280, 1, 1000, b"N-", [-1]),
}


def _reads(rng, n, lo, hi, other):
    base = rng.integers(0, 4, hi + 8)
    out = []
    for k in range(n):
        s = base.copy()
        hit = rng.random(s.size) < rng.choice([0.01, 0.08, 0.3])
        s[hit] = rng.integers(0, 4, hit.sum())
        for _ in range(3):
            s = np.delete(s, rng.integers(0, s.size))
            s = np.insert(s, rng.integers(0, s.size), rng.integers(0, 4))
        a = np.frombuffer(b"ACGT", np.uint8)[s][rng.integers(0, 8):][:rng.integers(lo, hi + 1)].copy()
        if other and rng.random() < 0.5:
            at = rng.integers(0, a.size, max(1, a.size // 20))
            a[at] = np.frombuffer(other, np.uint8)[rng.integers(0, len(other), at.size)]
        out.append(a.tobytes())
    return out


@pytest.mark.parametrize("name", list(CASES))
def test_packed_equals_unpacked_and_oracle(name):
    n, lo, hi, band, npairs, other, limits = CASES[name]
    print(name, flush=True)
    rng = np.random.default_rng(sorted(CASES).index(name))
    reads = ca.Reads.from_list(_reads(rng, n, lo, hi, other))
    pairs = rng.integers(0, n, (npairs, 2)).astype(np.int32)
    some = rng.permutation(npairs)[:400]
    want, _, _ = O.nw_pairs(O.Reads(reads.bases, reads.offsets, reads.maxlen), np.ascontiguousarray(pairs[some]), band)
    with ca.Context(0) as ctx:
        lib = ctx._L
        lib.crispy_ctx_scratch_bytes.restype = ctypes.c_int64

        def limited(limit):
            ctx._check(lib.crispy_ctx_set_scratch_limit(ctx._h, ctypes.c_int64(limit)))

        ctx.upload_reads(ca.NW, reads)
        limited(0)
        plain = ctx.nw_dists(pairs, band)
        assert lib.crispy_ctx_scratch_bytes(ctx._h) == 0
        assert np.array_equal(plain[some].view(np.uint32), want.view(np.uint32))
        for limit in limits:
            limited(limit)
            for _ in range(3):  # launched, then replayed from the captured graph
                got = ctx.nw_dists(pairs, band)
                assert np.array_equal(got.view(np.uint32), plain.view(np.uint32))
            held = lib.crispy_ctx_scratch_bytes(ctx._h)
            assert limit < 0 or held <= limit
            if limit < 0:
                assert held > 0 or len(other) > 12


def test_scratch_makes_room_for_other_buffers():
    """Under a memory limit that holds a job without directions' scratch, a
    smaller job's scratch is given back when the larger one's buffers grow."""
    print("scratch makes room", flush=True)
    rng = np.random.default_rng(5)
    small = ca.Reads.from_list(_reads(rng, 300, 200, 300, b""))
    large = ca.Reads.from_list(_reads(rng, 6000, 200, 300, b""))
    pairs = rng.integers(0, 300, (40000, 2)).astype(np.int32)

    def job(ctx, reads):
        ctx.upload_reads(ca.KMER, reads)
        ctx.upload_reads(ca.NW, reads)
        ctx.kmer_run(6, 0.3)
        return ctx.nw_dists(pairs, 10)

    with ca.Context(0) as ctx:
        lib = ctx._L
        lib.crispy_ctx_scratch_bytes.restype = ctypes.c_int64
        ctx._check(lib.crispy_ctx_set_scratch_limit(ctx._h, ctypes.c_int64(0)))
        want = [job(ctx, small), job(ctx, large)]
        need = ctx.device_bytes()
    with ca.Context(0) as ctx:
        ctx._check(lib.crispy_ctx_set_mem_limit(ctx._h, ctypes.c_int64(need + (1 << 20))))
        got = job(ctx, small)
        assert np.array_equal(got, want[0])
        assert lib.crispy_ctx_scratch_bytes(ctx._h) > 0
        for _ in range(2):
            got = job(ctx, large)
            assert np.array_equal(got, want[1])
            assert ctx.device_bytes() <= need + (1 << 20)
