"""The packed NW kernels' direction scratch: next to the generic kernel's under a
memory limit that holds the call without it, and no larger than the waves that
the chip holds."""
import ctypes

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


def test_reads_with_other_bytes_take_slots_for_their_waves():
    """Their kernels run fewer waves per SIMD (4 for 5 at these widths), so a
    call that fills the chip needs as many fewer direction slots."""
    rng = np.random.default_rng(5)
    plain = _reads(rng.integers(60, 101, 400), 6)
    bases = bytearray(plain.bases)
    bases[int(plain.offsets[200]) + 7] = ord("N")
    ambiguous = ca.Reads(bytes(bases), plain.offsets)
    pairs = rng.integers(0, plain.n, (800000, 2)).astype(np.int32)
    held, got = [], []
    for reads in (plain, ambiguous):
        with ca.Context(0) as c:
            c._L.crispy_ctx_scratch_bytes.restype = ctypes.c_int64
            c.upload_reads(ca.NW, reads)
            got.append(c.nw_dists(pairs, 10))
            held.append(c._L.crispy_ctx_scratch_bytes(c._h))
    print(held, flush=True)
    assert 0 < held[1] <= 0.8 * held[0] + 1
    clean = (pairs != 200).all(1)
    assert np.array_equal(got[0][clean], got[1][clean])
