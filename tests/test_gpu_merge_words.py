"""The duplicate merge's word-wise compare at the edges of its words and blocks:
lengths 0 to 100, the one differing byte at every position, bytes above 127 and
NUL, equal reads whose following bytes differ, at every alignment."""
import numpy as np
import pytest

import crispy_amd as ca

pytestmark = pytest.mark.gpu


def _merge(seqs):
    """Stable (length, bytes) order, each run of equal reads on its last one."""
    order = sorted(range(len(seqs)), key=lambda r: (len(seqs[r]), seqs[r]))
    out, freq = [], []
    for r in order:
        if out and seqs[out[-1]] == seqs[r]:
            out[-1] = r
            freq[-1] += 1
        else:
            out.append(r)
            freq.append(1)
    return out, freq


@pytest.mark.parametrize("lengths", [range(0, 10), range(28, 42), range(60, 70), (96, 97, 300)])
def test_word_compare_edges(lengths):
    print("merge words", list(lengths), flush=True)
    rng = np.random.default_rng(len(lengths))
    seqs = []
    for n in lengths:
        base = rng.integers(0, 256, n).astype(np.uint8)
        seqs += [base.tobytes(), base.tobytes()]
        for p in range(n):
            for b in (0, 1, 127, 128, 255):
                s = base.copy()
                s[p] = b
                seqs.append(s.tobytes())
    seqs = [seqs[k] for k in rng.permutation(len(seqs))]
    with ca.Context(0) as ctx:
        order, freq = ctx.preprocess_order(ca.Reads.from_list(seqs), np.ones(len(seqs), np.int32))
    want_o, want_f = _merge(seqs)
    assert np.array_equal(order, want_o) and np.array_equal(freq, want_f)
