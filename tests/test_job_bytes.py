"""The server's estimate of a job's device bytes, without a GPU."""
import numpy as np
import pytest

import crispy_amd as ca


def _estimate(n, length, K):
    """Both read slots, profiles, k-mer result at its first size, up to 256
    passing pairs per read; K = 7, 8 also the K-mer lists and the candidates.
    K = 6 runs need no candidates: large ones take them where there is room."""
    nb, nbases = (n + 127) // 128, n * length
    guess = min(1 << 22, max(4096, nb * (nb + 1) // 2 * 128 * 128))
    pairs = min(n * (n - 1) // 2, 256 * n)
    words = max(16, 4 ** min(K, 6) // 32)
    est = 2 * (nbases + nbases // 4 + 48 * n) + n * (4 * words + 48) + 6 * nbases + 12 * guess + 72 * pairs + (8 << 20)
    if K > 6:
        est += 2 * nbases + 276 * n + 16 * (max(guess, pairs) + 256) + (1 << 20)
    return est


@pytest.mark.parametrize("K", [4, 6, 7, 8])
@pytest.mark.parametrize("n", [1, 100, 28000, 28500, 40000, 50000])
def test_estimate_is_what_the_job_cannot_do_without(n, K):
    length = 40
    reads = ca.Reads(b"ACGT" * (n * length // 4), np.arange(n + 1, dtype=np.int64) * length)
    assert ca.job_bytes(reads, K, 10) == _estimate(n, length, K)
