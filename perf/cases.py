"""Performance cases of the kmerDist -> genDist path, through the Python API.

Each case is what a program does with one read set: the whole distance step
(k-mer profiles, all-pairs k-mer filter, banded NW on the passing pairs, the
output files sorted by (dist, i, j)), NW distances of given pairs, a served
job stream, or the duplicate merge of the input side.  Reads are synthetic
16S-like sets: one backbone, species copies of a window of it, per-base noise,
lengths by a length law, in the (length, bytes) order the preprocess stage
writes, so i < j implies len(i) <= len(j).
"""
import math
from itertools import groupby

import numpy as np
import torch

import crispy_amd as ca
from crispy_amd.pipeline import OutputBuffers, fused_output_files

LETTERS = b"ACGT"  # in byte order, so codes compare like bytes

# Fields: n reads, lengths lo..hi (uniform, or log-normal around `median` with
# `sigma`, clipped), species, divergence of a species in [div_lo, div_hi],
# substitution / indel rates per base, k, band.
LISTED = [
    # One small sample through the two executables' defaults (k 6, band 2),
    # host reads in, files out: launches, read-backs and host work count.
    dict(name="sample600_defaults", kind="pipeline", n=600, lo=200, hi=300, median=0, sigma=0.0, species=20,
         div_lo=0.03, div_hi=0.10, p_sub=0.01, p_indel=0.005, k=6, band=2, amb=0.0),
    # The 1,000-read configuration with the reads resident: the smallest step.
    dict(name="step_1k", kind="step", n=1000, lo=200, hi=300, median=0, sigma=0.0, species=20,
         div_lo=0.03, div_hi=0.10, p_sub=0.01, p_indel=0.005, k=6, band=10, amb=0.0),
    # A mid-size job from host reads to files: what each job of a stream is,
    # uploads and packing included; ragged lengths.
    dict(name="pipeline_9k", kind="pipeline", n=9001, lo=150, hi=550, median=300, sigma=0.35, species=45,
         div_lo=0.03, div_hi=0.10, p_sub=0.01, p_indel=0.005, k=6, band=10, amb=0.0),
    # The 20,000-read configuration: most of the step is banded NW.
    dict(name="step_20k", kind="step", n=20000, lo=200, hi=300, median=0, sigma=0.0, species=100,
         div_lo=0.03, div_hi=0.10, p_sub=0.01, p_indel=0.005, k=6, band=10, amb=0.0),
    # The 100,000-read configuration, k 6: the k-mer filter as candidates, NW
    # over a wide spread of lengths, several output files.
    dict(name="step_100k_k6", kind="step", n=100000, lo=150, hi=550, median=300, sigma=0.35, species=500,
         div_lo=0.01, div_hi=0.15, p_sub=0.01, p_indel=0.005, k=6, band=10, amb=0.0),
    # The same read set at k 8: the exact signed-order merges of the lists.
    dict(name="step_100k_k8", kind="step", n=100000, lo=150, hi=550, median=300, sigma=0.35, species=500,
         div_lo=0.01, div_hi=0.15, p_sub=0.01, p_indel=0.005, k=8, band=10, amb=0.0),
    # The 250,000-read configuration, band 5: the largest run on one device.
    dict(name="step_250k", kind="step", n=250000, lo=400, hi=900, median=0, sigma=0.0, species=2000,
         div_lo=0.01, div_hi=0.15, p_sub=0.015, p_indel=0.005, k=6, band=5, amb=0.0),
    # Real read sets hold some ambiguous bases: 2 % of the reads carry an N.
    dict(name="step_ambiguous", kind="step", n=4000, lo=300, hi=500, median=0, sigma=0.0, species=20,
         div_lo=0.03, div_hi=0.10, p_sub=0.01, p_indel=0.005, k=6, band=10, amb=0.02),
    # Distances of given pairs of near full-length reads.
    dict(name="nw_long", kind="nw", n=2000, pairs=20000, lo=1100, hi=1500, median=0, sigma=0.0, species=20,
         div_lo=0.03, div_hi=0.10, p_sub=0.01, p_indel=0.005, band=10),
    # Full alignments (band 1) of given pairs.
    dict(name="nw_full", kind="nw", n=600, pairs=3000, lo=200, hi=300, median=0, sigma=0.0, species=20,
         div_lo=0.03, div_hi=0.10, p_sub=0.01, p_indel=0.005, band=1),
    # A burst of jobs at the job server (4 slots): submit all, fetch all.
    dict(name="serve_8jobs", kind="serve", jobs=8, n=4000, lo=150, hi=550, median=300, sigma=0.35, species=20,
         div_lo=0.03, div_hi=0.10, p_sub=0.01, p_indel=0.005, k=6, band=10, slots=4),
    # Input side: a raw file's records ordered and its duplicates merged.
    dict(name="merge_60k", kind="merge", n=60000, unique=40000, lo=200, hi=300, median=0, sigma=0.0, species=100,
         div_lo=0.03, div_hi=0.10, p_sub=0.01, p_indel=0.005),
]


def listed():
    return [dict(c) for c in LISTED]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: read counts over the logarithm of their range, lengths,
    species, k and band over what the listed cases span."""
    kind = rng.choice(["pipeline", "step", "step", "step", "nw", "nw", "serve", "merge"])
    lo = rng.randint(100, 420)
    hi = lo + rng.randint(0, 480)
    lognormal = rng.random() < 0.4 and hi > lo + 50
    c = dict(kind=kind, lo=lo, hi=hi, median=(lo + hi) // 2 if lognormal else 0, sigma=0.35 if lognormal else 0.0,
             div_lo=rng.uniform(0.01, 0.03), div_hi=rng.uniform(0.08, 0.15), p_sub=rng.uniform(0.005, 0.015),
             p_indel=rng.uniform(0.002, 0.006))
    if kind in ("pipeline", "step"):
        c["n"] = _log_int(rng, 500, 60000 if kind == "step" else 20000)
        c["k"] = rng.choice([5, 6, 6, 6, 7, 8])
        # the default band 2 is a fifth of the read length: small samples only
        c["band"] = rng.choice([5, 8, 10, 10, 20]) if c["n"] > 2000 else rng.choice([2, 3, 5, 10, 10])
        c["species"] = max(5, c["n"] // rng.randint(100, 200))
        c["amb"] = rng.choice([0.0, 0.0, 0.0, 0.01]) if c["n"] <= 4000 else 0.0
    elif kind == "nw":
        c["n"] = _log_int(rng, 300, 3000)
        c["band"] = rng.choice([1, 2, 5, 8, 10, 10, 15, 20])
        c["lo"], c["hi"] = (lo, hi) if c["band"] > 2 else (lo // 2, lo // 2 + 120)
        if c["band"] >= 8 and rng.random() < 0.5:
            c["lo"], c["hi"] = 900, rng.randint(1000, 1500)
        c["median"], c["sigma"] = 0, 0.0
        c["species"] = max(5, c["n"] // 100)
        c["pairs"] = _log_int(rng, 100, 50000 if c["band"] > 2 else 3000)
    elif kind == "serve":
        c.update(n=_log_int(rng, 500, 5000), jobs=rng.randint(2, 8), k=6, band=10, slots=rng.randint(1, 4))
        c["species"] = max(5, c["n"] // 200)
    else:
        c["n"] = _log_int(rng, 1000, 80000)
        c.update(unique=max(1, int(c["n"] * rng.uniform(0.4, 0.95))), species=100)
    return c


# ------------------------------------------------------------------ inputs
def _codes(c, n, seed):
    """(codes (n, hi) uint8 in 0..3 and 0 past the length, lengths), sorted by
    (length, bytes), exact duplicates dropped; on the GPU."""
    dev = torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(seed)

    def rand(*s):
        return torch.rand(*s, generator=g, device=dev)

    def randint(hi, *s):
        return torch.randint(hi, s, generator=g, device=dev, dtype=torch.uint8)

    win = c["hi"]
    if c["median"]:
        z = torch.randn(n, generator=g, device=dev)
        lens = torch.round(c["median"] * torch.exp(c["sigma"] * z)).clamp(c["lo"], c["hi"]).long()
    else:
        lens = c["lo"] + torch.floor(rand(n) * (c["hi"] - c["lo"] + 1)).clamp(max=c["hi"] - c["lo"]).long()
    base = randint(4, win)
    div = c["div_lo"] + (c["div_hi"] - c["div_lo"]) * rand(c["species"], 1)
    spec = base.repeat(c["species"], 1)
    spec = torch.where(rand(c["species"], win) < div, (spec + 1 + randint(3, c["species"], win)) % 4, spec)
    sid = torch.floor(rand(n) * c["species"]).clamp(max=c["species"] - 1).long()
    pos = torch.arange(win, device=dev)
    out = torch.empty(n, win, dtype=torch.uint8, device=dev)
    for b in range(0, n, 32768):
        e = min(n, b + 32768)
        u = rand(e - b, win)
        # one base copied per position; an insertion stays on its source base
        # and writes a random one, a deletion skips one more
        ins, dele = u < c["p_indel"] / 2, (u >= c["p_indel"] / 2) & (u < c["p_indel"])
        src = torch.cumsum(torch.where(ins, 0, torch.where(dele, 2, 1)).to(torch.int16), 1, dtype=torch.int16).long() - 1
        r = torch.gather(spec[sid[b:e]], 1, src.clamp(0, win - 1))
        sub = (u >= c["p_indel"]) & (u < c["p_indel"] + c["p_sub"])
        r = torch.where(sub, (r + 1 + randint(3, e - b, win)) % 4, r)
        r = torch.where(ins | (src >= win), randint(4, e - b, win), r)
        out[b:e] = torch.where(pos < lens[b:e, None], r, torch.zeros_like(r))
    perm = torch.arange(n, device=dev)
    for w in range((win - 1) // 31, -1, -1):  # least significant 31 bases first
        part = out[:, 31 * w:31 * w + 31].long()
        key = (part << (2 * torch.arange(part.shape[1] - 1, -1, -1, device=dev))).sum(1)
        perm = perm[torch.sort(key[perm], stable=True).indices]
    perm = perm[torch.sort(lens[perm], stable=True).indices]
    out, lens = out[perm], lens[perm]
    keep = torch.ones(n, dtype=torch.bool, device=dev)
    keep[1:] = (lens[1:] != lens[:-1]) | (out[1:] != out[:-1]).any(1)
    return out[keep], lens[keep]


def _bytes(codes, lens, amb=0.0, seed=0):
    """Flat read bytes (uint8 numpy) and offsets; `amb` of the reads get one N
    inside (never at their ends, which the reader trims)."""
    table = torch.tensor(list(LETTERS), dtype=torch.uint8, device=codes.device)
    m = table[codes.long()]
    if amb:
        g = torch.Generator(device=codes.device).manual_seed(seed + 7)
        hit = torch.rand(len(lens), generator=g, device=codes.device) < amb
        at = 1 + torch.floor(torch.rand(len(lens), generator=g, device=codes.device) * (lens - 2).float()).long()
        rows = torch.nonzero(hit).flatten()
        m[rows, at[rows]] = ord("N")
    flat = m[torch.arange(m.shape[1], device=codes.device) < lens[:, None]]
    offs = np.zeros(len(lens) + 1, np.int64)
    offs[1:] = np.cumsum(lens.cpu().numpy())
    return flat.cpu().numpy(), offs


def _reads(c, seed, n=None):
    codes, lens = _codes(c, n or c["n"], seed)
    flat, offs = _bytes(codes, lens, c.get("amb", 0.0), seed)
    return ca.Reads(flat.tobytes(), offs)


def _pairs(c, n, seed):
    """`pairs` read pairs i < j in (i, j) order, as a program that picks its
    own candidates passes them."""
    r = np.random.default_rng(seed)
    p = np.sort(r.integers(0, n, (c["pairs"], 2), dtype=np.int32), axis=1)
    p[:, 1] = np.where(p[:, 0] == p[:, 1], (p[:, 1] + 1) % n, p[:, 1])
    p.sort(axis=1)
    return np.ascontiguousarray(p[np.lexsort((p[:, 1], p[:, 0]))])


def _thresholds(n):
    return ca.kmer_default_threshold(n), ca.nw_default_threshold(n)


MAX_FILES = 64


def _room(c, n):
    """Result entries a program makes room for: every pair of a set so small
    that its threshold is loose (up to 500 reads), otherwise about the pairs
    of one species, less where the threshold is tight (large sets)."""
    if n < 600:
        return n * (n - 1) // 2
    same = n * (n - 1) / 2 / c["species"]
    return int(same * (1.3 if n <= 60000 else 0.6 if n < 150000 else 0.1)) + 8000


def prepare(case, seed):
    c = case
    if c["kind"] == "serve":
        # jobs of a stream differ in size
        sizes = [max(50, c["n"] * (q + 1) // c["jobs"]) for q in range(c["jobs"])]
        jobs = [_reads(c, seed * 1000 + q, s) for q, s in enumerate(sizes)]
        return dict(case=c, server=ca.Server(0, slots=c["slots"]), jobs=jobs, thr=[_thresholds(j.n) for j in jobs],
                    out=[(np.zeros((_room(c, s), 2), np.int32), np.zeros(_room(c, s), np.float32)) for s in sizes])
    if c["kind"] == "merge":
        uniq = _reads(c, seed, c["unique"])
        r = np.random.default_rng(seed)
        pick = r.permutation(np.concatenate([np.arange(uniq.n), r.integers(0, uniq.n, c["n"] - uniq.n)])
                             if c["n"] > uniq.n else np.arange(uniq.n))
        flat = np.frombuffer(uniq.bases, np.uint8)
        lens = np.diff(uniq.offsets)[pick]
        offs = np.zeros(len(pick) + 1, np.int64)
        offs[1:] = np.cumsum(lens)
        at = np.repeat(uniq.offsets[pick] - offs[:-1], lens) + np.arange(offs[-1])
        return dict(case=c, ctx=ca.Context(0), reads=ca.Reads(flat[at].tobytes(), offs),
                    freq=np.ones(len(pick), np.int32),
                    out=(np.zeros(len(pick), np.int32), np.zeros(len(pick), np.int32)))
    reads = _reads(c, seed)
    st = dict(case=c, ctx=ca.Context(0), reads=reads, thr=_thresholds(reads.n))
    if c["kind"] == "nw":
        st["pairs"] = _pairs(c, reads.n, seed)
        st["ctx"].upload_reads(ca.NW, reads)
    else:
        # the program's output arrays, kept from pass to pass
        st["buffers"] = OutputBuffers()
        st["buffers"].reserve(_room(c, c["n"]))
        st["buffers"].pairs[:] = 0
        st["buffers"].dists[:] = 0
        if c["kind"] == "step":
            st["ctx"].upload_reads(ca.KMER, reads)
            st["ctx"].upload_reads(ca.NW, reads)
    return st


def run(state):
    c = state["case"]
    if c["kind"] == "serve":
        srv = state["server"]
        ids = [srv.submit(r, c["k"], kt, c["band"], nt) for r, (kt, nt) in zip(state["jobs"], state["thr"])]
        for i, (pairs, dists) in zip(ids, state["out"]):
            p, d = srv.fetch(i)
            pairs[:len(p)], dists[:len(d)] = p, d
        return state["out"]
    ctx = state["ctx"]
    if c["kind"] == "merge":
        order, freq = ctx.preprocess_order(state["reads"], state["freq"])
        state["out"][0][:len(order)], state["out"][1][:len(freq)] = order, freq
        return state["out"]
    if c["kind"] == "nw":
        return ctx.nw_dists(state["pairs"], c["band"])
    if c["kind"] == "pipeline":
        ctx.upload_reads(ca.KMER, state["reads"])
        ctx.upload_reads(ca.NW, state["reads"])
    kthr, nthr = state["thr"]
    ctx.kmer_run(c["k"], kthr)
    ctx.nw_run_on_kmer(c["band"], nthr)
    return _as_output([len(d) for _, d in fused_output_files(ctx, state["buffers"])], state["buffers"].pairs,
                      state["buffers"].dists)


def _as_output(counts, pairs, dists):
    """The files of a step back to back in the program's arrays (zeros past the
    last), and the number of pairs in each."""
    per_file = np.zeros(MAX_FILES, np.int64)
    per_file[:len(counts)] = counts
    return dict(files=per_file, pairs=pairs, dists=dists)


# -------------------------------------------------------------------- work
def _mean_len(c):
    return c["median"] or (c["lo"] + c["hi"]) / 2


def _cells(c, band):
    """In-band cells of one pair of mean-length reads."""
    L = _mean_len(c)
    return L * L if band <= 1 else max(L * (2 * int(L / band) + 1) - (L / band) ** 2, 1.0)


def _step_work(c, n):
    # k-mer lists merged once per pair (T_i + T_j visits); NW at 13 operations
    # per in-band cell on the pairs of one species that pass, about a third
    # (a fiftieth once the threshold is tight against 1.5 % noise)
    L, k = _mean_len(c), c["k"]
    same = n * (n - 1) / 2 / c["species"] * (0.35 if n < 150000 else 0.02)
    return dict(bytes=n * (L + 8) + same * 12, flops=n * (n - 1) / 2 * 2 * (L - k + 1) + same * 13 * _cells(c, c["band"]))


def work(case):
    c = case
    if c["kind"] in ("step", "pipeline"):
        return _step_work(c, c["n"])
    if c["kind"] == "serve":
        parts = [_step_work(c, max(50, c["n"] * (q + 1) // c["jobs"])) for q in range(c["jobs"])]
        return dict(bytes=sum(p["bytes"] for p in parts), flops=sum(p["flops"] for p in parts))
    if c["kind"] == "nw":
        return dict(bytes=c["n"] * (_mean_len(c) + 8) + c["pairs"] * 12, flops=c["pairs"] * 13 * _cells(c, c["band"]))
    return dict(bytes=c["n"] * (_mean_len(c) + 12) + c["unique"] * 8, flops=c["n"] * math.log2(c["n"]))


# ------------------------------------------------------------------- exact
def _passes(dist64, thr):
    d = np.asarray(dist64).astype(np.float32)
    t = np.float32(thr)
    return (d < t) | (np.abs(d - t).astype(np.float64) < 0.00001)


def _kmer_exact(mat, lens, k, thr):
    """Pairs i < j that pass the k-mer filter, in (i, j) order, from
    mat (n, hi) int64 base codes in the order A0 G1 T2 C3 (k <= 7, where the
    merge is the multiset intersection)."""
    n, dev = len(lens), mat.device
    T = lens - k + 1
    code = torch.zeros(n, mat.shape[1] - k + 1, dtype=torch.long, device=dev)
    for q in range(k):
        code = code * 4 + mat[:, q:mat.shape[1] - k + 1 + q]
    valid = torch.arange(code.shape[1], device=dev) < T[:, None]
    counts = torch.zeros(n, 4 ** k, dtype=torch.int16, device=dev)
    counts.scatter_add_(1, code, valid.to(torch.int16))
    out = []
    for i in range(n - 1):
        m = torch.minimum(counts[i], counts[i + 1:]).sum(1, dtype=torch.long)
        d = (1.0 - m.double() / torch.minimum(T[i], T[i + 1:]).double()).cpu().numpy()
        j = np.nonzero(_passes(d, thr))[0]
        out.append(np.stack([np.full(len(j), i), j + i + 1], 1))
    return np.concatenate(out)


def _nw_exact(mat, lens, pairs, band):
    """ML / AL in float64 of every pair: the recurrence along anti-diagonals
    (read i of the pair over columns, read j over rows), all pairs at once."""
    dev, NEG = mat.device, -1000000
    a, b = mat[pairs[:, 0]], mat[pairs[:, 1]]
    L1, L2 = lens[pairs[:, 0]][:, None], lens[pairs[:, 1]][:, None]
    kb = L1 + L2 if band <= 1 else (L1 + L2) // (2 * band)
    rows = int(L2.max()) + 1
    i = torch.arange(rows, device=dev)[None, :]
    z = torch.zeros(len(pairs), rows, dtype=torch.long, device=dev)

    def down(x, fill):  # value of row i - 1 at row i
        return torch.cat([torch.full_like(x[:, :1], fill), x[:, :-1]], 1)

    hist = []  # (M, U, ML, AL, valid) of the last two anti-diagonals
    best = {"I": [torch.full_like(L1, NEG), torch.zeros_like(L1), torch.ones_like(L1)],
            "J": [torch.full_like(L1, NEG), torch.zeros_like(L1), torch.ones_like(L1)]}
    for t in range(0, int(L1.max()) + rows):
        j = t - i
        ok = (j >= 0) & (j <= L1) & (i <= L2) & ((i - j).abs() <= kb)
        edge = ok & ((i == 0) | (j == 0))
        M, U, ML, AL = z.clone(), z.clone(), z.clone(), torch.where(edge, i + j, z)
        if len(hist) == 2:
            inner = ok & ~edge
            dM, dU, dML, dAL, dv = hist[0]
            pM, pU, pML, pAL, pv = hist[1]
            s1 = torch.gather(a, 1, (j - 1).clamp(0, a.shape[1] - 1).expand(len(pairs), -1))
            s2 = torch.gather(b, 1, (i - 1).clamp(0, b.shape[1] - 1).expand(len(pairs), -1))
            eq = (s1 == s2).long()
            diag = down(dM, NEG) + 9 * eq - 4
            up = torch.where(pv, pM + torch.where(pU == 1, -10, torch.where(pU == 3, -1, 0)), NEG)
            lv = down(pM, NEG) + torch.where(down(pU, 0) == 1, -10, torch.where(down(pU, 0) == 2, -1, 0))
            left = torch.where(down(pv.long(), 0) > 0, lv, NEG)
            m = torch.maximum(torch.maximum(diag, up), left)
            u = torch.where(m == diag, 1, torch.where(m == up, 3, 2))
            ml = torch.where(u == 1, down(dML, 0) + 1 - eq, torch.where(u == 3, pML, down(pML, 0)) + 1)
            al = torch.where(u == 1, down(dAL, 0), torch.where(u == 3, pAL, down(pAL, 0))) + 1
            M, U = torch.where(inner, m, M), torch.where(inner, u, U)
            ML, AL = torch.where(inner, ml, ML), torch.where(inner, al, AL)
            for key, line in (("I", inner & (i == L2)), ("J", inner & (j == L1))):
                at = line.long().argmax(1, keepdim=True)
                v, l, x = (torch.gather(q, 1, at) for q in (M, ML, AL))
                take = line.any(1, keepdim=True) & (v >= best[key][0])
                best[key] = [torch.where(take, q, o) for q, o in zip((v, l, x), best[key])]
        hist = (hist + [(M, U, ML, AL, ok)])[-2:]
    last_row = best["I"][0] > best["J"][0]
    ml = torch.where(last_row, best["I"][1], best["J"][1]).double()
    al = torch.where(last_row, best["I"][2], best["J"][2]).double()
    return (ml / al).flatten().cpu().numpy()


def _matrix(reads, lut):
    """(n, maxlen) int64 codes of the read bytes through `lut`."""
    lens = np.diff(reads.offsets)
    flat = lut[np.frombuffer(reads.bases, np.uint8)]
    m = np.zeros((reads.n, int(lens.max())), np.int64)
    m[np.arange(m.shape[1]) < lens[:, None]] = flat
    dev = torch.device("cuda")
    return torch.from_numpy(m).to(dev), torch.from_numpy(lens).to(dev)


def exact(case, seed):
    c = case
    if c["kind"] in ("serve", "merge"):
        return None  # whole numbers (merge); the steps below cover the jobs
    if c["kind"] == "nw":
        if c["pairs"] * c["hi"] ** 2 > 1.5e9:
            return None
        reads = _reads(c, seed)
        mat, lens = _matrix(reads, np.arange(256))
        return _nw_exact(mat, lens, _pairs(c, reads.n, seed).astype(np.int64), c["band"])
    if c["n"] > 1500 or c["k"] > 7:
        return None
    reads = _reads(c, seed)
    kthr, nthr = _thresholds(reads.n)
    code = np.zeros(256, np.int64)
    code[[ord("G"), ord("T"), ord("C")]] = [1, 2, 3]
    mat, lens = _matrix(reads, code)
    pairs = _kmer_exact(mat, lens, c["k"], kthr)
    if len(pairs) * c["hi"] ** 2 > 6e9:
        return None
    raw, lens = _matrix(reads, np.arange(256))
    d = np.concatenate([_nw_exact(raw, lens, pairs[b:b + 20000], c["band"]) for b in range(0, len(pairs), 20000)]
                       or [np.zeros(0)])
    keep = _passes(d, nthr)
    # the files: input pairs in chunks of 589,824, a file closed once it holds
    # 147,456 passing pairs; each ordered by (float32 dist, i, j)
    first = 0
    chunk = np.arange(len(pairs)) // 589824
    ends, done = [], 0
    for _, grp in groupby(range(len(pairs)), key=lambda q: chunk[q]):
        done += int(keep[list(grp)].sum())
        if done - first >= 147456:
            ends.append(done)
            first = done
    if done > first:
        ends.append(done)
    p, d = pairs[keep], d[keep]
    out_p, out_d = np.zeros((_room(c, c["n"]), 2), np.int64), np.zeros(_room(c, c["n"]))
    counts, first = [], 0
    for e in ends:
        o = first + np.lexsort((p[first:e, 1], p[first:e, 0], d[first:e].astype(np.float32)))
        out_p[first:e], out_d[first:e] = p[o], d[o]
        counts.append(e - first)
        first = e
    return _as_output(counts, out_p, out_d)
