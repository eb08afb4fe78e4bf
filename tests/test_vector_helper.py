"""The mapping layer's 1-error search, BWSearch1VectorHelper
(search/search.c:1491-1709) over the interval vectors of
BWExactSearchVectorBackward/Forward (bwt.c:1940-1950, 1994-2003; seed windows
bwt.c:1447-1479).

CPU: the oracle against the golden vectors of the compiled reference (whole
reads and windows), against the compiled reference live when it is built,
and its mismatch records against a brute-force scan of the text (every
single substitution that occurs, once, with its occurrence count).
GPU: fmi_search1_vector_batch through the C ABI against the golden vectors
and the oracle (reads with N, windows, the mismatch projection, truncation,
strand masks)."""
import numpy as np
import pytest

import fmoracle as fo
from conftest import split_golden_hits
from hpgfm import synth


@pytest.fixture(scope="module", params=["golden_small", "golden_repeats"])
def golden(request):
    g = request.getfixturevalue(request.param)
    return g, fo.Oracle(g["genome"], ratio=int(g["ratio"]))


def test_golden_vector_helper(golden):
    g, o = golden
    reads, offs = g["reads"], g["offsets"]
    cap = int(g["cap"])
    whole = split_golden_hits(g, "s1v")
    win = split_golden_hits(g, "s1w")
    for i in range(len(offs) - 1):
        W = reads[offs[i]:offs[i + 1]]
        a, b = (int(x) for x in g["s1w_bounds"][i])
        for s in (0, 1):
            n, h = o.search1_vector(s, W, 0, len(W) - 1, cap=cap)
            assert n == int(g["s1v_counts"][i, s]) and fo.hits_equal(h, whole[(i, s)]), (i, s)
            n, h = o.search1_vector(s, W, a, b, cap=cap)
            assert n == int(g["s1w_counts"][i, s]) and fo.hits_equal(h, win[(i, s)]), (i, s, a, b)


def count_occ(text, pat):
    t = text.tobytes()
    p = pat.tobytes()
    c, i = 0, t.find(p)
    while i >= 0:
        c += 1
        i = t.find(p, i + 1)
    return c


def substitution_positions(hits, start):
    """Position of the substituted base of every MISMATCH record.  A mismatch
    at W[start] that follows an insertion record in the first block carries
    that record's err_pos, the base b in 0..3 (search.c:1556 writes b into
    it); with start >= 4 no other record of the backward half has err_pos
    below start, so such a record is at W[start]."""
    assert start >= 4
    out = []
    for h in hits:
        if h["num_mismatches"] == 0 or int(h["err_kind"]) != fo.MISMATCH:
            continue
        p = int(h["err_pos"])
        if h["dir"] == 0 and p < start:
            p = start
        out.append((p, int(h["err_base"]), int(h["l"] - h["k"] + 1)))
    return out


@pytest.mark.parametrize("seed", [4, 5])
def test_mismatch_records_are_hamming1(seed):
    """Every single substitution of W[start..end] (of its reverse complement
    on strand 1) that occurs in X appears once, with l - k + 1 = its count;
    the exact record counts W itself."""
    g, _, _ = synth.genome(3000, seed=seed, repeat_frac=0.3, fam_len=(100, 400),
                           divergence=(0.0, 0.03), copies_per_family=6)
    o = fo.Oracle(g, ratio=8)
    reads, offs, _ = synth.reads(g, 100, length=30, seed=seed + 10, sub_rate=0.04)
    rng = np.random.default_rng(seed)
    for i in range(len(offs) - 1):
        R = reads[offs[i]:offs[i + 1]]
        a = int(rng.integers(4, 8))
        b = int(rng.integers(len(R) - 6, len(R)))
        for s in (0, 1):
            n, hits = o.search1_vector(s, R, a, b, cap=4096)
            got = {}
            for (p, base, c) in substitution_positions(hits, a):
                assert (p, base) not in got, (i, s, p, base)
                got[(p, base)] = c
            ex = [int(h["l"] - h["k"] + 1) for h in hits if h["num_mismatches"] == 0]
            W = R[a:b + 1]
            c0 = count_occ(g, W if s == 0 else synth.revcomp(W))
            assert ex == ([c0] if c0 else [])
            want = {}
            for p in range(len(W)):
                for base in range(4):
                    if base == W[p]:
                        continue
                    V = W.copy()
                    V[p] = base
                    c = count_occ(g, V if s == 0 else synth.revcomp(V))
                    if c:
                        want[(a + p, base)] = c
            assert got == want, (i, s)
            # the mismatch projection keeps the same records in order
            n_mm, mm = o.search1_vector(s, R, a, b, cap=4096, mismatch_only=True)
            keep = (hits["num_mismatches"] == 0) | (hits["err_kind"] == fo.MISMATCH)
            assert fo.hits_equal(mm, hits[keep])


ref_only = pytest.mark.skipif(not fo.ref_available(), reason="oracle/_ref not built")


@ref_only
def test_oracle_matches_reference_vector_helper():
    g, _, _ = synth.genome(30000, seed=61, repeat_frac=0.3, fam_len=(200, 1500),
                           divergence=(0.0, 0.05))
    o = fo.Oracle(g, ratio=8)
    r = fo.RefCore(oracle=o)
    lens = np.random.default_rng(62).integers(3, 110, 250)
    reads, offs, _ = synth.reads(g, 250, seed=63, sub_rate=0.02, lengths=lens)
    rng = np.random.default_rng(64)
    for i in range(len(offs) - 1):
        W = reads[offs[i]:offs[i + 1]]
        L = len(W)
        a = int(rng.integers(0, L - 2))
        b = int(rng.integers(a + 2, L))
        for (st, en) in ((0, L - 1), (a, b)):
            for s in (0, 1):
                n1, h1 = o.search1_vector(s, W, st, en)
                n2, h2, full = r.search1_vector(s, W, st, en)
                assert n1 == n2 and not full and fo.hits_equal(h1, h2), (i, st, en, s)
                n3, h3, full3 = r.search1_vector(s, W, st, en, cap=2)
                assert fo.hits_equal(h3, h1[:2]) and full3 == (n1 > 2)
    r.close()


# ------------------------------------------------------------------ GPU

@pytest.fixture(scope="module", params=["golden_small", "golden_repeats"])
def vgold(request, gpu_engine):
    g = request.getfixturevalue(request.param)
    ix = gpu_engine.Index.build(g["genome"], int(g["ratio"])).to_device()
    batch = gpu_engine.ReadBatch(g["reads"], g["offsets"])
    yield gpu_engine, g, ix, batch
    batch.free()
    ix.close()


def check(counts, hits, want, cap, project=False):
    for (i, s), w in want.items():
        if project:
            w = w[(w["num_mismatches"] == 0) | (w["err_kind"] == fo.MISMATCH)]
        assert int(counts[i, s]) == len(w), (i, s)
        assert fo.hits_equal(hits[i, s, :min(len(w), cap)], w[:cap]), (i, s)


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["edit", "mismatch"])
def test_gpu_vector_helper_golden(vgold, mode):
    hp, g, ix, batch = vgold
    cap = int(g["cap"])
    m = hp.MODE_EDIT if mode == "edit" else hp.MODE_MISMATCH
    counts, hits = hp.search1_vector_batch(ix, batch, cap=cap, mode=m)
    check(counts, hits, split_golden_hits(g, "s1v"), cap, project=mode == "mismatch")
    counts, hits = hp.search1_vector_batch(ix, batch, cap=cap, mode=m, bounds=g["s1w_bounds"])
    check(counts, hits, split_golden_hits(g, "s1w"), cap, project=mode == "mismatch")


@pytest.mark.gpu
def test_gpu_vector_helper_truncation_and_strands(vgold):
    hp, g, ix, batch = vgold
    want = split_golden_hits(g, "s1v")
    counts, hits = hp.search1_vector_batch(ix, batch, cap=3)
    check(counts, hits, want, 3)
    for mask, s in ((hp.STRAND_PLUS, 0), (hp.STRAND_MINUS, 1)):
        counts, hits = hp.search1_vector_batch(ix, batch, cap=64, strand_mask=mask)
        assert np.all(counts[:, 1 - s] == 0)
        for i in range(counts.shape[0]):
            w = want[(i, s)]
            assert int(counts[i, s]) == len(w)
            assert fo.hits_equal(hits[i, s, :min(len(w), 64)], w[:64])


@pytest.mark.gpu
def test_gpu_vector_helper_vs_oracle_with_n(gpu_engine):
    """Reads with N bases (code 4, a symbol that never occurs), ragged
    lengths 0..250 and random windows, against the oracle."""
    hp = gpu_engine
    g, _, _ = synth.genome(300_000, seed=71, repeat_frac=0.3, fam_len=(300, 2000),
                           divergence=(0.0, 0.05))
    ix = hp.Index.build(g, 16).to_device()
    o = fo.Oracle(g, ratio=16)
    lens = np.random.default_rng(72).integers(0, 251, 1500)
    reads, offs, _ = synth.reads(g, 1500, seed=73, sub_rate=0.01, n_rate=0.003, lengths=lens)
    rng = np.random.default_rng(74)
    bounds = np.zeros((1500, 2), np.int16)
    for i in range(1500):
        L = int(lens[i])
        if L >= 3:
            a = int(rng.integers(0, L - 2))
            bounds[i] = (a, int(rng.integers(a + 2, L)))
        else:
            bounds[i] = (0, L - 1)
    batch = hp.ReadBatch(reads, offs)
    cap = 48
    for bnd in (None, bounds):
        counts, hits = hp.search1_vector_batch(ix, batch, cap=cap, bounds=bnd)
        for i in range(1500):
            W = reads[offs[i]:offs[i + 1]]
            a, b = (0, len(W) - 1) if bnd is None else (int(bnd[i, 0]), int(bnd[i, 1]))
            for s in (0, 1):
                n, h = o.search1_vector(s, W, a, b, cap=cap)
                assert int(counts[i, s]) == n, (i, s, a, b)
                assert fo.hits_equal(hits[i, s, :min(n, cap)], h), (i, s)
    batch.free()
    ix.close()


@pytest.mark.gpu
@pytest.mark.parametrize("n,kmer", [(120_000, 0), (120_000, 7), (120_000, 10), (70, 4), (70, 9)])
def test_gpu_vector_helper_on_text(gpu_engine, n, kmer):
    """The expanded index: windows of 3 to 400 bases (row contexts up to 29,
    the text above, the vectors where more than four rows reach half the
    window), reads past the 256 bases that are staged, on copies (three and
    twelve of them), runs of one base and both ends of the text, in both
    modes and at a capacity that truncates, against the oracle."""
    hp = gpu_engine
    rng = np.random.default_rng(81)
    g = rng.integers(0, 4, n).astype(np.uint8)
    if n > 1000:
        g[100:400] = 0
        for c in range(3):
            g[2000 + 500 * c:2400 + 500 * c] = g[1000:1400]
        for c in range(12):
            g[8000 + 200 * c:8120 + 200 * c] = g[7000:7120]
    ix = hp.Index.build(g, 16).to_device()
    ix.expand()
    if kmer:
        ix.kmer_table(kmer)
    o = fo.Oracle(g, ratio=16)
    reads, bounds = [], []
    spots = [0, n] + ([1000, 1100, 2050, 7000, 8010, 150, 50_000] if n > 1000 else [20])
    for L in (3, 4, 7, 15, 28, 29, 30, 31, 32, 45, 64, 65, 100, 255, 256, 257, 400):
        for p in spots:
            p = min(p, max(n - L, 0))
            w = g[p:p + L].copy()
            for kind in range(5):
                v = w.copy()
                e = int(rng.integers(0, len(v)))
                if kind == 1:
                    v[e] = (v[e] + 1) % 4
                elif kind == 2:
                    v = np.delete(v, e)
                elif kind == 3:
                    v = np.insert(v, e, rng.integers(0, 4))
                elif kind == 4:
                    v[e] = 4
                if rng.random() < 0.5:
                    v = synth.revcomp(v)
                pre, post = rng.integers(0, 4, rng.integers(0, 18)), rng.integers(0, 4, 5)
                reads.append(np.concatenate([pre, v, post]).astype(np.uint8))
                bounds.append((len(pre), len(pre) + len(v) - 1))
    offs = np.concatenate([[0], np.cumsum([len(r) for r in reads])]).astype(np.uint64)
    batch = hp.ReadBatch(np.concatenate(reads), offs)
    try:
        for mode, cap in ((hp.MODE_EDIT, 40), (hp.MODE_MISMATCH, 40), (hp.MODE_EDIT, 2)):
            counts, hits = hp.search1_vector_batch(ix, batch, cap=cap, mode=mode,
                                                   bounds=np.array(bounds, np.int16))
            for i, W in enumerate(reads):
                for s in (0, 1):
                    m, h = o.search1_vector(s, W, *bounds[i], cap=cap,
                                            mismatch_only=mode == hp.MODE_MISMATCH)[:2]
                    assert int(counts[i, s]) == m, (i, s, bounds[i])
                    assert fo.hits_equal(hits[i, s, :min(m, cap)], h), (i, s, bounds[i])
    finally:
        batch.free()
        ix.close()


@pytest.mark.gpu
@pytest.mark.parametrize("kmer", [0, 9])
def test_gpu_vector_helper_many_copies(gpu_engine, kmer):
    """Windows of 1200 exact copies (a half's interval is given up early), with
    and without one error, against the oracle."""
    hp = gpu_engine
    rng = np.random.default_rng(91)
    g = rng.integers(0, 4, 200_000).astype(np.uint8)
    unit = rng.integers(0, 4, 130).astype(np.uint8)
    for i in range(1200):
        g[50 + 140 * i:180 + 140 * i] = unit
    ix = hp.Index.build(g, 16).to_device()
    ix.expand()
    if kmer:
        ix.kmer_table(kmer)
    o = fo.Oracle(bwts=(*ix.bwt(0), *ix.bwt(1)), ratio=16)
    reads = []
    for L in (31, 40, 60, 120, 130):
        for e in (-1, 0, L // 2 - 1, L // 2, L - 1):
            w = unit[:L].copy()
            if e >= 0:
                w[e] = (w[e] + 1) % 4
            reads += [w, synth.revcomp(w)]
    offs = np.concatenate([[0], np.cumsum([len(r) for r in reads])]).astype(np.uint64)
    batch = hp.ReadBatch(np.concatenate(reads).astype(np.uint8), offs)
    try:
        counts, hits = hp.search1_vector_batch(ix, batch, cap=30, mode=hp.MODE_EDIT)
        for i, W in enumerate(reads):
            for s in (0, 1):
                m, h = o.search1_vector(s, W, 0, len(W) - 1, cap=30, mismatch_only=False)[:2]
                assert int(counts[i, s]) == m, (i, s)
                assert fo.hits_equal(hits[i, s, :min(m, 30)], h), (i, s)
    finally:
        batch.free()
        ix.close()
