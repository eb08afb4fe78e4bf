"""Exact seed mapping, bwt_map_exact_seed (bwt.c:1200-1294).

CPU: the oracle's restatement against closed forms -- a seed cut from a
known position of a known contig yields a region at that contig's 1-based
coordinate on the right strand, with the one-short length of bwt.c:1214;
occurrences crossing a contig end yield none; the cumulative filter skips
exactly the strands the reference's running `int` count exceeds.
GPU: fmi_seed_map_batch equals the oracle region for region, in order."""
import ctypes as C
import time

import numpy as np
import pytest

import fmoracle as fo
from hpgfm import synth


def karyotype(n, cuts):
    starts = np.concatenate([[0], cuts]).astype(np.uint64)
    lens = np.diff(np.concatenate([starts, [n]])).astype(np.uint64)
    koff = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint64)
    kstart = np.full(len(lens), 1000, np.uint64)          # contigs start at coordinate 1000
    return koff, kstart


@pytest.fixture(scope="module")
def seeded():
    g, _, _ = synth.genome(30_000, seed=17)
    o = fo.Oracle(g, ratio=8)
    koff, kstart = karyotype(len(g), [9000, 20000])
    return g, o, koff, kstart


def test_seed_regions_closed_form(seeded):
    g, o, koff, kstart = seeded
    rng = np.random.default_rng(3)
    L, sl, st = 60, 18, 5
    checked = 0
    for _ in range(200):
        p = int(rng.integers(0, len(g) - L))
        for strand in (0, 1):
            W = g[p:p + L].copy() if strand == 0 else synth.revcomp(g[p:p + L])
            regs, info = o.seed_map(W, sl, st, 1000, koff, kstart)
            for q in range(len(info)):
                s0 = q * st
                tpos = p + s0 if strand == 0 else p + (L - s0 - sl)   # text position of the seed
                c = int(np.searchsorted(koff, tpos, side="right")) - 1
                fits = tpos + (sl - 1) <= int(koff[c + 1])
                mine = regs[(regs["seed_id"] == q) & (regs["strand"] == strand)]
                want_start = int(kstart[c]) + tpos - int(koff[c]) + 1
                hit = mine[(mine["valid"] == 1) & (mine["start"] == want_start)]
                if fits:
                    assert len(hit) == 1, (p, strand, q)
                    assert int(hit[0]["end"]) == want_start + sl - 1
                    assert int(hit[0]["chrom_idx"]) == c + 1
                    exp_ss = s0 if strand == 0 else L - (s0 + sl - 1) - 1
                    assert int(hit[0]["seq_start"]) == exp_ss
                    checked += 1
                else:
                    assert len(hit) == 0
    assert checked > 1000


def test_seed_filter_is_cumulative(seeded):
    g, o, koff, kstart = seeded
    # a seed made of one repeated base occurs many times on one strand
    W = np.zeros(18, np.uint8)
    regs, info = o.seed_map(W, 6, 1, 1 << 30, koff, kstart)
    kp, lp, km, lm = (int(x) for x in info[0, :4])
    cp, cm = lp - kp + 1, lm - km + 1
    assert cp > 2 and cm >= 1
    for filt in (cp - 1, cp, cp + cm - 1, cp + cm):
        _, inf = o.seed_map(W, 6, 1, filt, koff, kstart)
        rows_p, rows_m = int(inf[0, 4]), int(inf[0, 5])
        assert rows_p == (cp if cp <= filt else 0)
        assert rows_m == (cm if cp + cm <= filt else 0)


@pytest.mark.gpu
def test_seed_map_gpu_vs_oracle(gpu_engine):
    hp = gpu_engine
    g, _, _ = synth.genome(500_000, seed=23, repeat_frac=0.3, fam_len=(300, 2000),
                           divergence=(0.0, 0.05), n_frac=0.001, n_run=(5, 50))
    gi = synth.replace_n(g, seed=1)
    ix = hp.Index.build(gi, 8)
    cuts = [100_000, 250_000, 400_000]
    koff, kstart = karyotype(len(gi), cuts)
    ix.set_karyotype(kstart, kstart + np.diff(koff) - 1)
    ix.to_device()
    o = fo.Oracle(gi, ratio=8)
    lengths = np.random.default_rng(24).integers(0, 251, 1500)
    reads, offs, _ = synth.reads(g, 1500, seed=25, sub_rate=0.01, n_rate=0.002, lengths=lengths)
    batch = hp.ReadBatch(reads, offs)
    # seeds of up to 32 bases are searched from registers, longer ones from
    # the read's bytes; then the same on the expanded index with an 8-mer
    # table (the first 8 steps of each orientation from one table read)
    cases = ((18, 5, 1000), (12, 3, 7), (25, 25, 1), (32, 7, 1000), (33, 11, 1000), (40, 40, 50))
    for form in ("compact", "kmer8"):
        if form == "kmer8":
            ix.expand()
            ix.kmer_table(8)
        for sl, st, filt in cases:
            ns, nr, regs, info = hp.seed_map_batch(ix, batch, sl, st, filt)
            want, wi = [], []
            for i in range(batch.nreads):
                W = reads[offs[i]:offs[i + 1]]
                r, inf = o.seed_map(W, sl, st, filt, koff, kstart, read=i)
                want.append(r)
                wi.append(inf)
            want = np.concatenate(want)
            wi = np.concatenate([x for x in wi if len(x)]) if any(len(x) for x in wi) else np.zeros((0, 6))
            assert ns == len(wi) and nr == len(want), (form, sl)
            for key in ("k_plus", "l_plus", "k_minus", "l_minus"):
                assert np.array_equal(info[key], wi[:, ("k_plus", "l_plus", "k_minus", "l_minus").index(key)]), \
                    (form, sl, key)
            assert np.array_equal(info["rows_plus"], wi[:, 4]) and np.array_equal(info["rows_minus"], wi[:, 5])
            for key in want.dtype.names:
                assert np.array_equal(regs[key], want[key]), (form, sl, st, filt, key)
    # a capacity below the row count stores the first rows and reports all
    ns, nr, regs, _ = hp.seed_map_batch(ix, batch, 18, 5, 1000, region_cap=10, with_info=False)
    assert len(regs) == 10 and nr > 10
    batch.free()


@pytest.mark.gpu
@pytest.mark.parametrize("kmer,seed_len,stride", [(4, 4, 1), (8, 8, 3), (8, 9, 5), (8, 24, 7),
                                                  (8, 25, 1), (8, 32, 5), (12, 18, 5), (15, 31, 2)])
def test_gpu_seed_map_by_context(gpu_engine, kmer, seed_len, stride):
    """The expanded index with a table and no intervals asked for (row
    contexts), and the same call with them (occurrence blocks): equal to the
    oracle, for seeds of a k-mer's length to 32 bases, on copies (more rows
    than one look takes), runs of one base and the text's ends, with N bases,
    a filter that skips strands, reads without a seed, and room for a part of
    the regions only."""
    hp = gpu_engine
    rng = np.random.default_rng(61)
    n = 40_000
    g = rng.integers(0, 4, n).astype(np.uint8)
    g[500:800] = 2
    for i in range(120):
        g[3000 + 50 * i:3034 + 50 * i] = g[3000:3034]
    koff, kstart = karyotype(n, [9_000, 20_000])
    ix = hp.Index.build(g, 16)
    ix.set_karyotype(kstart, kstart + np.diff(koff) - 1)
    ix.to_device()
    ix.expand()
    ix.kmer_table(kmer)
    o = fo.Oracle(g, ratio=8)
    reads = [g[:60], g[n - 60:], g[450:560], g[3000:3080], g[8_970:9_030], g[:3], g[:0], g[100:131]]
    more, moffs, _ = synth.reads(g, 150, seed=62, sub_rate=0.01, n_rate=0.004,
                                 lengths=rng.integers(0, 120, 150))
    reads += [more[int(moffs[i]):int(moffs[i + 1])] for i in range(150)]
    reads += [synth.revcomp(r) for r in reads[:6]]
    offs = np.concatenate([[0], np.cumsum([len(r) for r in reads])]).astype(np.uint64)
    batch = hp.ReadBatch(np.concatenate(reads), offs)
    try:
        for filt in (5, 1000):
            want, winfo = [], []
            for i, W in enumerate(reads):
                if len(W) < seed_len:
                    continue
                regs, info = o.seed_map(W, seed_len, stride, filt, koff, kstart)
                regs = regs.copy()
                regs["read"] = i
                want.append(regs)
                winfo.append(info)
            want, winfo = np.concatenate(want), np.concatenate(winfo)
            ns, nr, regs, _ = hp.seed_map_batch(ix, batch, seed_len, stride, filt, with_info=False)
            assert (ns, nr) == (len(winfo), len(want))
            assert regs.tobytes() == want.tobytes()
            ns, nr, regs, info = hp.seed_map_batch(ix, batch, seed_len, stride, filt)
            assert regs.tobytes() == want.tobytes()
            for c, key in enumerate(("k_plus", "l_plus", "k_minus", "l_minus", "rows_plus",
                                     "rows_minus")):
                assert np.array_equal(info[key], winfo[:, c]), key
            for cap in (1, 63, 64, 65, max(nr - 1, 1)):
                _, nr2, regs, _ = hp.seed_map_batch(ix, batch, seed_len, stride, filt,
                                                    region_cap=cap, with_info=False)
                assert nr2 == nr and regs.tobytes() == want[:cap].tobytes()
    finally:
        batch.free()
        ix.close()


@pytest.mark.gpu
@pytest.mark.parametrize("expanded", [False, True])
def test_gpu_seed_map_rows_of_few_seeds(gpu_engine, expanded):
    """Seeds whose rows are many more than a wavefront writes at a time -- a run
    of one base and 700 exact copies, among seeds of no row -- equal to the
    oracle, whole and at every edge of a tile of rows; and one seed of 300,000
    rows, which has to be the work of the whole device: 0.1 ms where it is, 4.4
    ms (30 on a compact index) where one wavefront writes them all."""
    hp = gpu_engine
    rng = np.random.default_rng(71)
    n = 700_000
    g = rng.integers(0, 4, n).astype(np.uint8)
    g[1000:1000 + 1500] = 2
    for i in range(700):
        g[10_000 + 60 * i:10_030 + 60 * i] = g[10_000:10_030]
    g[390_000:690_030] = 0
    g[389_999] = g[690_030] = 1
    koff, kstart = karyotype(n, [60_000])
    ix = hp.Index.build(g, 16)
    ix.set_karyotype(kstart, kstart + np.diff(koff) - 1)
    ix.to_device()
    if expanded:
        ix.expand()
        ix.kmer_table(9)
    o = fo.Oracle(g, ratio=8)
    reads = [np.full(33, 2, np.uint8), g[10_000:10_030]]
    reads += [rng.integers(0, 4, 1000).astype(np.uint8) for _ in range(4)]
    reads += [g[10_000:10_024], g[200_000:200_030], synth.revcomp(g[10_000:10_030])]
    offs = np.concatenate([[0], np.cumsum([len(r) for r in reads])]).astype(np.uint64)
    batch = hp.ReadBatch(np.concatenate(reads).astype(np.uint8), offs)
    want = []
    for i, W in enumerate(reads):
        regs, _ = o.seed_map(W, 18, 3, 1 << 30, koff, kstart)
        regs = regs.copy()
        regs["read"] = i
        want.append(regs)
    want = np.concatenate(want)
    one = hp.ReadBatch(np.zeros(20, np.uint8), np.array([0, 20], np.uint64))
    try:
        assert len(want) > 10_000
        for cap in (None, 1, 63, 64, 65, 511, 512, 513, len(want) - 1):
            _, nr, regs, _ = hp.seed_map_batch(ix, batch, 18, 3, 1 << 30, region_cap=cap,
                                               with_info=False)
            assert nr == len(want) and regs.tobytes() == want[:cap].tobytes()
        L, got = hp.lib(), (C.c_uint64(), C.c_uint64())
        rows = hp.DeviceBuffer(32 * 400_000)
        took = []
        for _ in range(5):
            t = time.perf_counter()
            hp.check(L.fmi_seed_map_batch(ix.h, one.d_reads.ptr, one.d_offsets.ptr, 1, 18, 5, 1 << 30,
                                          None, 0, rows.ptr, 400_000, C.byref(got[0]),
                                          C.byref(got[1]), None))
            took.append(time.perf_counter() - t)
        rows.free()
        assert got[1].value == 300_013 and min(took) < 1.5e-3, (got[1].value, took)
    finally:
        one.free()
        batch.free()
        ix.close()
