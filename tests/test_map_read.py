"""Read-level 1-error mapping of __bwt_map_inexact_read (bwt.c:1890-2236):
only the error-free records of the vector-driven 1-error search become
alignments (bwt.c:2038), the running count of l - k over them is held to
filter_read_mappings (bwt.c:2145-2156), each SA row inside a contig gives an
alignment at its 0-based coordinate (bwt.c:2158-2166), and each strand's
alignments are deduplicated within 10 bp and handed over from last to first
with primary / secondary flags (bwt.c:2190-2233).

CPU: the oracle's restatement against a brute-force computation from the
text alone -- occurrences of the read and of its reverse complement found
by scanning, ordered as the suffix array orders them (suffixes of the text,
and of the reversed text for the - strand), the contig rule, the dedup rule
and the flags -- on a genome with tandem repeats (occurrences 1-7 bp apart),
far-apart copies, copies across contig ends, short reads, reads with N and
filters that are exceeded on either strand.
GPU: fmi_map_reads_batch against the oracle, record for record."""
import time

import numpy as np
import pytest

import fmoracle as fo
from hpgfm import synth

COMP = np.array([3, 2, 1, 0, 4], np.uint8)


def planted_genome(seed=7):
    rng = np.random.default_rng(seed)
    g = rng.integers(0, 4, 24_000).astype(np.uint8)
    unit7 = rng.integers(0, 4, 7).astype(np.uint8)
    g[3000:3210] = np.tile(unit7, 30)                    # period 7: occurrences 7 bp apart
    g[6000:6060] = 0                                     # A-run: occurrences 1 bp apart
    seg = rng.integers(0, 4, 60).astype(np.uint8)
    for p in (9000, 9500, 15000):                        # far-apart copies
        g[p:p + 60] = seg
    g[12000:12060] = COMP[seg][::-1]                     # a reverse-complement copy
    g[7995:8055] = seg                                   # spans the contig end at 8000
    near = rng.integers(0, 4, 40).astype(np.uint8)
    g[18000:18040] = near
    g[18006:18046] = near                                # overlapping copies 6 bp apart
    return g


def brute_force(text, W, filt, koff, kstart):
    """(status, [(position, chromosome, strand, secondary)]) from the text."""
    n = len(text)
    L = len(W)
    if L < 5:
        return 2, []
    tb = text.tobytes()
    rb = text[::-1].tobytes()
    out, status, tot = [], 0, 0
    if np.any(W > 3):
        return 0, []                      # an N never occurs in the index
    for strand in (0, 1):
        pat = W if strand == 0 else COMP[W][::-1]
        pb = pat.tobytes()
        occ = [p for p in range(n - L + 1) if tb[p:p + L] == pb]
        if not occ:
            continue
        tot += len(occ) - 1                   # l - k of the strand's exact record
        if tot > filt:
            status |= 1
            break
        if strand == 0:
            occ.sort(key=lambda p: tb[p:])                    # rows of the backward index
        else:
            occ.sort(key=lambda p: rb[n - p - L:])            # rows of the forward index
        tmp = []
        for p in occ:
            idx = int(np.searchsorted(koff, p, side="right"))   # upper bound
            if p + L <= koff[idx]:
                tmp.append((int(kstart[idx - 1] + p - koff[idx - 1]), idx - 1))
        keep = []
        for i, (pos, c) in enumerate(tmp):
            if not any(c == c2 and abs(pos - p2) < 10 for p2, c2 in tmp[:i]):
                keep.append((pos, c))
        for pos, c in reversed(keep):
            out.append((pos, c, strand, int(len(out) > 0)))
    return status, out


@pytest.fixture(scope="module")
def planted():
    g = planted_genome()
    lens = np.array([8000, 9000, 7000], np.uint64)
    kstart = np.array([0, 100, 0], np.uint64)
    koff = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint64)
    o = fo.Oracle(g, ratio=8)
    rng = np.random.default_rng(8)
    reads = [g[3000:3030], g[3010:3035], g[6000:6020], g[6005:6045], g[9000:9060],
             g[9010:9050], g[12000:12060], COMP[g[9000:9060]][::-1], g[7990:8030],
             g[18000:18040], g[18003:18043], g[100:104], g[200:203], g[300:305]]
    w = g[5000:5050].copy()
    w[20] = 4
    reads.append(w)
    for _ in range(60):
        p = int(rng.integers(0, len(g) - 80))
        L = int(rng.integers(5, 80))
        r = g[p:p + L].copy()
        if rng.random() < 0.5:
            r = COMP[r][::-1]
        reads.append(r)
    return g, o, koff, kstart, reads


@pytest.mark.parametrize("filt", [1, 3, 10, 200])
def test_oracle_map_read_vs_brute_force(planted, filt):
    g, o, koff, kstart, reads = planted
    seen_exceeded = seen_dedup = 0
    for i, W in enumerate(reads):
        st, recs, total = o.map_read(W, filt, koff, kstart, read=i)
        want_st, want = brute_force(g, W, filt, koff, kstart)
        assert st == want_st, (i, filt)
        assert total == len(want) == len(recs), (i, filt)
        got = [(int(r["position"]), int(r["chromosome"]), int(r["strand"]), int(r["secondary"]))
               for r in recs]
        assert got == want, (i, filt)
        assert np.all(recs["cigar_len"] == len(W)) and np.all(recs["read"] == i)
        seen_exceeded += st & 1
        seen_dedup += int(len(W) >= 5 and len(want) < sum(
            (g[p:p + len(W)].tobytes() == W.tobytes()) for p in range(len(g) - len(W) + 1)))
    if filt == 3:
        assert seen_exceeded > 0
    if filt == 200:
        assert seen_dedup > 0


def test_oracle_map_read_strand_order_and_flags(planted):
    """A read with copies on both strands: + strand alignments first, in the
    reverse of the row order; only the very first is primary."""
    g, o, koff, kstart, _ = planted
    W = g[9000:9060]
    st, recs, _ = o.map_read(W, 100, koff, kstart)
    assert st == 0
    assert list(recs["strand"]) == sorted(recs["strand"])
    assert recs["secondary"][0] == 0 and np.all(recs["secondary"][1:] == 1)
    assert {int(p) for p in recs["position"][recs["strand"] == 1]} == {12000 - 8000 + 100}


@pytest.mark.gpu
@pytest.mark.parametrize("expanded", [False, True])
def test_gpu_map_reads_vs_oracle(gpu_engine, planted, expanded):
    hp = gpu_engine
    g, o, koff, kstart, reads = planted
    lens = np.array([8000, 9000, 7000], np.uint64)
    ix = hp.Index.build(g, 8)
    ix.set_karyotype(kstart, kstart + lens - 1)
    ix.to_device()
    if expanded:
        ix.expand()
        ix.kmer_table(6)
    g2, _, _ = synth.genome(24_000, seed=9, repeat_frac=0.3, fam_len=(200, 1500))
    more, moffs, _ = synth.reads(g, 2000, seed=10, sub_rate=0.01, n_rate=0.002,
                                 lengths=np.random.default_rng(11).integers(3, 150, 2000))
    all_reads = reads + [more[int(moffs[i]):int(moffs[i + 1])] for i in range(2000)]
    offs = np.concatenate([[0], np.cumsum([len(r) for r in all_reads])]).astype(np.uint64)
    flat = np.concatenate(all_reads).astype(np.uint8)
    batch = hp.ReadBatch(flat, offs)
    try:
        for filt, cap in ((3, 4), (50, 16), (500, 64)):
            st, cnt, recs = hp.map_reads_batch(ix, batch, filt, cap)
            for i, W in enumerate(all_reads):
                ost, orecs, ototal = o.map_read(W, filt, koff, kstart, read=i, cap=cap)
                assert int(st[i]) == ost, (filt, i)
                assert int(cnt[i]) == ototal, (filt, i)
                m = min(ototal, cap)
                got = recs[i, :m]
                for key in ("position", "chromosome", "read", "strand", "secondary", "cigar_len"):
                    assert np.array_equal(got[key], orecs[key]), (filt, i, key)
    finally:
        batch.free()
        ix.close()


@pytest.mark.gpu
@pytest.mark.parametrize("stage", ["compact", "table", "expanded", "expanded + table"])
def test_map_read_lengths(gpu_engine, stage):
    """Reads around the limits of the two launches -- 256 bases staged in LDS
    and longer, a k-mer's length, 5 and 1000 bases -- that occur once, several
    times (also across the text's start and end) or not at all, against the
    oracle."""
    hp = gpu_engine
    rng = np.random.default_rng(12)
    g = rng.integers(0, 4, 30_000).astype(np.uint8)
    g[20_000:21_500] = g[1_000:2_500]                # two copies of 1500 bases
    lens = [4, 5, 7, 8, 9, 31, 32, 33, 63, 64, 65, 255, 256, 257, 272, 999, 1000]
    reads = []
    for L in lens:
        for p in (0, 1_100, 20_100, 5_000, len(g) - L):
            r = g[p:p + L].copy()
            reads += [r, COMP[r][::-1].copy()]
            bad = r.copy()
            bad[L // 2] = 4
            reads += [bad, rng.integers(0, 4, L).astype(np.uint8)]
    koff = np.array([0, 9_000, 30_000], np.uint64)
    kstart = np.ones(2, np.uint64)
    ix = hp.Index.build(g, 16)
    ix.set_karyotype(kstart, np.array([9_000, 21_000], np.uint64))
    ix.to_device()
    o = fo.Oracle(bwts=(*ix.bwt(0), *ix.bwt(1)), ratio=16)
    if "expanded" in stage:
        ix.expand()
    if "table" in stage:
        ix.kmer_table(8)
    offs = np.concatenate([[0], np.cumsum([len(r) for r in reads])]).astype(np.uint64)
    batch = hp.ReadBatch(np.concatenate(reads).astype(np.uint8), offs)
    try:
        for filt, cap in ((3, 2), (50, 8)):
            st, cnt, recs = hp.map_reads_batch(ix, batch, filt, cap)
            for i, W in enumerate(reads):
                ost, orecs, ototal = o.map_read(W, filt, koff, kstart, read=i, cap=cap)
                assert (int(st[i]), int(cnt[i])) == (ost, ototal), (filt, i, len(W))
                m = min(ototal, cap)
                for key in ("position", "chromosome", "read", "strand", "secondary", "cigar_len"):
                    assert np.array_equal(recs[i, :m][key], orecs[key]), (filt, i, key)
    finally:
        batch.free()
        ix.close()


@pytest.mark.gpu
@pytest.mark.parametrize("table", [0, 10])
def test_map_read_many_rows(gpu_engine, table):
    """Reads of 5, 60, 70 and 1200 copies, forward and reverse, at filters below,
    at and above their rows (a read over the filter ends where its rows are
    first known, one with more rows than that launch holds in the second),
    against the oracle; and a batch of reads over the filter costs their search,
    at most 1.6 times the exact search of both strands: 0.96 measured, 2.2 where
    the second launch repeats it."""
    hp = gpu_engine
    rng = np.random.default_rng(21)
    g = rng.integers(0, 4, 900_000).astype(np.uint8)
    at, reads = 100, []
    for count in (5, 60, 70, 1200):
        unit = rng.integers(0, 4, 300).astype(np.uint8)
        for _ in range(count):
            g[at:at + 300] = unit
            at += 320
        for L in (40, 100, 256, 280):
            reads += [unit[3:3 + L].copy(), COMP[unit[2:2 + L]][::-1].copy()]
    koff, kstart = np.array([0, len(g)], np.uint64), np.ones(1, np.uint64)
    ix = hp.Index.build(g, 16)
    ix.set_karyotype(kstart, np.array([len(g)], np.uint64))
    ix.to_device()
    o = fo.Oracle(bwts=(*ix.bwt(0), *ix.bwt(1)), ratio=16)
    ix.expand()
    if table:
        ix.kmer_table(table)
    offs = np.concatenate([[0], np.cumsum([len(r) for r in reads])]).astype(np.uint64)
    batch = hp.ReadBatch(np.concatenate(reads).astype(np.uint8), offs)
    n = 100_000
    rep = hp.ReadBatch(np.tile(reads[-6], n), np.arange(n + 1, dtype=np.uint64) * len(reads[-6]))
    try:
        for filt in (1, 3, 4, 58, 59, 60, 69, 1198, 1199, 1500):
            st, cnt, recs = hp.map_reads_batch(ix, batch, filt, 8)
            for i, W in enumerate(reads):
                ost, orecs, ototal = o.map_read(W, filt, koff, kstart, read=i, cap=8)
                assert (int(st[i]), int(cnt[i])) == (ost, ototal), (filt, i)
                m = min(ototal, 8)
                for key in ("position", "chromosome", "read", "strand", "secondary", "cigar_len"):
                    assert np.array_equal(recs[i, :m][key], orecs[key]), (filt, i, key)
        assert len(reads[-6]) == 100
        L, d = hp.lib(), rep
        bufs = [hp.DeviceBuffer(b) for b in (24 * n, 4 * n, n, 32 * n)]

        def mapped():
            hp.check(L.fmi_map_reads_batch(ix.h, d.d_reads.ptr, d.d_offsets.ptr, n, 50, 1,
                                           bufs[0].ptr, bufs[1].ptr, bufs[2].ptr, None))

        def exact():
            for t, view in ((0, hp.VIEW_BACKWARD), (1, hp.VIEW_BACKWARD_REV)):
                hp.check(L.fmi_exact_batch(ix.h, view, t, d.d_reads.ptr, d.d_offsets.ptr, n,
                                           bufs[3].ptr, None, None))

        took = []
        for f in (mapped, exact):
            best = 1.0
            for _ in range(8):
                hp.sync()
                t0 = time.perf_counter()
                f()
                hp.sync()
                best = min(best, time.perf_counter() - t0)
            took.append(best)
        for b in bufs:
            b.free()
        print(took)
        assert took[0] < 1.6 * took[1], took
    finally:
        batch.free()
        rep.free()
        ix.close()
