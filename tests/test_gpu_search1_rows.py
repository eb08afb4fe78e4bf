"""The 1-error search of an expanded index where its launches part the reads:
anchors of one to four rows (a thread per strand), five to 64 (a wavefront per
read), more (step by step), halves of 15 and 16 bases, reads of 256 and 257,
on copies of every such number, runs of one base and both ends of the text,
with N bases and one error anywhere, against the oracle record for record."""
import time

import numpy as np
import pytest

import fmoracle as fo
from hpgfm import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def copies():
    rng = np.random.default_rng(401)
    g = rng.integers(0, 4, 150_000).astype(np.uint8)
    at, spots = 1000, [0]
    for count in (2, 4, 5, 33, 64, 65, 100):
        unit = rng.integers(0, 4, 280).astype(np.uint8)
        spots.append(at)
        for _ in range(count):
            g[at:at + 280] = unit
            if rng.random() < 0.3:                   # most copies exact, some with a change
                g[at + int(rng.integers(0, 280))] ^= 1
            at += 300
    g[at:at + 400] = 3
    spots += [at, at + 350, len(g) - 400]
    reads = []
    for L in (0, 1, 2, 29, 30, 31, 32, 33, 60, 64, 65, 150, 255, 256, 257, 270):
        for p in spots + [len(g) - L]:
            w = g[p:p + L].copy()
            for kind in range(4):
                v = w.copy()
                if kind and L:
                    e = int(rng.integers(0, L))
                    if kind == 1:
                        v[e] = (v[e] + 1) % 4
                    elif kind == 2:
                        v = np.delete(v, e) if rng.random() < 0.5 else \
                            np.insert(v, e, rng.integers(0, 4))
                    else:
                        v[e] = 4
                reads.append(synth.revcomp(v) if rng.random() < 0.5 else v.astype(np.uint8))
    offs = np.concatenate([[0], np.cumsum([len(r) for r in reads])]).astype(np.uint64)
    return g, np.concatenate(reads).astype(np.uint8), offs, fo.Oracle(g, ratio=16)


@pytest.mark.parametrize("kmer", [0, 7, 11])
def test_search1_rows(gpu_engine, copies, kmer):
    hp = gpu_engine
    g, reads, offs, o = copies
    ix = hp.Index.build(g, 16).to_device()
    ix.expand()
    if kmer:
        ix.kmer_table(kmer)
    batch = hp.ReadBatch(reads, offs)
    try:
        for mode, cap in ((hp.MODE_EDIT, 24), (hp.MODE_MISMATCH, 24), (hp.MODE_EDIT, 1)):
            _, oc, oh = o.search1_batch(reads, offs, cap=cap,
                                        mismatch_only=mode == hp.MODE_MISMATCH)
            oc, oh = oc.reshape(-1, 2), oh.reshape(-1, 2, cap)
            for mask in (3, hp.STRAND_PLUS, hp.STRAND_MINUS):
                counts, hits = hp.search1_batch(ix, batch, cap=cap, mode=mode, strand_mask=mask)
                for s in (0, 1):
                    if not (mask >> s) & 1:
                        assert np.all(counts[:, s] == 0)
                        continue
                    assert np.array_equal(counts[:, s], oc[:, s])
                    for i in range(batch.nreads):
                        c = min(int(oc[i, s]), cap)
                        assert fo.hits_equal(hits[i, s, :c], oh[i, s, :c]), (mode, mask, i, s)
    finally:
        batch.free()
        ix.close()


@pytest.mark.parametrize("nreads", [131_072, 131_073])
def test_search1_rows_batch_size(gpu_engine, copies, nreads):
    """The last batch whose groups are all resident and the first past it
    (registers held for more waves): the same reads over and over have the
    records of the one batch that meets the oracle above."""
    hp = gpu_engine
    g, reads, offs, _ = copies
    ix = hp.Index.build(g, 16).to_device()
    ix.expand()
    ix.kmer_table(11)
    lens = np.diff(offs.astype(np.int64))
    m = len(lens)
    times = -(-nreads // m)
    many = np.concatenate([[0], np.cumsum(np.tile(lens, times)[:nreads])]).astype(np.uint64)
    few = hp.ReadBatch(reads, offs)
    batch = hp.ReadBatch(np.tile(reads, times)[:int(many[-1])], many)
    try:
        for mode in (hp.MODE_EDIT, hp.MODE_MISMATCH):
            wc, wh = hp.search1_batch(ix, few, cap=4, mode=mode)
            counts, hits = hp.search1_batch(ix, batch, cap=4, mode=mode)
            assert np.array_equal(counts, np.tile(wc, (times, 1))[:nreads])
            stored = np.minimum(wc, 4)[..., None] > np.arange(4)
            for t in range(times):
                part = hits[t * m:min((t + 1) * m, nreads)]
                keep = stored[:len(part)]
                assert part[keep].tobytes() == wh[:len(part)][keep].tobytes()
    finally:
        batch.free()
        few.free()
        ix.close()


@pytest.fixture(scope="module")
def satellite():
    """1200 exact copies of 300 bases (an anchor of them is given up early), 90 of
    300 (its rows are no wavefront's) and 40 (they are), and reads of them with
    reads longer than a slot and too short for an anchor in between."""
    rng = np.random.default_rng(411)
    g = rng.integers(0, 4, 1_500_000).astype(np.uint8)
    spots, at = [], 500
    for count in (1200, 90, 40):
        unit = rng.integers(0, 4, 300).astype(np.uint8)
        spots.append(at)
        for _ in range(count):
            g[at:at + 300] = unit
            at += 310
    assert at < len(g) - 1000
    return g, spots


def _batch(g, spots, lens, seed):
    rng = np.random.default_rng(seed)
    reads = []
    for L in lens:
        p = int(rng.choice(spots)) + int(rng.integers(0, max(301 - L, 1))) if rng.random() < 0.8 \
            else int(rng.integers(0, len(g) - L))
        w = g[p:p + L].copy()
        if L and rng.random() < 0.6:
            e = int(rng.integers(0, L))
            w[e] = (w[e] + 1) % 4
        reads.append(synth.revcomp(w) if rng.random() < 0.5 else w)
    offs = np.concatenate([[0], np.cumsum([len(r) for r in reads])]).astype(np.uint64)
    return np.concatenate(reads).astype(np.uint8), offs


@pytest.mark.parametrize("nreads", [1, 255, 256, 257, 700])
def test_search1_left_reads(gpu_engine, satellite, nreads):
    """Groups whose reads go on in all three lists, part full and over a group's
    edge: record for record the oracle's."""
    hp = gpu_engine
    g, spots = satellite
    ix = hp.Index.build_gpu(g, 16)
    ix.expand()
    ix.kmer_table(11)
    o = fo.Oracle(bwts=(*ix.bwt(0), *ix.bwt(1)), ratio=16)
    rng = np.random.default_rng(412)
    lens = rng.choice([0, 20, 31, 32, 60, 100, 150, 256, 257, 290], nreads)
    reads, offs = _batch(g, spots, lens, 413)
    batch = hp.ReadBatch(reads, offs)
    try:
        for mode in (hp.MODE_EDIT, hp.MODE_MISMATCH):
            _, oc, oh = o.search1_batch(reads, offs, cap=8, mismatch_only=mode == hp.MODE_MISMATCH)
            oc, oh = oc.reshape(-1, 2), oh.reshape(-1, 2, 8)
            counts, hits = hp.search1_batch(ix, batch, cap=8, mode=mode)
            assert np.array_equal(counts, oc)
            for i in range(nreads):
                for s in (0, 1):
                    c = min(int(oc[i, s]), 8)
                    assert fo.hits_equal(hits[i, s, :c], oh[i, s, :c]), (mode, i, s)
    finally:
        batch.free()
        ix.close()


@pytest.mark.parametrize("kind", ["satellite", "short"])
def test_search1_left_reads_cost(gpu_engine, satellite, kind):
    """Reads that the text kernels leave cost what the step-by-step search of
    them does (the same batch without staging never meets the text kernels), not
    a multiple of it: at most 1.25 times, where a wavefront for each read of too
    many rows made it 2.5 and a walk over the other kernel's reads 1.33."""
    hp = gpu_engine
    g, spots = satellite
    ix = hp.Index.build_gpu(g, 16)
    ix.expand()
    ix.kmer_table(13)
    n = 60_000
    reads, offs = _batch(g, spots[:1], np.full(500, {"satellite": 100, "short": 30}[kind]),
                         414)
    batch = hp.ReadBatch(np.tile(reads, n // 500),
                         np.arange(n + 1, dtype=np.uint64) * (offs[1] - offs[0]))
    out = hp.Search1Output(n, 4)
    took = {}
    try:
        for staging in (True, False, True, False):
            hp.set_staging(staging)
            for _ in range(6):
                hp.sync()
                t = time.perf_counter()
                hp.search1_launch(ix, batch, out)
                hp.sync()
                took[staging] = min(took.get(staging, 1.0), time.perf_counter() - t)
        print(kind, took)
        assert took[True] < 1.25 * took[False], took
    finally:
        hp.set_staging(True)
        out.free()
        batch.free()
        ix.close()
