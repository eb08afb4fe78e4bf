"""The 1-error search of an expanded index where its launches part the reads:
anchors of one to four rows (a thread per strand), five to 64 (a wavefront per
read), more (step by step), halves of 15 and 16 bases, reads of 256 and 257,
on copies of every such number, runs of one base and both ends of the text,
with N bases and one error anywhere, against the oracle record for record."""
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
