"""The row contexts of an expanded index and the memory they take: what a program
allocates after fmi_index_expand fits as if there were none (the k-mer tables,
also where other memory ran short meanwhile), they can be given up, and the
searches answer alike with and without them, record for record the oracle's."""
import ctypes as C

import numpy as np
import pytest

import fmoracle as fo
from hpgfm import synth

pytestmark = pytest.mark.gpu
MB = 1 << 20
TABLE15 = 16 * (4 ** 15 + 4 ** 11)


def fill(hp, leave):
    """Device memory taken until about `leave` bytes are free."""
    free, _ = hp.mem_info()
    return hp.DeviceBuffer(free - leave)


def held(ix):
    """Whether the index has contexts: 8 bytes per base beside 16.25."""
    return ix.layout_bytes()["sa_isa_text"] > 20 * ix.n


@pytest.fixture(scope="module")
def text():
    return np.random.default_rng(501).integers(0, 4, 100_000_000).astype(np.uint8)


@pytest.mark.parametrize("room,kept", [(TABLE15 + 2 * 800 * MB + 200 * MB, True),
                                       (TABLE15 + 800 * MB, False)])
def test_contexts_leave_room_for_the_largest_table(gpu_engine, text, room, kept):
    hp = gpu_engine
    ix = hp.Index.build_gpu(text, 16)
    full = 16 * len(text) + len(text) // 4
    block = fill(hp, full + room)
    try:
        ix.expand()
        assert held(ix) == kept
        ix.kmer_table(15)
        assert ix.layout_bytes()["kmer_tables"] == TABLE15
        ix.kmer_table(0)
    finally:
        block.free()
        ix.close()


def test_contexts_give_way_to_a_table(gpu_engine, text):
    hp = gpu_engine
    ix = hp.Index.build_gpu(text, 16).expand()
    assert held(ix)
    blocks = [fill(hp, 1 << 30)]
    try:
        for _ in range(64):                          # what is free and not reported so
            blocks.append(hp.DeviceBuffer(128 * MB))
    except hp.FmiError:
        pass
    try:
        ix.kmer_table(12)                            # 0.27 GB
        assert not held(ix) and ix.layout_bytes()["kmer_tables"] == 16 * (4 ** 12 + 4 ** 8)
    finally:
        for b in blocks:
            b.free()
        ix.close()


def test_failed_allocation_leaves_no_error(gpu_engine):
    hp = gpu_engine
    g = np.random.default_rng(504).integers(0, 4, 5000).astype(np.uint8)
    ix = hp.Index.build(g, 16).to_device()
    batch = hp.ReadBatch(g[:100], np.array([0, 100], np.uint64))
    with pytest.raises(hp.FmiError):
        hp.DeviceBuffer(1 << 60)
    counts, _ = hp.search1_batch(ix, batch, cap=4)   # its launch's check saw that failure
    assert counts[0, 0] >= 1
    batch.free()
    ix.close()


def test_inexact_seeds_in_little_memory(gpu_engine):
    """600 K windows with 200 MB free: the lanes' record lists (312 MB with their
    intervals) do not fit, the intervals (88 MB) do, and the regions are the
    same."""
    hp = gpu_engine
    rng = np.random.default_rng(503)
    g = rng.integers(0, 4, 200_000).astype(np.uint8)
    ix = hp.Index.build(g, 16)
    ix.set_karyotype(np.ones(1, np.uint64), np.array([len(g)], np.uint64))
    ix.to_device().expand()
    ix.kmer_table(10)
    n, nwin = 100_000, 600_000
    at = rng.integers(0, len(g) - 108, n)
    batch = hp.ReadBatch(g[at[:, None] + np.arange(108)].reshape(-1), np.arange(n + 1, dtype=np.uint64) * 108)
    bufs = [hp.DeviceBuffer(b) for b in (2 * nwin * 48, 2 * nwin * 4, 2 * nwin)]
    got, out, blocks = C.c_uint64(), [], []

    def call():
        hp.check(hp.lib().fmi_map_inexact_seeds_batch(ix.h, batch.d_reads.ptr, batch.d_offsets.ptr, n, 18,
                                                      16, 64, 1, nwin, bufs[0].ptr, bufs[1].ptr,
                                                      bufs[2].ptr, C.byref(got), None))
        out.append([b.download(np.uint8, b.nbytes) for b in bufs])

    try:
        call()
        blocks = [fill(hp, 1 << 30)]
        try:
            for _ in range(256):
                blocks.append(hp.DeviceBuffer(40 * MB))
        except hp.FmiError:
            pass
        for b in blocks[-5:]:
            b.free()
        call()
        assert got.value == nwin and np.array_equal(out[0][1], out[1][1])
        assert np.array_equal(out[0][2], out[1][2])
        kept = out[0][1].view(np.uint32) > 0
        assert kept.sum() > nwin and np.array_equal(out[0][0].reshape(-1, 48)[kept],
                                                    out[1][0].reshape(-1, 48)[kept])
    finally:
        for b in blocks + bufs:
            b.free()
        batch.free()
        ix.close()


def test_dropped_contexts(gpu_engine):
    hp = gpu_engine
    g = np.random.default_rng(502).integers(0, 4, 50_000).astype(np.uint8)
    ix = hp.Index.build(g, 16).to_device()
    ix.drop_contexts()                               # none yet
    ix.expand()
    before = ix.device_bytes
    assert held(ix)
    ix.drop_contexts()
    assert not held(ix) and before - ix.device_bytes >= 8 * ix.n
    ix.drop_contexts()
    ix.expand()                                      # expanded already: stays as it is
    assert not held(ix)
    ix.close()


@pytest.fixture(scope="module", params=[0, 7, 11])
def without(gpu_engine, request):
    """A text with 2 to 1200 copies, an expanded index of it without contexts, and
    reads of every length that a launch parts them at."""
    hp = gpu_engine
    rng = np.random.default_rng(511)
    g = rng.integers(0, 4, 600_000).astype(np.uint8)
    at, spots = 1000, [0]
    for count in (2, 4, 5, 33, 64, 65, 1200):
        unit = rng.integers(0, 4, 280).astype(np.uint8)
        spots.append(at)
        for _ in range(count):
            g[at:at + 280] = unit
            if rng.random() < 0.2:
                g[at + int(rng.integers(0, 280))] ^= 1
            at += 300
    g[at:at + 400] = 3
    spots += [at, at + 350, len(g) - 300]
    reads = []
    for L in (3, 18, 29, 30, 31, 32, 33, 60, 100, 255, 256, 257, 270):
        for p in spots:
            for kind in range(3):
                w = g[p:p + L].copy()
                e = int(rng.integers(0, L))
                if kind == 1:
                    w[e] = (w[e] + 1) % 4
                elif kind == 2:
                    w = np.delete(w, e) if rng.random() < 0.5 else np.insert(w, e, rng.integers(0, 5))
                reads.append(synth.revcomp(w) if rng.random() < 0.5 else w.astype(np.uint8))
    offs = np.concatenate([[0], np.cumsum([len(r) for r in reads])]).astype(np.uint64)
    koff, kstart = np.array([0, 300_000, len(g)], np.uint64), np.ones(2, np.uint64)
    ix = hp.Index.build(g, 16)
    ix.set_karyotype(kstart, np.diff(koff))
    ix.to_device()
    o = fo.Oracle(bwts=(*ix.bwt(0), *ix.bwt(1)), ratio=16)
    ix.expand().drop_contexts()
    if request.param:
        ix.kmer_table(request.param)
    batch = hp.ReadBatch(np.concatenate(reads).astype(np.uint8), offs)
    yield hp, ix, o, reads, offs, batch, koff, kstart
    batch.free()
    ix.close()


def test_search1_without(without):
    hp, ix, o, reads, offs, batch, _, _ = without
    flat = np.concatenate(reads).astype(np.uint8)
    for mode in (hp.MODE_EDIT, hp.MODE_MISMATCH):
        _, oc, oh = o.search1_batch(flat, offs, cap=12, mismatch_only=mode == hp.MODE_MISMATCH)
        oc, oh = oc.reshape(-1, 2), oh.reshape(-1, 2, 12)
        counts, hits = hp.search1_batch(ix, batch, cap=12, mode=mode)
        assert np.array_equal(counts, oc)
        for i in range(batch.nreads):
            for s in (0, 1):
                c = min(int(oc[i, s]), 12)
                assert fo.hits_equal(hits[i, s, :c], oh[i, s, :c]), (mode, i, s)


def test_vector_without(without):
    hp, ix, o, reads, _, batch, _, _ = without
    counts, hits = hp.search1_vector_batch(ix, batch, cap=30, mode=hp.MODE_EDIT)
    for i, W in enumerate(reads):
        for s in (0, 1):
            m, h = o.search1_vector(s, W, 0, len(W) - 1, cap=30, mismatch_only=False)[:2]
            assert int(counts[i, s]) == m, (i, s)
            assert fo.hits_equal(hits[i, s, :min(m, 30)], h), (i, s)


def test_map_without(without):
    hp, ix, o, reads, _, batch, koff, kstart = without
    for filt in (3, 70):
        st, cnt, recs = hp.map_reads_batch(ix, batch, filt, 8)
        for i, W in enumerate(reads):
            ost, orecs, ototal = o.map_read(W, filt, koff, kstart, read=i, cap=8)
            assert (int(st[i]), int(cnt[i])) == (ost, ototal), (filt, i)
            m = min(ototal, 8)
            for key in ("position", "chromosome", "read", "strand", "secondary", "cigar_len"):
                assert np.array_equal(recs[i, :m][key], orecs[key]), (filt, i, key)


def test_seeds_without(without):
    hp, ix, o, reads, _, batch, koff, kstart = without
    for seed_len in (11, 18, 33):
        want = []
        for i, W in enumerate(reads):
            if len(W) >= seed_len:
                regs = o.seed_map(W, seed_len, 4, 500, koff, kstart)[0].copy()
                regs["read"] = i
                want.append(regs)
        want = np.concatenate(want)
        _, nr, regs, _ = hp.seed_map_batch(ix, batch, seed_len, 4, 500, with_info=False)
        assert nr == len(want) and regs.tobytes() == want.tobytes()


def test_inexact_without(without):
    hp, ix, o, reads, _, batch, koff, kstart = without
    short = [i for i, r in enumerate(reads) if len(r) <= 100]
    for seed_size, min_seed in ((18, 5), (29, 16)):
        res = hp.map_inexact_seeds_batch(ix, batch, seed_size, min_seed, 256, 48)
        for i in short:
            want = o.map_inexact_seeds(reads[i], seed_size, min_seed, koff, kstart, read=i,
                                       rec_cap=256, region_cap=48)
            w0 = int(res.window_base[i])
            for t, (regs, st) in enumerate(want):
                w, s = w0 + t // 2, t % 2
                assert int(res.status[w, s]) == st, (seed_size, i, t)
                assert res.regions(w, s).tobytes() == regs.tobytes(), (seed_size, i, t)
