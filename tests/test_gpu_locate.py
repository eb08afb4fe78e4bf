"""Row location and position resolution at the sizes where their work is
shared out differently: fewer intervals than a wavefront, a wavefront's
edges, capacities around 64, intervals of no row, one row and thousands, few
intervals (several wavefronts share one set) and many."""
import numpy as np
import pytest

from hpgfm import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def index(gpu_engine):
    g, _, _ = synth.genome(60_000, seed=301, repeat_frac=0.4, fam_len=(100, 800),
                           divergence=(0.0, 0.03))
    ix = gpu_engine.Index.build(g, 16)
    ix.set_karyotype(np.ones(3, np.uint64), np.array([10_000, 20_000, 30_000], np.uint64))
    ix.to_device()
    compact = gpu_engine.Index.build(g, 16).to_device()
    ix.expand()
    yield gpu_engine, g, ix, compact, [ix.full_arrays(d) for d in (0, 1)]
    ix.close()
    compact.close()


@pytest.mark.parametrize("cap", [1, 2, 63, 64, 65, 3000])
@pytest.mark.parametrize("count", [1, 63, 64, 65, 257, 20_000])
def test_locate_shares(index, count, cap):
    hp, g, ix, compact, full = index
    if count * cap > 2_000_000:
        count = 2_000_000 // cap
    rng = np.random.default_rng(302)
    n = ix.n
    k = rng.integers(0, n + 1, count)
    rows = rng.choice([0, 1, 1, 1, 2, 5, 64, 700, 5000], count)
    l = np.minimum(k + rows - 1, n)
    k[-1], l[-1] = (0, n) if cap > 64 else (5, 2)
    if count > 3:
        k[0], l[0] = -1, 4                           # rows outside the index: none
        k[1], l[1] = n, n + 1
    for dsel in (0, 1):
        sa = full[dsel][0].astype(np.uint64)
        for one in (ix, compact):
            pos, nrows = hp.locate_batch(one, k, l, cap, forward=dsel)
            ok = (k >= 0) & (l <= n) & (k <= l)
            want = np.where(ok, np.minimum(l - k + 1, cap), 0)
            assert np.array_equal(nrows, want)
            for i in range(count):
                m = int(want[i])
                assert np.array_equal(pos[i, :m], sa[k[i]:k[i] + m]), (dsel, i)


@pytest.mark.parametrize("row_cap", [1, 3, 64, 100])
@pytest.mark.parametrize("nreads,cap", [(1, 40), (33, 3), (5000, 3)])
def test_resolve_shares(index, nreads, cap, row_cap):
    hp, g, ix, compact, full = index
    reads, offs, _ = synth.reads(g, nreads, seed=303, sub_rate=0.02,
                                 lengths=np.random.default_rng(304).integers(15, 80, nreads))
    reads[:15] = g[30_000:30_015]
    batch = hp.ReadBatch(reads, offs)
    out = hp.Search1Output(nreads, cap)
    hp.search1_launch(ix, batch, out, mode=hp.MODE_EDIT)
    counts = out.counts().reshape(nreads, 2)
    hits = out.hits()
    koff = np.array([0, 10_000, 30_000, 60_000])
    for text_rule in (False, True):
        chrom, coord = hp.resolve_hits(ix, batch, out, row_cap, text_rule=text_rule)
        for i in range(nreads):
            for s in (0, 1):
                for h in range(min(int(counts[i, s]), cap)):
                    r = hits[i, s, h]
                    ln = int(r["end"]) - int(r["start"]) + 1 if text_rule else \
                        int(offs[i + 1] - offs[i])
                    if r["num_mismatches"]:
                        ln += {hp.DELETION: -1, hp.INSERTION: 1}.get(int(r["err_kind"]), 0)
                    fwd = (1 - int(r["dir"])) if s else int(r["dir"])
                    for j in range(row_cap):
                        row = int(r["k"]) + j
                        want = (-1, 0)
                        if row <= int(r["l"]):
                            sa = int(full[fwd][0][row])
                            key = (ix.n + 1 - sa - ln - 1 if fwd else sa) % (1 << 64)
                            c = int(np.searchsorted(koff[:3], key, side="right"))
                            if c and key + ln <= koff[c]:
                                want = (c - 1, 1 + key - koff[c - 1])
                        assert (int(chrom[i, s, h, j]), int(coord[i, s, h, j])) == want, (i, s, h, j)
    out.free()
    batch.free()
