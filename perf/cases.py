"""The measured work of the engine: one call (or the short chain of calls that
belong together) through the C ABI of include/fmi.h, as an aligner's host code
makes it over reads resident in HBM.

A case names its path, the reference text it searches (its bases, whether the
index is expanded and the k-mer table it holds), the reads (number, lengths,
substitution and N rates) and the path's own options:

  search1   fmi_search1_batch, mismatch or edit records; with "resolve" the
            records' genome positions too (fmi_resolve_hits)
  exact     fmi_exact_batch + fmi_locate_hits on both strands
  search_k  fmi_search_k_batch, fragsize = len / 3 (two errors)
  vector    fmi_search1_vector_batch, edit records
  map       fmi_fastq_encode_batch + fmi_map_reads_batch (FASTQ text to
            alignments)
  seeds     fmi_seed_map_batch
  inexact   fmi_map_inexact_seeds_batch

The reference text of a size is always the same one, as a program's genome is,
and its index is built once and kept; the reads come from the seed.
"""
import ctypes as C
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "hpg-libs_amd"))

import hpgfm  # noqa: E402

MBP = 1_000_000


def _case(name, path, genome, reads, length, **more):
    c = dict(name=name, path=path, genome=genome, expand=True, kmer=_kmer_of(genome),
             reads=reads, length=length, sub=0.01, n_rate=0.0)
    c.update(more)
    return c


def _kmer_of(genome):
    """Two bases past the smallest k with 4^k >= n, at most 15."""
    k = 4
    while 4 ** k < genome:
        k += 1
    return min(15, k + 2)


def listed():
    return [
        # one small request of a mapping service: 500 reads, where the launches
        # and the longest read count
        _case("request_64m", "search1", 64 * MBP, 500, 150, mode=hpgfm.MODE_MISMATCH, cap=16,
              resolve=False),
        # the headline batch: a million reads over a chromosome-sized reference
        _case("search1_64m", "search1", 64 * MBP, 1_000_000, 150, mode=hpgfm.MODE_MISMATCH,
              cap=32, resolve=False),
        # the same search over a human-sized genome (45% repeats)
        _case("search1_3g", "search1", 3100 * MBP, 2_000_000, 150, mode=hpgfm.MODE_MISMATCH,
              cap=32, resolve=False),
        # reads of mixed lengths with N bases, indels allowed, and the genome
        # positions of every record: one sequencing lane's budget-1 group
        _case("edit_256m", "search1", 256 * MBP, 700_000, 0, n_rate=0.005,
              mode=hpgfm.MODE_EDIT, cap=16, resolve=True),
        # an index used as it was loaded: no expansion, no table
        _case("compact_64m", "search1", 64 * MBP, 200_000, 100, expand=False, kmer=0,
              mode=hpgfm.MODE_MISMATCH, cap=32, resolve=False),
        # error-free short reads over a bacterial genome
        _case("exact_1m", "exact", 1 * MBP, 100_000, 100, sub=0.0, cap=64),
        # the budget-0 group of the mixed lane, located
        _case("exact_256m", "exact", 256 * MBP, 2_000_000, 0, n_rate=0.005, cap=16),
        # the budget-2 group of the mixed lane
        _case("search_k_256m", "search_k", 256 * MBP, 600_000, 0, n_rate=0.005, list_cap=128,
              anchor_cap=16),
        # seeding of long reads over a human-sized genome
        _case("seeds_3g", "seeds", 3100 * MBP, 1_000_000, 250, seed_len=18, stride=5,
              filter=1000),
        # seeding with one error per window
        _case("inexact_64m", "inexact", 64 * MBP, 250_000, 150, seed_size=18, min_seed=16,
              region_cap=32),
        # the mapping layer's own 1-error search
        _case("vector_64m", "vector", 64 * MBP, 250_000, 150, cap=32),
        # FASTQ text to alignments, read by read
        _case("map_fastq_64m", "map", 64 * MBP, 500_000, 100, sub=0.002, cap=16, filter=50),
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(lo * (hi / lo) ** rng.random()))

    path = rng.choice(["search1", "search1", "exact", "search_k", "seeds", "inexact", "vector",
                       "map"])
    genome = log_int(1 * MBP, 256 * MBP)
    if path in ("search1", "seeds") and rng.random() < 0.2:
        genome = 3100 * MBP
    expand = genome > 1000 * MBP or rng.random() < 0.8
    kmer = _kmer_of(genome) if expand else rng.choice([0, 12])
    most = {"search1": 2_000_000, "exact": 2_000_000, "search_k": 600_000, "seeds": 1_000_000,
            "inexact": 250_000, "vector": 250_000, "map": 500_000}[path]
    reads = log_int(500, most if expand else most // 8)
    length = 0 if rng.random() < 0.35 else log_int(60, 250)
    if path in ("vector", "inexact", "map"):
        length = min(length, 150)
    more = {
        "search1": lambda: dict(mode=rng.choice([hpgfm.MODE_MISMATCH, hpgfm.MODE_EDIT]),
                                cap=rng.choice([8, 16, 32]), resolve=rng.random() < 0.3),
        "exact": lambda: dict(cap=rng.choice([16, 64])),
        "search_k": lambda: dict(list_cap=rng.choice([64, 128]), anchor_cap=16),
        "seeds": lambda: dict(seed_len=rng.randint(18, 32), stride=rng.randint(5, 18),
                              filter=rng.choice([100, 1000])),
        "inexact": lambda: dict(seed_size=rng.randint(18, 24), min_seed=16, region_cap=32),
        "vector": lambda: dict(cap=32),
        "map": lambda: dict(cap=16, filter=rng.choice([10, 50])),
    }[path]()
    c = _case("", path, genome, reads, length, expand=expand, kmer=kmer,
              sub=round(rng.uniform(0.002, 0.02), 4), n_rate=rng.choice([0.0, 0.005]), **more)
    del c["name"]
    return c


# ---------------------------------------------------------------- inputs

_INDEXES = {}                        # the program's indexes: (bases, expand, k) -> (index, text)
_TEXTS = {}


def _text(n):
    """The reference text of n bases on the GPU: i.i.d. bases at 41% GC, from
    16 Mbp on with repeat families (20 mutated copies of a consensus of 300
    to 6000 bases each, half of them reverse-complemented) over 20% of it, 45%
    from 1 Gbp on.  Copies sit in slots of their own, so that the text does
    not depend on the order of the writes."""
    if n in _TEXTS:
        return _TEXTS[n]
    gen = torch.Generator(device="cuda").manual_seed(n)
    g = torch.empty(n, dtype=torch.uint8, device="cuda")
    lut = torch.zeros(256, dtype=torch.uint8, device="cuda")
    lut[75:] = 1                     # A T at 75 / 256 each, C G at 53
    lut[128:] = 2
    lut[181:] = 3
    for a in range(0, n, 1 << 28):
        b = min(n, a + (1 << 28))
        r = torch.randint(0, 256, (b - a,), generator=gen, device="cuda", dtype=torch.uint8)
        g[a:b] = lut[r.int()]
    frac = 0.0 if n < 16 * MBP else (0.45 if n > 1000 * MBP else 0.2)
    nslots = n // 6000
    copies = int(frac * n / 3150) // 20 * 20
    if copies:
        slots = torch.randperm(nslots, generator=gen, device="cuda")[:copies]
        fam_len = torch.randint(300, 6001, (copies // 20,), generator=gen, device="cuda")
        cons_at = torch.randint(0, n - 6000, (copies // 20,), generator=gen, device="cuda")
        src = g.clone()              # a family's consensus is a stretch of the i.i.d. bases
        for a in range(0, copies, 4000):
            s = slots[a:a + 4000]
            fam = torch.arange(a, a + len(s), device="cuda") // 20
            ln = fam_len[fam]
            col = torch.arange(6000, device="cuda")[None, :]
            keep = col < ln[:, None]
            flip = (torch.rand(len(s), generator=gen, device="cuda") < 0.5)[:, None]
            at = torch.where(flip, ln[:, None] - 1 - col, col).clamp_(min=0)
            c = src[cons_at[fam][:, None] + at]
            c = torch.where(flip, 3 - c, c)
            div = 0.02 + 0.13 * torch.rand(len(s), generator=gen, device="cuda")
            m = torch.rand(c.shape, generator=gen, device="cuda") < div[:, None]
            c = torch.where(m, (c + torch.randint(1, 4, c.shape, generator=gen, device="cuda",
                                                  dtype=torch.uint8)) % 4, c)
            dst = s[:, None] * 6000 + col
            g[dst[keep]] = c[keep]
    while len(_TEXTS) >= 6:          # drawn sizes come and go
        _TEXTS.pop(next(iter(_TEXTS)))
    _TEXTS[n] = g
    return g


def _index(case):
    key = (case["genome"], case["expand"], case["kmer"])
    if key not in _INDEXES:
        text = _text(case["genome"])
        host = text.cpu().numpy()
        torch.cuda.empty_cache()
        ix = hpgfm.Index.build_gpu(host, 16)
        if case["expand"]:
            ix.expand()
        if case["kmer"]:
            ix.kmer_table(case["kmer"])
        while len(_INDEXES) >= 6:
            _INDEXES.pop(next(iter(_INDEXES)))
        _INDEXES[key] = ix
    return _INDEXES[key], _text(case["genome"])


def _reads(case, text, seed):
    """(codes uint8, offsets int64) on the GPU: reads from random positions of
    either strand with uniform substitutions and N bases; length 0 draws
    log-normal lengths (median 120, 50 to 250)."""
    gen = torch.Generator(device="cuda").manual_seed(1_000_003 * int(seed) + 17)
    n = case["reads"]
    if case["length"]:
        lens = torch.full((n,), case["length"], dtype=torch.int64, device="cuda")
    else:
        z = torch.randn(n, generator=gen, device="cuda", dtype=torch.float64)
        lens = (120.0 * torch.exp(0.35 * z)).round().clamp(50, 250).long()
    offs = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    offs[1:] = lens.cumsum(0)
    pos = (torch.rand(n, generator=gen, device="cuda", dtype=torch.float64) *
           (len(text) - 250)).long()
    rev = torch.rand(n, generator=gen, device="cuda") < 0.5
    codes = torch.empty(int(offs[-1]), dtype=torch.uint8, device="cuda")
    for a in range(0, n, 200_000):   # in pieces: the index arithmetic is 64-bit
        b = min(n, a + 200_000)
        row = torch.repeat_interleave(torch.arange(a, b, device="cuda"), lens[a:b])
        o0, o1 = int(offs[a]), int(offs[b])
        local = torch.arange(o0, o1, device="cuda") - offs[row]
        rv = rev[row]
        s = text[pos[row] + torch.where(rv, lens[row] - 1 - local, local)]
        s = torch.where(rv, 3 - s, s)
        m = torch.rand(len(s), generator=gen, device="cuda") < case["sub"]
        s = torch.where(m, (s + torch.randint(1, 4, s.shape, generator=gen, device="cuda",
                                              dtype=torch.uint8)) % 4, s)
        if case["n_rate"]:
            s[torch.rand(len(s), generator=gen, device="cuda") < case["n_rate"]] = 4
        codes[o0:o1] = s
    if case["path"] == "exact" and not case["sub"]:   # a tenth of the reads is not from the text
        k = n // 10
        codes[:int(offs[k])] = torch.randint(0, 4, (int(offs[k]),), generator=gen, device="cuda",
                                             dtype=torch.uint8)
    return codes, offs


def _out(n, words):
    """n zeroed records of `words` 8-byte words."""
    return torch.zeros((max(n, 1), words), dtype=torch.int64, device="cuda")


def _p(t):
    return None if t is None else C.c_void_p(t.data_ptr())


def prepare(case, seed):
    ix, text = _index(case)
    codes, offs = _reads(case, text, seed)
    n = case["reads"]
    s = dict(case=case, ix=ix, codes=codes, offs=offs, n=n)
    path = case["path"]
    i32 = dict(dtype=torch.int32, device="cuda")
    if path == "search1":
        s["hits"] = _out(2 * n * case["cap"], 4)
        s["counts"] = torch.zeros(2 * n, **i32)
        if case["resolve"]:
            s["chrom"] = torch.zeros((2 * n * case["cap"], 4), **i32)
            s["coord"] = _out(2 * n * case["cap"], 4)
    elif path == "vector":
        s["hits"] = _out(2 * n * case["cap"], 4)
        s["counts"] = torch.zeros(2 * n, **i32)
    elif path == "exact":
        s["recs"] = [_out(n, 4) for _ in range(2)]
        s["pos"] = [_out(n, case["cap"]) for _ in range(2)]
        s["rows"] = [torch.zeros(n, **i32) for _ in range(2)]
    elif path == "search_k":
        s["frag"] = ((offs[1:] - offs[:-1]) // 3).to(torch.int16)
        s["final"] = _out(2 * n * case["list_cap"], 8)
        s["nfinal"] = torch.zeros(2 * n, **i32)
        s["anchors"] = _out(2 * n * case["anchor_cap"], 8)
        s["nanchors"] = torch.zeros(2 * n, **i32)
        s["full"] = torch.zeros(2 * n, dtype=torch.uint8, device="cuda")
    elif path == "seeds":
        s["got"] = (C.c_uint64(), C.c_uint64())
        s["region_cap"] = 2 * _seeds(case)
        s["regions"] = _out(s["region_cap"], 4)
    elif path == "inexact":
        s["nwin"] = n * ((case["length"] or 160) // case["seed_size"] + 1)
        s["regions"] = _out(2 * s["nwin"] * case["region_cap"], 6)
        s["nreg"] = torch.zeros(2 * s["nwin"], **i32)
        s["status"] = torch.zeros(2 * s["nwin"], dtype=torch.uint8, device="cuda")
        s["got"] = C.c_uint64()
    elif path == "map":
        letters = torch.tensor([65, 67, 71, 84, 78], dtype=torch.uint8, device="cuda")
        read = torch.repeat_interleave(torch.arange(n, device="cuda"), offs[1:] - offs[:-1])
        s["seq"] = torch.zeros(len(codes) + n, dtype=torch.uint8, device="cuda")
        s["seq"][torch.arange(len(codes), device="cuda") + read] = letters[codes.int()]
        s["indices"] = (offs + torch.arange(n + 1, device="cuda")).to(torch.int32)
        s["codes"] = torch.zeros(n * (case["length"] or 160), dtype=torch.uint8, device="cuda")
        s["offs"] = torch.zeros_like(offs)
        s["maps"] = _out(n * case["cap"], 3)
        s["counts"] = torch.zeros(n, **i32)
        s["status"] = torch.zeros(n, dtype=torch.uint8, device="cuda")
    return s


def run(s):
    case, ix, n, L = s["case"], s["ix"], s["n"], hpgfm.lib()
    codes, offs = _p(s["codes"]), _p(s["offs"])
    path = case["path"]
    if path == "search1":
        hpgfm.check(L.fmi_search1_batch(ix.h, case["mode"], 3, codes, offs, n, case["cap"],
                                        _p(s["hits"]), _p(s["counts"]), None))
        if not case["resolve"]:
            return {"hits": s["hits"], "counts": s["counts"]}
        hpgfm.check(L.fmi_resolve_hits(ix.h, _p(s["hits"]), _p(s["counts"]), offs, n, case["cap"],
                                       4, _p(s["chrom"]), _p(s["coord"]), None))
        return {k: s[k] for k in ("hits", "counts", "chrom", "coord")}
    if path == "vector":
        hpgfm.check(L.fmi_search1_vector_batch(ix.h, hpgfm.MODE_EDIT, 3, codes, offs, None, n,
                                               case["cap"], _p(s["hits"]), _p(s["counts"]), None))
        return {"hits": s["hits"], "counts": s["counts"]}
    if path == "exact":
        for t, view in ((0, hpgfm.VIEW_BACKWARD), (1, hpgfm.VIEW_BACKWARD_REV)):
            hpgfm.check(L.fmi_exact_batch(ix.h, view, t, codes, offs, n, _p(s["recs"][t]), None,
                                          None))
            hpgfm.check(L.fmi_locate_hits(ix.h, 0, _p(s["recs"][t]), n, case["cap"],
                                          _p(s["pos"][t]), _p(s["rows"][t]), None))
        return {k: s[k] for k in ("recs", "pos", "rows")}
    if path == "search_k":
        hpgfm.check(L.fmi_search_k_batch(ix.h, 3, codes, offs, _p(s["frag"]), n, case["list_cap"],
                                         case["anchor_cap"], _p(s["final"]), _p(s["nfinal"]),
                                         _p(s["anchors"]), _p(s["nanchors"]), _p(s["full"]),
                                         None))
        return {k: s[k] for k in ("final", "nfinal", "anchors", "nanchors", "full")}
    if path == "seeds":
        hpgfm.check(L.fmi_seed_map_batch(ix.h, codes, offs, n, case["seed_len"], case["stride"],
                                         case["filter"], None, 0, _p(s["regions"]),
                                         s["region_cap"], C.byref(s["got"][0]),
                                         C.byref(s["got"][1]), None))
        return {"regions": s["regions"], "nseeds": int(s["got"][0].value),
                "nrows": int(s["got"][1].value)}
    if path == "inexact":
        hpgfm.check(L.fmi_map_inexact_seeds_batch(ix.h, codes, offs, n, case["seed_size"],
                                                  case["min_seed"], 256, case["region_cap"],
                                                  s["nwin"], _p(s["regions"]), _p(s["nreg"]),
                                                  _p(s["status"]), C.byref(s["got"]), None))
        return {k: s[k] for k in ("regions", "nreg", "status")}
    hpgfm.check(L.fmi_fastq_encode_batch(_p(s["seq"]), _p(s["indices"]), n, len(s["seq"]), codes,
                                         offs, None))
    hpgfm.check(L.fmi_map_reads_batch(ix.h, codes, offs, n, case["filter"], case["cap"],
                                      _p(s["maps"]), _p(s["counts"]), _p(s["status"]), None))
    return {k: s[k] for k in ("maps", "counts", "status", "codes", "offs")}


# ---------------------------------------------------------------- what a pass needs

def _seeds(case):
    """Seeds of a batch (of its mean length when lengths are drawn)."""
    return case["reads"] * max(
        1, ((case["length"] or 127) - case["seed_len"]) // case["stride"] + 1)


def work(case):
    """Reads and offsets read once, results written once, and the index lines
    of 64 bytes that any search with these structures has to touch at random:
    per read and strand a table entry (or its first block) per pass, and for
    the strand the read was drawn from a suffix-array entry, the text under
    the read and the row of its record."""
    n = case["reads"]
    length = case["length"] or 125
    bases = n * length
    path = case["path"]
    line = 64
    text = -(-length // 256) + 1     # lines of 2-bit text under a read
    if path == "search1":
        b = bases + 8 * n + 2 * 4 * n + 32 * n + line * n * (4 + 2 + text)
        if case["resolve"]:
            b += n * (32 + 12 + line)
    elif path == "vector":
        b = bases + 8 * n + 2 * 4 * n + 32 * n + line * n * (4 + 2 + text)
    elif path == "exact":
        b = 2 * (bases + 8 * n + 2 * 32 * n + 8 * n + 4 * n) + line * n * (2 + 2 + text)
    elif path == "search_k":
        b = bases + 8 * n + n * 2 * 9 + 64 * 2 * n + line * n * (6 + 3 + text)
    elif path == "seeds":
        seeds = _seeds(case)
        b = bases + 8 * n + line * 2 * seeds + seeds * (line + 32)
    elif path == "inexact":
        win = n * max(1, length // case["seed_size"])
        b = bases + 8 * n + win * (2 * 5 + 48) + line * win * (4 + 2)
    else:
        b = 2 * (bases + n) + 16 * n + n * (24 + 5) + line * n * (2 + 1 + text)
    return {"bytes": float(b), "flops": 0.0}


def tolerance(case):
    if case["path"] == "search_k":
        # the error entries of a record past its num_mismatches are not part
        # of it and hold what an earlier record left there: 8e-5 of the
        # 8-byte words differ between two runs on the same inputs, all in
        # those entries
        return {"rel": 0.0, "max": 0.0, "differ": 4e-4}
    return "exact"                   # records, positions and counts are whole numbers
