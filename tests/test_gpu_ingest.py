"""Read ingestion from the reference's fastq_batch_t layout
(bioformats/fastq/fastq_batch.h:24-34: sequences with a NUL after each,
int data_indices): the device encoding equals encode_bases
(bwt_commons.c:99-102, fmi_encode_bases on the host) byte for byte with the
offsets the NULs imply; the 2-bit packing holds every code and N flag; and
requests submitted to the serving loop in that layout get the records of
fmi_search1_batch on their encoded reads."""
import numpy as np
import pytest

import fmoracle as fo
from hpgfm import synth

pytestmark = pytest.mark.gpu

LETTERS = np.frombuffer(b"ACGTacgtNnRYKM.-", np.uint8)


def random_texts(rng, n, lo=0, hi=160, odd=0.02):
    out = []
    for _ in range(n):
        L = int(rng.integers(lo, hi))
        t = LETTERS[rng.integers(0, 4, L)].copy()
        low = rng.random(L) < 0.1
        t[low] = LETTERS[rng.integers(4, 8, int(low.sum()))]
        weird = rng.random(L) < odd
        t[weird] = LETTERS[rng.integers(8, 16, int(weird.sum()))]
        out.append(t.tobytes())
    return out


def test_fastq_encode_equals_host_encoding(gpu_engine):
    hp = gpu_engine
    texts = random_texts(np.random.default_rng(141), 3000)
    texts[:3] = [b"", b"A", b""]                     # empty reads keep their NUL
    seq, di = hp.fastq_batch(texts)
    codes, offs = hp.fastq_encode_batch(seq, di)
    want = hp.encode_bases(b"".join(texts))
    assert np.array_equal(codes, want)
    lens = np.array([len(t) for t in texts])
    assert np.array_equal(offs, np.concatenate([[0], np.cumsum(lens)]).astype(np.uint64))
    # data_indices that do not start at 0 (a window of a larger batch)
    codes2, offs2 = hp.fastq_encode_batch(seq, di[1000:2001])
    assert np.array_equal(codes2, want[int(offs[1000]):int(offs[2000])])
    assert np.array_equal(offs2, offs[1000:2001] - offs[1000])


def test_pack_codes_roundtrip(gpu_engine):
    hp = gpu_engine
    rng = np.random.default_rng(142)
    codes = rng.integers(0, 4, 100_003).astype(np.uint8)
    codes[rng.random(len(codes)) < 0.01] = 4
    packed, nmask = hp.pack_codes(codes)
    i = np.arange(len(codes))
    got = (packed[i // 16] >> (2 * (i % 16)).astype(np.uint32)) & 3
    isn = (nmask[i // 16] >> (i % 16).astype(np.uint16)) & 1
    assert np.array_equal(isn.astype(bool), codes > 3)
    assert np.array_equal(got[codes < 4], codes[codes < 4])
    assert np.all(got[codes > 3] == 0)


def test_server_fastq_requests(gpu_engine):
    hp = gpu_engine
    g, _, _ = synth.genome(1_000_000, seed=143, repeat_frac=0.2)
    ix = hp.Index.build(g, 16).to_device()
    rng = np.random.default_rng(144)
    reads, offs, _ = synth.reads(g, 20_000, seed=145, sub_rate=0.01, n_rate=0.002,
                                 lengths=rng.integers(20, 200, 20_000))
    alpha = np.frombuffer(b"ACGTN", np.uint8)
    cap = 6
    srv = hp.Server(ix, budget_bytes=32 << 20, max_inflight=3, max_batch_reads=8000, cap=cap)
    try:
        jobs = []
        a = 0
        while a < 20_000:
            b = min(20_000, a + int(rng.integers(1, 3000)))
            texts = [alpha[reads[int(offs[i]):int(offs[i + 1])]].tobytes() for i in range(a, b)]
            if len(jobs) % 2:
                texts = [t.lower() for t in texts]
            seq, di = hp.fastq_batch(texts)
            if len(jobs) % 3 == 0:
                rid = srv.submit_fastq(seq, di)
            else:
                o = offs[a:b + 1]
                rid = srv.submit(reads[int(o[0]):int(o[-1])], o - o[0])
            jobs.append((a, b, rid))
            a = b
        for a, b, rid in jobs:
            c, h, _ = srv.wait(rid, timeout_us=60_000_000)
            o = offs[a:b + 1]
            batch = hp.ReadBatch(reads[int(o[0]):int(o[-1])], o - o[0])
            c2, h2 = hp.search1_batch(ix, batch, cap=cap, mode=hp.MODE_MISMATCH)
            batch.free()
            assert np.array_equal(c, c2), (a, b)
            alone = h2[np.arange(cap)[None, None, :] < np.minimum(c2, cap)[:, :, None]]
            assert fo.hits_equal(h, alone), (a, b)
    finally:
        srv.close()
        ix.close()


@pytest.mark.parametrize("kind", ["tile edges", "empty reads", "one long read", "tiny"])
def test_fastq_encode_tiles(gpu_engine, kind):
    """Reads that end on, before and after the 8192-byte tiles of the encoding
    kernel, more reads in a tile than it stages ends for, one read over many
    tiles, and batches of a few bytes, each from every 16-byte alignment."""
    hp = gpu_engine
    rng = np.random.default_rng(146)
    lens = {"tile edges": [8190, 0, 8191, 8192, 1, 8160, 15, 16, 17, 4095, 4096],
            "empty reads": [0] * 5000 + [3, 0, 2] * 400 + [0] * 1030,
            "one long read": [70_001],
            "tiny": [1]}[kind]
    texts = [LETTERS[rng.integers(0, 16, n)].tobytes() for n in lens]
    for lead in range(16):
        seq, di = hp.fastq_batch([b"G" * lead] + texts if lead else texts)
        first = 1 if lead else 0
        codes, offs = hp.fastq_encode_batch(seq, di[first:])
        assert np.array_equal(codes, hp.encode_bases(b"".join(texts))), lead
        assert np.array_equal(offs, np.concatenate([[0], np.cumsum(lens)]).astype(np.uint64))


@pytest.mark.parametrize("nbytes", [1 << 19, (1 << 19) + 1, 1 << 24, (1 << 24) + 1])
@pytest.mark.parametrize("shape", ["long", "short", "empty"])
def test_fastq_encode_at_the_sizes_of_its_kernels(gpu_engine, nbytes, shape):
    """Batches at the sizes where another kernel or tile takes over, of reads of 0
    to 300 bases, of 0 to 3, and of none at all: the host's codes and offsets."""
    hp = gpu_engine
    rng = np.random.default_rng(nbytes)
    most = {"long": 300, "short": 3, "empty": 0}[shape]
    lens = rng.integers(0, most + 1, nbytes // (most // 2 + 1) + 10)
    ends = np.cumsum(lens + 1)
    m = int(np.searchsorted(ends, nbytes, side="right"))
    di = np.concatenate([[0], ends[:m], [nbytes] if ends[m - 1] < nbytes else []]).astype(np.int32)
    seq = LETTERS[rng.integers(0, 16, nbytes)]
    seq[di[1:] - 1] = 0
    codes, offs = hp.fastq_encode_batch(seq, di)
    keep = np.ones(nbytes, bool)
    keep[di[1:] - 1] = False
    assert np.array_equal(codes, hp.encode_bases(seq[keep].tobytes()))
    assert np.array_equal(offs, (di - np.arange(len(di))).astype(np.uint64))


def test_fastq_encode_small_batches_cost(gpu_engine):
    """A service's batch of 100 reads is as quick as its launch: 6.2 us on the
    device, 11.5 where two workgroups took it."""
    hp = gpu_engine
    seq, di = hp.fastq_batch([b"ACGT" * 25] * 100)
    d = [hp.DeviceBuffer.from_array(np.frombuffer(bytes(seq), np.uint8)),
         hp.DeviceBuffer.from_array(np.asarray(di, np.int32)), hp.DeviceBuffer(10_200),
         hp.DeviceBuffer(8 * 101)]
    took = []
    for _ in range(60):
        hp.check(hp.lib().fmi_fastq_encode_batch(d[0].ptr, d[1].ptr, 100, 10_100, d[2].ptr, d[3].ptr, None))
        took.append(hp.last_kernel_ms())
    for b in d:
        b.free()
    assert np.median(took) < 9e-3, np.median(took)
