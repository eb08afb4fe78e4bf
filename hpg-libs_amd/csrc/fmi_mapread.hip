// fmi_mapread.hip -- the read-level 1-error mapping of __bwt_map_inexact_read
// (bwt.c:1890-2236) up to its list of alignments, per read on the device.
//
// Only the error-free records of the read's 1-error search become
// alignments (bwt.c:2038), and the vector-driven search yields at most one
// per strand: the exact interval of the whole read on the strand pair's
// first index (its backward vector's entry 0, search.c:1505-1508) -- here a
// plain backward search on BACKWARD (+ strand) or FORWARD_REV (- strand).
// The running count of l - k over them is held to filter_read_mappings
// before each strand's rows (bwt.c:2145-2156); each SA row inside a contig
// gives an alignment at its 0-based coordinate (bwt.c:2158-2166); each
// strand's alignments are deduplicated within 10 bp on the reference's int
// positions and handed over from last to first with the secondary flag
// (bwt.c:2190-2233).
//
// Two launches.  map_single_kernel, a thread per read, settles every read of
// at most kStagedMaxLen bases whose strands have at most kTextRows rows each
// (one on a compact index) or more than the filter lets through, and marks the
// others in counts;
// map_reads_kernel's lanes stride over the marked reads, a lane keeping the
// current strand's alignments in its scratch slice (at most filter + 1 of
// them: a strand's rows number l - k + 1 <= filter + 1 once the count has
// passed) for the dedup.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "../../include/fmi.h"
#include "fmi_device.h"
#include "fmi_internal.h"
#include "fmi_kernels.h"
#include "fmi_rows.h"

namespace fmi {

namespace {

struct MapTmp {
  uint64_t pos;
  uint32_t chrom;
  uint32_t del;
};

struct MapParams {
  DevIndex ix;
  const uint8_t *reads;
  const uint64_t *offsets;
  const uint64_t *koff;       // kcount + 1 contig offsets
  const uint64_t *kstart;     // kcount contig starts
  uint32_t kcount, nreads, filter, cap;
  fmi_read_mapping *out;
  uint32_t *counts;
  uint8_t *status;
  MapTmp *scratch;            // lanes * (filter + 1)
  int32_t wide_m;             // of map_single_kernel's searches (search_rows)
};

// A read's count while the read waits for map_reads_kernel (a count is at
// most 2 (filter + 1)).
constexpr uint32_t kMapWaits = 0xFFFFFFFFu;

// BWExactSearchBackward of the whole read from [0, n] on one view: whether its
// interval is not empty (kRowsNone: an empty one is not formed, no caller sees
// it), and then its rows' suffixes R, or on a compact index, or where there are
// more of them, the rows k..l (R.n = 0).  wide_m, kRowsCut: as search_rows.
template <bool STAGED>
__device__ __forceinline__ uint32_t live_interval(const DevIndex &ix, uint32_t dsel, uint32_t comp,
                                                  const ReadBases<STAGED> &rd, int32_t len,
                                                  uint32_t &k, uint32_t &l, TextRows &R,
                                                  int32_t wide_m = INT32_MAX) {
  const DevDir &D = dir_of(ix, dsel);
  R.n = 0u;
  if (ix.text != nullptr)
    return search_rows<STAGED>(ix, dsel, comp, rd, len - 1, -1, len, R, k, l, wide_m);
  const int32_t K = ix.kmer_k && len >= (int32_t)ix.kmer_k ? (int32_t)ix.kmer_k : 0;
  k = 0u;
  l = ix.n;
  if (K) {
    uint32_t c;
    if (!rd.code(len - 1, -1, K, comp, c)) return kRowsNone;
    const uint64_t e = (dsel ? ix.kmer[1] : ix.kmer[0])[c];
    k = (uint32_t)e;
    l = (uint32_t)(e >> 32);
    if (k > l) return kRowsNone;
  }
  for (int32_t i = len - 1 - K; i >= 0; --i) {
    uint32_t a, b;
    const uint32_t sym = STAGED ? lf_sym(D, k, l, rd.at(i), comp, a, b)
                                : lf_read(D, k, l, rd.W + i, comp, a, b);
    if (sym > 3u || a > b) return kRowsNone;
    k = a;
    l = b;
  }
  return kRowsMany;
}

// The contig of an occurrence at text position key of len bases (binsearch,
// search/io.h:43-64): its index + 1, or 0 when it lies in none.
__device__ __forceinline__ uint32_t contig_of(const uint64_t *koff, uint32_t kcount, uint64_t key,
                                              uint64_t len) {
  uint32_t lo = 0, cnt = kcount;       // upper_bound of key in koff[0 .. kcount)
  while (cnt > 0) {
    const uint32_t w = cnt / 2;
    if (koff[lo + w] <= key) { lo += w + 1; cnt -= w + 1; }
    else cnt = w;
  }
  return lo == 0 || key + len > koff[lo] ? 0u : lo;
}

__device__ __forceinline__ void store_mapping(fmi_read_mapping *out, uint64_t pos, uint32_t chrom,
                                              uint32_t rd, uint32_t strand, uint32_t secondary,
                                              int32_t len) {
  fmi_read_mapping o;
  o.position = pos;
  o.chromosome = chrom;
  o.read = rd;
  o.strand = (uint8_t)strand;
  o.secondary = (uint8_t)secondary;
  o.cigar_len = (uint16_t)len;
  o.pad = 0u;
  *out = o;
}

// One thread per read.  The read is packed into the thread's LDS slot once
// for both strands, and each is searched to its rows on the text (search_rows):
// about six dependent loads for a read that occurs once where an LF step per
// base and strand took 100 and more.  Bound by those loads' lines
// (an entry per strand, then SA and text for one of them); the slots
// (24 KB a workgroup) leave 6 workgroups a CU.  500 K reads of 100 bases over
// 64 Mbp: 145 us, where one launch of 64 K lanes (the scratch allows no more)
// took 1540, and 125 went to the marked reads when they were those with more
// than one row.  A strand over the filter ends its read here: 100 K reads of 3000
// copies 209 us at a filter of 50, where searching them again took 479 (LF steps
// alone 318).  Reads of 5 copies to the filter are searched twice: of 130 copies
// at a filter of 1000 4.03 ms, 3.80 by LF steps alone.
__global__ __launch_bounds__(256) void map_single_kernel(MapParams P) {
  __shared__ uint32_t slots[kReadRecordWords * 256u];
  const uint32_t rd = blockIdx.x * 256u + threadIdx.x;
  if (rd >= P.nreads) return;
  const uint64_t off = P.offsets[rd];
  const uint64_t len64 = P.offsets[rd + 1] - off;
  if (len64 < 5 || len64 > kMaxReadLen) {
    P.counts[rd] = 0;
    P.status[rd] = len64 < 5 ? 2u : 4u;
    return;
  }
  if (len64 > kStagedMaxLen) {
    P.counts[rd] = kMapWaits;
    return;
  }
  const uint8_t *W = P.reads + off;
  const int32_t len = (int32_t)len64;
  uint32_t *slot = slots + threadIdx.x;
  stage_read(W, (uint32_t)len, slot);
  const uint32_t n = P.ix.n;
  const ReadBases<true> bases{W, slot};
  uint32_t nout = 0, tot = 0;
  uint8_t st = 0;
  for (uint32_t strand = 0; strand < 2u; ++strand) {
    // + strand: BACKWARD; - strand: FORWARD_REV (bwt.c:1996-2001)
    uint32_t k, l;
    TextRows R;
    const uint32_t found = live_interval<true>(P.ix, strand, strand, bases, len, k, l, R, P.wide_m);
    if (found == kRowsNone) continue;
    if (R.n == 0u) {
      if (found == kRowsMany && k != l && l - k > P.filter - tot) {
        st = 1u;
        break;
      }
      if (found == kRowsCut || k != l) {
        P.counts[rd] = kMapWaits;
        return;
      }
      R.n = 1u;
      R.q[0] = sa_value(dir_of(P.ix, strand), P.ix.ratio, n, k);
    }
    tot += R.n - 1u;
    if (tot > P.filter) { st = 1u; break; }
    uint64_t pos[kTextRows];
    uint32_t chrom[kTextRows];               // contig + 1, 0: no alignment
#pragma unroll
    for (uint32_t j = 0; j < kTextRows; ++j) {
      pos[j] = 0u;
      chrom[j] = 0u;
      if (j >= R.n) continue;
      // direction: the record's dir is 0; + keeps it, - flips it
      const uint64_t key =
          strand ? (uint64_t)n + 1u - R.q[j] - (uint64_t)len - 1u : (uint64_t)R.q[j];
      chrom[j] = contig_of(P.koff, P.kcount, key, (uint64_t)len);
      if (chrom[j]) pos[j] = P.kstart[chrom[j] - 1u] + (key - P.koff[chrom[j] - 1u]);
    }
    // within 10 bp on the int positions an earlier alignment drops a later
    // one; the others are handed over from the last to the first
#pragma unroll
    for (int32_t a1 = (int32_t)kTextRows - 1; a1 >= 0; --a1) {
      bool stays = chrom[a1] != 0u;
#pragma unroll
      for (int32_t a2 = 0; a2 < a1; ++a2) {
        const int32_t d = (int32_t)((uint32_t)pos[a1] - (uint32_t)pos[a2]);
        const int64_t ad = d < 0 ? -(int64_t)d : (int64_t)d;
        if (chrom[a2] == chrom[a1] && ad < 10) stays = false;
      }
      if (!stays) continue;
      if (nout < P.cap)
        store_mapping(P.out + (uint64_t)rd * P.cap + nout, pos[a1], chrom[a1] - 1u, rd, strand,
                      nout > 0 ? 1u : 0u, len);
      ++nout;
    }
  }
  P.counts[rd] = nout;
  P.status[rd] = st;
}

__global__ __launch_bounds__(256) void map_reads_kernel(MapParams P) {
  const uint32_t lane = blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t lanes = gridDim.x * blockDim.x;
  MapTmp *tmp = P.scratch + (uint64_t)lane * (P.filter + 1u);
  const uint32_t n = P.ix.n;
  for (uint32_t rd = lane; rd < P.nreads; rd += lanes) {
    if (P.counts[rd] != kMapWaits) continue;
    const uint64_t off = P.offsets[rd];
    const uint8_t *W = P.reads + off;
    fmi_read_mapping *out = P.out + (uint64_t)rd * P.cap;
    const int32_t len = (int32_t)(P.offsets[rd + 1] - off);
    const ReadBases<false> bases{W, nullptr};
    uint64_t tot = 0;
    uint32_t nout = 0;
    uint8_t st = 0;
    for (int type = 1; type >= 0; --type) {
      // + strand: BACKWARD; - strand: FORWARD_REV (bwt.c:1996-2001)
      const uint32_t dsel = type ? 0u : 1u;
      const DevDir &D = dir_of(P.ix, dsel);
      uint32_t k, l;
      TextRows R;
      uint32_t m = 0;
      if (live_interval<false>(P.ix, dsel, dsel, bases, len, k, l, R) != kRowsNone) {
        if (R.n) { k = 0u; l = R.n - 1u; }             // the rows' suffixes are known
        tot += (uint64_t)(l - k);
        if (tot > P.filter) { st |= 1u; break; }
        for (uint32_t j = k; j <= l; ++j) {
          // direction: the record's dir is 0; + keeps it, - flips it
          const uint64_t sa = R.n ? pick4(R.q, j) : sa_value(D, P.ix.ratio, n, j);
          const uint64_t key = type ? sa : (uint64_t)n + 1u - sa - (uint64_t)len - 1u;
          const uint32_t c = contig_of(P.koff, P.kcount, key, (uint64_t)len);
          if (c == 0u) continue;
          tmp[m].pos = P.kstart[c - 1] + (key - P.koff[c - 1]);
          tmp[m].chrom = c - 1u;
          tmp[m].del = 0u;
          ++m;
        }
      }
      // within 10 bp on the int positions: a later alignment goes when an
      // earlier one (all carry one CIGAR operation) sits within 10
      for (int32_t a1 = (int32_t)m - 1; a1 >= 1; --a1) {
        const int32_t p1 = (int32_t)(uint32_t)tmp[a1].pos;
        for (int32_t a2 = a1 - 1; a2 >= 0; --a2) {
          const int32_t d = (int32_t)((uint32_t)p1 - (uint32_t)tmp[a2].pos);
          const int64_t ad = d < 0 ? -(int64_t)d : (int64_t)d;
          if (tmp[a1].chrom == tmp[a2].chrom && ad < 10) { tmp[a1].del = 1u; break; }
        }
      }
      const bool created_primary = nout == 0;
      bool primary_delete = false;
      for (int32_t a = (int32_t)m - 1; a >= 0; --a) {
        if (tmp[a].del) {
          primary_delete |= created_primary;
          continue;
        }
        if (nout < P.cap) {
          store_mapping(out + nout, tmp[a].pos, tmp[a].chrom, rd, type ? 0u : 1u,
                        nout > 0 ? 1u : 0u, len);
        }
        ++nout;
      }
      if (primary_delete && nout > 0 && P.cap > 0) out[0].secondary = 0;
    }
    P.counts[rd] = nout;
    P.status[rd] = st;
  }
}

}  // namespace

uint32_t map_reads_lanes(uint32_t nreads, uint32_t filter) {
  const uint64_t per = (uint64_t)(filter + 1) * sizeof(MapTmp);
  uint64_t lanes = ((uint64_t)nreads + 255) / 256 * 256;
  uint64_t most = ((1ull << 30) / per) / 256 * 256;
  if (most < 256) most = 256;
  if (lanes > most) lanes = most;
  if (lanes > 64 * 1024) lanes = 64 * 1024;
  return (uint32_t)lanes;
}

uint64_t map_reads_scratch_bytes(uint32_t lanes, uint32_t filter) {
  return (uint64_t)lanes * (filter + 1) * sizeof(MapTmp);
}

hipError_t launch_map_reads(const DevIndex &ix, const uint8_t *reads, const uint64_t *offsets,
                            uint32_t nreads, const uint64_t *koff, const uint64_t *kstart,
                            uint32_t kcount, uint32_t filter, uint32_t cap, fmi_read_mapping *out,
                            uint32_t *counts, uint8_t *status, void *scratch, uint32_t lanes,
                            hipStream_t s) {
  if (nreads == 0 || lanes == 0) return hipSuccess;
  // With a filter below kManyRows an interval of that many rows most likely ends
  // its read, once it is known, in map_single_kernel itself.
  MapParams P{ix,     reads,  offsets, koff,   kstart, kcount, nreads, filter, cap,
              out,    counts, status,  static_cast<MapTmp *>(scratch),
              filter < kManyRows ? INT32_MAX : rows_wide_m(ix.n)};
  hipLaunchKernelGGL(map_single_kernel, dim3((nreads + 255u) / 256u), dim3(256), 0, s, P);
  hipLaunchKernelGGL(map_reads_kernel, dim3(lanes / 256), dim3(256), 0, s, P);
  return hipGetLastError();
}

}  // namespace fmi
