// fmi_search1t.hip -- the 1-error search (BWSearch1CPU, search/search.c:1876-
// 1933) of an expanded index on the text.
//
// A pass searches its anchor half exactly and scans the other half from there:
// a node (the interval of the anchor and some bases more) has branches when
// the scan's next step changes its size, which on the text is where a row's
// text and the read part.  So a pass is the anchor's rows (search_rows), how
// far each goes on with the read, and at each such place the comparisons of
// node_strings -- a dozen dependent reads where the step-by-step state machine
// (search1_kernel) takes one per step, a few hundred in a repeat.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "../../include/fmi.h"
#include "fmi_device.h"
#include "fmi_internal.h"
#include "fmi_kernels.h"
#include "fmi_rows.h"

namespace fmi {

namespace {

struct S1tParams {
  DevIndex ix;
  const uint8_t *reads;
  const uint64_t *offsets;
  fmi_hit *hits;
  uint32_t *counts;
  uint32_t *rec;                   // the left reads' records (kReadRecordWords words each)
  // the reads left to search1_wave_kernel, and from wide[nreads - 1] downward
  // those longer than a slot, left to search1_kernel unstaged
  uint32_t *wide, *wide_n, *long_n;
  uint32_t *list, *list_n;         // the reads left to search1_kernel staged
  uint32_t nreads, strand_mask, cap;
  int32_t wide_m;                  // rows_wide_m
};

// Anchor halves shorter than this go to search1_kernel at once: they have more
// than kTextRows rows in a repeat (and from 3.1 Gbp, 4^16, by chance), and the
// passes here would mostly be run in vain.
constexpr int32_t kTextHalf = 16;

// In the count of a read left to search1_kernel (which writes it anew): no
// wavefront can take it, for one of its anchors' more than 64 rows or its length.
constexpr uint32_t kManyRead = 0x80000000u;

struct S1tOut {
  fmi_hit *out;
  uint32_t cap, cnt, strand;
  __device__ __forceinline__ void add(const DevDir &D, uint32_t q, uint32_t rows, int32_t start,
                                      int32_t pos, int32_t end, int32_t err_pos, uint32_t dir,
                                      uint32_t nmm, uint32_t kind, uint32_t base) {
    if (cnt < cap) {
      const uint32_t k = D.isa[q];
      store_hit(out + cnt, (int64_t)k, (int64_t)(k + rows - 1u), (int16_t)start, (int16_t)pos,
                (int16_t)end, (int16_t)err_pos, (uint8_t)dir, (uint8_t)nmm, (uint8_t)kind,
                (uint8_t)base, (uint8_t)strand);
    }
    cnt++;
  }
};

// A record of a node's string number bit at read position p.
__device__ __forceinline__ void add_string(S1tOut &O, const DevDir &D, uint32_t bit, uint32_t q,
                                           uint32_t rows, uint32_t pass, int32_t len, int32_t p) {
  const int32_t half = len / 2;
  O.add(D, q, rows, pass ? half : 0, pass ? len : -1, pass ? len - 1 : half - 1, p, pass, 1u,
        bit == 0u ? FMI_DELETION : ((bit & 1u) ? FMI_INSERTION : FMI_MISMATCH),
        bit == 0u ? 0xFFu : (bit - 1u) >> 1);
}

// One pass (0: the right half backward on the pair's first index, then the
// left; 1: the left half forward on the second, then the right); false when
// the anchor has more rows than it can take (then kManyRead in the count).
template <bool MM_ONLY>
__device__ __forceinline__ bool text_pass(const DevIndex &ix, uint32_t pass, uint32_t strand,
                                          const ReadBases<true> &rd, int32_t len, int32_t wide_m,
                                          S1tOut &O) {
  const uint32_t dsel = pass ^ strand;
  const DevDir &D = dir_of(ix, dsel);
  const int32_t half = len / 2, d = pass ? 1 : -1, p0 = pass ? 0 : len - 1;
  const int32_t m0 = pass ? half : len - half, N = len - m0;
  TextRows R;
  uint32_t k, l;
  const uint32_t found = search_rows<true>(ix, dsel, strand, rd, p0, d, m0, R, k, l, wide_m);
  if (found != kRowsFew) {
    if (found == kRowsNone) return true;
    if (l - k >= 64u) O.cnt |= kManyRead;
    return false;
  }
  int32_t run[kTextRows] = {-1, -1, -1, -1};
#pragma unroll
  for (uint32_t j = 0; j < kTextRows; ++j)
    if (j < R.n) run[j] = rd.match(ix, dsel, strand, R.q[j], p0 + m0 * d, d, N);
  // the nodes with branches, from the anchor outward
  for (int32_t cur = -1;;) {
    int32_t a = N;
#pragma unroll
    for (uint32_t j = 0; j < kTextRows; ++j)
      if (run[j] > cur) a = min(a, run[j]);
    if (a == N) break;
    cur = a;
    const int32_t p = p0 + (m0 + a) * d;
    const NodeStrings T =
        node_strings<true, MM_ONLY>(ix, dsel, strand, rd, R, run, a, p, d, N - 1 - a);
#pragma unroll
    for (uint32_t bit = MM_ONLY ? 2u : 0u; bit < 9u; bit += MM_ONLY ? 2u : 1u) {
      if (!((T.live >> bit) & 1u)) continue;
      add_string(O, D, bit, T.q[bit], (T.cnts >> (3u * bit)) & 7u, pass, len, p);
    }
  }
  if (pass == 0u) {
    uint32_t first = 0u, rows = 0u;
#pragma unroll
    for (uint32_t j = 0; j < kTextRows; ++j)
      if (run[j] == N) {
        if (rows++ == 0u) first = R.q[j] - (uint32_t)N;
      }
    if (rows) O.add(D, first, rows, 0, -1, len - 1, 0, 0u, 0u, 0u, 0u);
  }
  return true;
}

// A thread per (read, strand); a read's two threads pack it into one LDS slot.
// A read with more than kTextRows rows at half of it is left to
// search1_wave_kernel, one with more than 64, an anchor of less than kTextHalf
// bases or more bases than a slot to search1_kernel; its record is written from
// the slot.
// Bound by the latency of a pass's chain and the lines it reads (an entry,
// contexts, suffixes, text and the records' rows), with 20 of 64 lanes active:
// the strand a read is not from ends after its table entry.  At 4 waves: 1 M
// reads of 150 bases over 64 Mbp: 576 us, where the records, the state machine
// and its records' rows took 1284; 2 M over 3.1 Gbp 1552 of 2300; a request of
// 500 reads 43 of 500.
// MINW: the waves per SIMD the registers are held to.  4 (none spilled) where
// every group of the batch is resident at once, and a read's own chain is
// what counts; 6 (80 VGPRs, 24 to 28 spilled: three groups a CU instead of two)
// beyond, where more lines in flight are worth the spills.  Calls: 1 M x 150 at
// 64 Mbp 610 to 569 us (554 now), 2 M at 3.1 Gbp 1608 to 1460 (1437), 700 K of
// 50-250 with indels and positions at 256 Mbp 627 to 557 (582), but 500 reads 60
// to 64.  5 waves (6 spilled) hold no third group.
template <bool MM_ONLY, int MINW>
__global__ __launch_bounds__(512, MINW) void search1_text_kernel(S1tParams P) {
  __shared__ uint32_t slots[kReadRecordWords * 256u];
  __shared__ uint32_t ids[256], nids, narrived;    // the group's left reads
  const uint64_t t64 = (uint64_t)blockIdx.x * 512u + threadIdx.x;
  const uint32_t rd = (uint32_t)(t64 >> 1), strand = (uint32_t)t64 & 1u;
  const bool mine = t64 < 2ull * P.nreads;
  uint32_t *slot = slots + (threadIdx.x >> 1);
  uint64_t off = 0;
  int32_t len = 0;
  if (mine) {
    off = P.offsets[rd];
    len = (int32_t)(P.offsets[rd + 1] - off);
  }
  const bool staged = mine && len <= (int32_t)kStagedMaxLen;
  if (staged) {
    // 32 bases at a time, the two threads in turn, from the 16-byte chunks
    // that hold them (none past the chunk of the read's last byte)
    const uint8_t *W = P.reads + off, *z = W + (len - 1);
    const uint8_t *zc = z - (reinterpret_cast<uintptr_t>(z) & 15u);
    for (uint32_t u = strand; 32 * (int32_t)u < len; u += 2u) {
      const uint8_t *a = W + 32u * u;
      const uint32_t mis = (uint32_t)(reinterpret_cast<uintptr_t>(a) & 15u), sh = 2u * mis;
      const uint8_t *c = a - mis;
      uint4 c1 = make_uint4(0u, 0u, 0u, 0u), c2 = c1;
      const uint4 c0 = *reinterpret_cast<const uint4 *>(c);
      if (c + 16 <= zc) c1 = *reinterpret_cast<const uint4 *>(c + 16);
      if (c + 32 <= zc) c2 = *reinterpret_cast<const uint4 *>(c + 32);
      uint32_t k0, k1, k2, f0, f1, f2;
      pack16(c0, k0, f0);
      pack16(c1, k1, f1);
      pack16(c2, k2, f2);
      const uint64_t lo = ((uint64_t)k1 << 32) | k0;
      const uint64_t code = sh ? (lo >> sh) | ((uint64_t)k2 << (64u - sh)) : lo;
      const uint64_t fl = (uint64_t)f0 | ((uint64_t)f1 << 16) | ((uint64_t)f2 << 32);
      slot[(2u * u) * 256u] = (uint32_t)code;
      slot[(2u * u + 1u) * 256u] = (uint32_t)(code >> 32);
      slot[(16u + u) * 256u] = (uint32_t)(fl >> mis);
    }
  }
  if (threadIdx.x == 0u) nids = narrived = 0u;
  __syncthreads();
  bool left = false;
  uint32_t cnt = 0u;
  if (mine) {
    const bool asked = ((P.strand_mask >> strand) & 1u) != 0u;
    S1tOut O{P.hits + (uint64_t)t64 * P.cap, P.cap, 0u, strand};
    if (!staged || len / 2 < kTextHalf) {
      left = true;
      O.cnt = kManyRead;
    } else if (asked) {
      const ReadBases<true> bases{nullptr, slot};
      for (uint32_t pass = 0; pass < 2u && !left; ++pass)
        left = !text_pass<MM_ONLY>(P.ix, pass, strand, bases, len, P.wide_m, O);
    }
    cnt = O.cnt;
    P.counts[t64] = cnt;
  }
  // the left reads, their records first
  const uint64_t pair = 0x5555555555555555ull;
  uint64_t any = __ballot(left), list = __ballot(cnt >= kManyRead);
  any = (any | (any >> 1)) & pair;
  list = (list | (list >> 1)) & pair;              // a strand's wider anchor decides
  const uint32_t lane = threadIdx.x & 63u;
  const uint64_t me = 1ull << (lane & ~1u);
  if ((any & me) && staged) {
    uint4 *out = reinterpret_cast<uint4 *>(P.rec + (uint64_t)rd * kReadRecordWords);
    for (uint32_t i = strand; i < kReadRecordWords / 4u; i += 2u)
      out[i] = make_uint4(slot[(4u * i) * 256u], slot[(4u * i + 1u) * 256u],
                          slot[(4u * i + 2u) * 256u], slot[(4u * i + 3u) * 256u]);
  }
  // The group's last wavefront to come here appends them all to the lists: an
  // atomic per group.  One per wavefront, 3125 to one address, took 30 of the
  // 42 us that listing 100 K reads of 20 bases took.
  uint32_t at = 0u;
  if (lane == 0u && any) at = atomicAdd(&nids, (uint32_t)__popcll(any));
  at = __shfl(at, 0);
  if ((any & me) && strand == 0u) {
    const uint32_t to = !(list & me) ? 0u : (staged ? 1u : 2u);
    ids[at + (uint32_t)__popcll(any & (me - 1ull))] = (threadIdx.x >> 1) | (to << 8);
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  uint32_t before = 0u;
  if (lane == 0u) before = atomicAdd(&narrived, 1u);
  if (__shfl(before, 0) != 512u / 64u - 1u) return;
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  const uint32_t n = nids;
#pragma unroll 1
  for (uint32_t c = 0; c < 3u; ++c) {
    uint32_t cnt = 0u, at_c = 0u;
#pragma unroll 1
    for (uint32_t i = lane; i - lane < n; i += 64u)
      cnt += (uint32_t)__popcll(__ballot(i < n && ids[min(i, 255u)] >> 8 == c));
    if (cnt == 0u) continue;
    if (lane == 0u) at_c = atomicAdd(c == 0u ? P.wide_n : (c == 1u ? P.list_n : P.long_n), cnt);
    at_c = __shfl(at_c, 0);
#pragma unroll 1
    for (uint32_t i = lane; i - lane < n; i += 64u) {
      const uint32_t id = ids[min(i, 255u)];
      const bool is = i < n && id >> 8 == c;
      const uint64_t m = __ballot(is);
      const uint32_t p = at_c + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
      if (is)
        (c == 1u ? P.list : P.wide)[c == 2u ? P.nreads - 1u - p : p] =
            blockIdx.x * 256u + (id & 255u);
      at_c += (uint32_t)__popcll(m);
    }
  }
}

// text_pass by a wavefront, a row a lane, for anchors of up to 64 rows: the
// rows compare at the same time and a string's rows are a ballot.  Every lane
// calls it with the same arguments; lane 0 stores.
template <bool MM_ONLY>
__device__ __forceinline__ bool wave_pass(const DevIndex &ix, uint32_t pass, uint32_t strand,
                                          const ReadBases<true> &rd, int32_t len, S1tOut &O) {
  const uint32_t dsel = pass ^ strand, lane = threadIdx.x & 63u;
  const DevDir &D = dir_of(ix, dsel);
  const int32_t half = len / 2, d = pass ? 1 : -1, p0 = pass ? 0 : len - 1;
  const int32_t m0 = pass ? half : len - half, N = len - m0;
  uint32_t k = 0u, l = ix.n;
  int32_t m = 0;
  const int32_t K = (int32_t)ix.kmer_k <= m0
                        ? (int32_t)ix.kmer_k
                        : ((int32_t)ix.kmer2_k <= m0 ? (int32_t)ix.kmer2_k : 0);
  if (K) {
    uint32_t c;
    if (!rd.code(p0, d, K, strand, c)) return true;
    const uint64_t e = (K == (int32_t)ix.kmer_k ? (dsel ? ix.kmer[1] : ix.kmer[0])
                                                : (dsel ? ix.kmer2[1] : ix.kmer2[0]))[c];
    k = (uint32_t)e;
    l = (uint32_t)(e >> 32);
    if (k > l) return true;
    m = K;
  }
  for (; m < m0 && l - k >= 64u; ++m) {
    uint32_t a, b;
    if (lf_sym(D, k, l, rd.at(p0 + m * d), strand, a, b) > 3u || a > b) return true;
    k = a;
    l = b;
  }
  if (l - k >= 64u) return false;
  uint32_t q = 0u;
  int32_t run = -1;
  if (lane <= l - k) {
    q = D.sa[k + lane];
    if (rd.match(ix, dsel, strand, q, p0 + m * d, d, m0 - m) == m0 - m) {
      q -= (uint32_t)(m0 - m);
      run = rd.match(ix, dsel, strand, q, p0 + m0 * d, d, N);
    }
  }
  auto put = [&](uint64_t rows, uint32_t bit, uint32_t suffix, int32_t p) {
    if (!rows) return;
    const uint32_t first = __shfl(suffix, (int)__builtin_ctzll(rows));
    if (lane == 0u) add_string(O, D, bit, first, (uint32_t)__popcll(rows), pass, len, p);
  };
  for (int32_t cur = -1;;) {
    int32_t a = run > cur ? run : N;
#pragma unroll
    for (uint32_t x = 32u; x >= 1u; x >>= 1) a = min(a, __shfl_xor(a, (int)x));
    if (a >= N) break;
    cur = a;
    const int32_t p = p0 + (m0 + a) * d, c1 = N - 1 - a;
    const uint32_t w = rd.at(p), sm = w > 3u ? 4u : (strand ? 3u - w : w);
    const uint32_t qa = q - (uint32_t)a;
    bool del = false, mis = false, ins = false;
    uint32_t lb = 0u;
    if (run >= a) {
      if (!MM_ONLY) del = rd.match(ix, dsel, strand, qa, p + d, d, c1) == c1;
      if (qa != 0u) {
        const uint32_t b = (uint32_t)text_window32(ix, dsel, qa) & 3u;
        lb = strand ? 3u - b : b;
        mis = b != sm && rd.match(ix, dsel, strand, qa - 1u, p + d, d, c1) == c1;
        if (!MM_ONLY) ins = rd.match(ix, dsel, strand, qa - 1u, p, d, c1 + 1) == c1 + 1;
      }
    }
    if (!MM_ONLY) put(__ballot(del), 0u, qa - (uint32_t)c1, p);
#pragma unroll
    for (uint32_t b = 0; b < 4u; ++b) {
      if (!MM_ONLY) put(__ballot(ins && lb == b), 1u + 2u * b, qa - 2u - (uint32_t)c1, p);
      put(__ballot(mis && lb == b), 2u + 2u * b, qa - 1u - (uint32_t)c1, p);
    }
  }
  if (pass == 0u) {
    const uint64_t rows = __ballot(run == N);
    if (rows) {
      const uint32_t first = __shfl(q - (uint32_t)N, (int)__builtin_ctzll(rows));
      if (lane == 0u)
        O.add(D, first, (uint32_t)__popcll(rows), 0, -1, len - 1, 0, 0u, 0u, 0u, 0u);
    }
  }
  return true;
}

// The reads that search1_text_kernel left for their 5 to 64 rows, a wavefront
// per read (with those of more rows, whose steps it takes in vain, 100 K reads
// of a repeat of 3000 copies took 1.3 ms here); one whose second pass has more
// goes on to search1_kernel, which takes a
// step per memory access (a read of a repeat then takes 0.3-1 ms from its
// first step to its last, which a launch waits for: with these reads there
// the batches above took 870 and 2370 us, and 700 K reads of 50-250 bases
// over 256 Mbp 1035 us for them alone, 41 here).
template <bool MM_ONLY>
__global__ __launch_bounds__(256) void search1_wave_kernel(S1tParams P) {
  __shared__ uint32_t slots[kReadRecordWords * 256u];
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  const uint32_t n = *P.wide_n;
  uint32_t *slot = slots + wave;
  for (uint32_t i = blockIdx.x * 4u + wave; i < n; i += gridDim.x * 4u) {
    const uint32_t rd = P.wide[i];
    const int32_t len = (int32_t)(P.offsets[rd + 1] - P.offsets[rd]);
    __builtin_amdgcn_wave_barrier();
    if (lane < kReadRecordWords) slot[lane * 256u] = P.rec[(uint64_t)rd * kReadRecordWords + lane];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
    __builtin_amdgcn_wave_barrier();
    const ReadBases<true> bases{nullptr, slot};
    bool left = false;
    for (uint32_t strand = 0; strand < 2u && !left; ++strand) {
      if (!((P.strand_mask >> strand) & 1u)) continue;
      const uint64_t t = 2ull * rd + strand;
      S1tOut O{P.hits + t * P.cap, P.cap, 0u, strand};
      for (uint32_t pass = 0; pass < 2u && !left; ++pass)
        left = !wave_pass<MM_ONLY>(P.ix, pass, strand, bases, len, O);
      if (lane == 0u) P.counts[t] = O.cnt;
    }
    if (left && lane == 0u) P.list[atomicAdd(P.list_n, 1u)] = rd;
  }
}

}  // namespace

hipError_t launch_search1_text(const DevIndex &ix, bool mm_only, uint32_t strand_mask,
                               const uint8_t *reads, const uint64_t *offsets, uint32_t nreads,
                               uint32_t cap, fmi_hit *hits, uint32_t *counts, uint32_t *rec,
                               uint32_t *wide, uint32_t *wide_n, uint32_t *long_n, uint32_t *list,
                               uint32_t *list_n, uint32_t cus, hipStream_t s) {
  S1tParams P{ix,     reads,  offsets, hits,   counts, rec,         wide,
              wide_n, long_n, list,    list_n, nreads, strand_mask, cap,
              rows_wide_m(ix.n)};
  const dim3 g((uint32_t)((2ull * nreads + 511u) / 512u));
  const dim3 w(std::min<uint32_t>((nreads + 3u) / 4u, cus * 6u));   // resident (24 KB of LDS each)
  const bool resident = g.x <= 2u * cus;   // two groups a CU at 4 waves
  if (mm_only) {
    if (resident) hipLaunchKernelGGL((search1_text_kernel<true, 4>), g, dim3(512), 0, s, P);
    else hipLaunchKernelGGL((search1_text_kernel<true, 6>), g, dim3(512), 0, s, P);
    hipLaunchKernelGGL(search1_wave_kernel<true>, w, dim3(256), 0, s, P);
  } else {
    if (resident) hipLaunchKernelGGL((search1_text_kernel<false, 4>), g, dim3(512), 0, s, P);
    else hipLaunchKernelGGL((search1_text_kernel<false, 6>), g, dim3(512), 0, s, P);
    hipLaunchKernelGGL(search1_wave_kernel<false>, w, dim3(256), 0, s, P);
  }
  return hipGetLastError();
}

}  // namespace fmi
