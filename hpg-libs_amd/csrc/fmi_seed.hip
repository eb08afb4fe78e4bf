// fmi_seed.hip -- exact seed mapping (fmi_seed_map_batch): bwt_map_exact_seed
// (bwt.c:1200-1294) for every seed of a batch of reads.
//
//   1. seeds per read, exclusive scan -> global seed numbering
//   2. one lane per seed: + strand backward search on BACKWARD, - strand
//      forward search on BACKWARD_REV (both over the seed's seed_len symbols),
//      the cumulative filter of bwt.c:1250-1269 (a signed 32-bit running
//      count, as the reference's `int actual_mappings`), rows to resolve,
//      and the rows of every 64 seeds
//   3. exclusive scan of those sums
//   4. the rows of 64 seeds (or, where some bring very many, of a tile of rows)
//      shared out in a wavefront: locate (getScompValue) on BACKWARD, binsearch
//      over the karyotype offsets, the contig-end check key + len <= offset[idx]
//      with len = seq_end - seq_start (one short, bwt.c:1214), region record.
#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstring>   // rocprim's texture_cache_iterator uses memset

#include <rocprim/rocprim.hpp>

#include <algorithm>
#include <cstdint>
#include <string>

#include "../../include/fmi.h"
#include "fmi_device.h"
#include "fmi_index.h"
#include "fmi_internal.h"
#include "fmi_kernels.h"
#include "fmi_vhelper.h"
#include "fmi_window.h"

namespace fmi {

namespace {

__global__ void seed_count_kernel(const uint64_t *offsets, uint32_t nreads, uint32_t seed_len,
                                  uint32_t stride, uint64_t *cnt) {
  for (uint64_t r = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; r <= nreads;
       r += (uint64_t)gridDim.x * blockDim.x) {
    uint64_t c = 0;
    if (r < nreads) {
      const uint64_t len = offsets[r + 1] - offsets[r];
      if (len >= seed_len) c = (len - seed_len) / stride + 1;
    }
    cnt[r] = c;
  }
}

// Largest r in [0, n) with base[r] <= g (base is non-decreasing, base[0] = 0).
__device__ __forceinline__ uint64_t owner(const uint64_t *base, uint64_t n, uint64_t g) {
  uint64_t lo = 0, hi = n;   // invariant: base[lo] <= g, answer in [lo, hi)
  while (hi - lo > 1) {
    const uint64_t mid = (lo + hi) / 2;
    if (base[mid] <= g) lo = mid;
    else hi = mid;
  }
  return lo;
}

// The last i in [lo, hi) with base[i] <= g (base is non-decreasing, base[lo] <=
// g), by 64 probes a round of the whole wavefront, whose lanes all call it with
// the same arguments.
__device__ __forceinline__ uint64_t wave_last(const uint64_t *base, uint64_t lo, uint64_t hi,
                                              uint64_t g) {
  const uint32_t lane = threadIdx.x & 63u;
  while (hi - lo > 1u) {
    const uint64_t step = (hi - lo + 63u) / 64u, idx = lo + lane * step;
    const uint64_t yes = __ballot(lane == 0u || (idx < hi && base[idx] <= g));
    lo += (63u - (uint32_t)__builtin_clzll(yes)) * step;
    hi = min(lo + step, hi);
  }
  return lo;
}

// owner for the lanes of a wavefront that hold consecutive g's (lane i:
// g0 + i, g0 + i < total): the owners of the first and the last by the whole
// wavefront, then a lane's own among those between them.  Every lane of the
// wavefront calls it; lanes past total get any answer.
__device__ __forceinline__ uint64_t wave_owner(const uint64_t *base, uint64_t n, uint64_t total,
                                               uint64_t g0) {
  const uint64_t a = wave_last(base, 0u, n, g0);
  const uint64_t b = wave_last(base, a, n, min(g0 + 63u, total - 1u));
  return a + owner(base + a, b - a + 1u, g0 + (threadIdx.x & 63u));
}

struct SeedParams {
  DevIndex ix;
  const uint8_t *reads;
  const uint64_t *offsets;
  const uint64_t *seed_base;   // nreads + 1
  uint64_t nseeds;
  uint32_t nreads, seed_len, stride;
  int32_t filter;
  fmi_seed_info *info;         // may be NULL
  uint64_t info_cap;
  // 2 * nseeds, + then - of every seed: x the first row (or the one row's text
  // position), y the rows (or kRowKnown)
  uint2 *slots;
  uint64_t *sums;              // rows of seeds 64 i .. 64 i + 63
  unsigned long long *most;    // the largest of them, if above kSeedBlockRows
};

// Rows of 64 seeds that one wavefront locates (seed_rows_kernel).
constexpr uint32_t kSeedBlockRows = 2048;

__device__ __forceinline__ void put_sum(const SeedParams &P, uint64_t i, uint64_t sum) {
  P.sums[i] = sum;
  if (sum > kSeedBlockRows) atomicMax(P.most, (unsigned long long)sum);
}

// A slot with one row whose text position is known (rows are below 2^32 - 2).
constexpr uint32_t kRowKnown = 0xFFFFFFFFu;

// The cumulative filter with the reference's int arithmetic (bwt.c:1250-1269)
// over the rows cp, cm of the + and - strands: the rows kept of each.
__device__ __forceinline__ void seed_filter(int32_t filter, uint64_t cp, uint64_t cm, uint32_t &rp,
                                            uint32_t &rm) {
  int32_t actual = (int32_t)(uint32_t)cp;
  rp = actual > filter ? 0u : (uint32_t)cp;
  actual = (int32_t)((uint32_t)actual + (uint32_t)cm);
  rm = actual > filter ? 0u : (uint32_t)cm;
}

// The sum of v over the wavefront's lanes, in every lane.
__device__ __forceinline__ uint64_t wave_sum(uint64_t v) {
  unsigned long long x = v;
#pragma unroll
  for (uint32_t d = 32u; d >= 1u; d >>= 1) x += __shfl_xor(x, (int)d);
  return x;
}

// REGS (seed_len <= 32): the seed's bases are packed into registers once
// (vh_regs) and every base below comes from there, not from a byte load.
template <bool REGS>
__global__ __launch_bounds__(256) void seed_search_kernel(SeedParams P) {
  const DevDir &D = P.ix.d[0];
  const uint32_t n = P.ix.n;
  const uint32_t lane = threadIdx.x & 63u;
  for (uint64_t g0 = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x - lane; g0 < P.nseeds;
       g0 += (uint64_t)gridDim.x * blockDim.x) {
    const uint64_t own = wave_owner(P.seed_base, P.nreads, P.nseeds, g0);
    const uint64_t g = g0 + lane;
    uint32_t rp = 0u, rm = 0u;
    if (g < P.nseeds) {
      const uint64_t r = own;
      const uint64_t s = (g - P.seed_base[r]) * P.stride;
      const uint8_t *W = P.reads + P.offsets[r] + s;
      VhRegs WR{0ull, 0u, 0};
      if (REGS) WR = vh_regs(W, 0, P.seed_len);
      auto base = [&](int32_t i) -> uint32_t { return REGS ? WR.at(i) : (uint32_t)W[i]; };
      // The first k steps of each search from the k-mer table when its k bases
      // are A/C/G/T and their interval is not empty (else step by step, so a
      // dead interval is the one the LF steps give).
      const uint32_t K = P.ix.kmer_k;
      const bool use_k = K && P.seed_len >= K;
      // + strand: BWExactSearchBackward over W[0 .. seed_len-1] on BACKWARD
      uint32_t kp = 0, lp = n;
      int32_t ip = (int32_t)P.seed_len - 1;
      // - strand: BWExactSearchForward on BACKWARD_REV (complemented symbols)
      uint32_t km = 0, lm = n;
      uint32_t im = 0;
      if (use_k) {
        uint32_t cp = 0u, cm = 0u, bad = 0u;
        for (uint32_t j = 0; j < K; ++j) {
          const uint32_t sp = base(ip - (int32_t)j), sm = base((int32_t)j);
          bad |= (sp > 3u || sm > 3u) ? 1u : 0u;
          cp |= (sp & 3u) << (2u * j);
          cm |= (sm & 3u) << (2u * j);
        }
        cm ^= (1u << (2u * K)) - 1u;
        if (!bad) {
          const uint64_t ep = P.ix.kmer[0][cp], em = P.ix.kmer[0][cm];
          if ((uint32_t)ep <= (uint32_t)(ep >> 32)) {
            kp = (uint32_t)ep; lp = (uint32_t)(ep >> 32); ip -= (int32_t)K;
          }
          if ((uint32_t)em <= (uint32_t)(em >> 32)) {
            km = (uint32_t)em; lm = (uint32_t)(em >> 32); im = K;
          }
        }
      }
      for (int32_t i = ip; i >= 0; --i) {
        uint32_t kn, ln;
        if (lf_sym(D, kp, lp, base(i), 0u, kn, ln) > 3u) { kp = n + 1; lp = n; break; }
        kp = kn; lp = ln;
        if (kp > lp) break;
      }
      for (uint32_t i = im; i < P.seed_len; ++i) {
        uint32_t kn, ln;
        if (lf_sym(D, km, lm, base((int32_t)i), 1u, kn, ln) > 3u) { km = n + 1; lm = n; break; }
        km = kn; lm = ln;
        if (km > lm) break;
      }
      seed_filter(P.filter, kp <= lp ? (uint64_t)lp - kp + 1u : 0u,
                  km <= lm ? (uint64_t)lm - km + 1u : 0u, rp, rm);
      P.slots[2 * g] = make_uint2(kp, rp);
      P.slots[2 * g + 1] = make_uint2(km, rm);
      if (P.info && g < P.info_cap) {
        fmi_seed_info inf;
        inf.k_plus = kp; inf.l_plus = lp; inf.k_minus = km; inf.l_minus = lm;
        inf.rows_plus = rp; inf.rows_minus = rm;
        P.info[g] = inf;
      }
    }
    const uint64_t sum = wave_sum((uint64_t)rp + rm);
    if (lane == 0u) put_sum(P, g0 >> 6, sum);
  }
}

// The same on an index with row contexts and a k-mer table, for seeds of
// kmer_k to 32 bases whose intervals are not asked for (no d_seed_info: where
// and how an absent seed's search dies is not seen).  A strand is a table
// entry, the contexts of its rows (those that go on with the seed's last
// bases) and, for a strand that occurs, the first row's suffix -- its position
// if it is the only one, else the row of it in the final interval.
// Bound by random lines: 2 entries, 2-3 of contexts and about one of SA a seed,
// where the entry and one or two occurrence blocks per base after it took
// about 9.  47 M seeds of 18 bases over 3.1 Gbp: 9.4 ms, 7.2 with the strands'
// contexts read one after the other, 6.5 as below (42 G lines/s, of the 47-50
// that a gather over this much memory reaches).
__global__ __launch_bounds__(256) void seed_context_kernel(SeedParams P) {
  const DevDir &D = P.ix.d[0];
  const uint32_t lane = threadIdx.x & 63u, K = P.ix.kmer_k, L = P.seed_len;
  for (uint64_t g0 = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x - lane; g0 < P.nseeds;
       g0 += (uint64_t)gridDim.x * blockDim.x) {
    const uint64_t r = wave_owner(P.seed_base, P.nreads, P.nseeds, g0);
    const uint64_t g = g0 + lane;
    uint32_t rp = 0u, rm = 0u;
    if (g < P.nseeds) {
      const uint64_t s = (g - P.seed_base[r]) * P.stride;
      const VhRegs W = vh_regs(P.reads + P.offsets[r] + s, 0, L);
      const uint32_t nmask = L >= 32u ? ~0u : (1u << L) - 1u;
      WinIv v[2];
      v[0].rows = v[1].rows = 0u;
      if ((W.nfl & nmask) == 0u) {                 // an N occurs nowhere
        const uint64_t v64 = __builtin_bitreverse64(W.code);
        // + strand: W[L-1], W[L-2], ...; - strand: W[0], W[1], ... complemented
        const uint64_t code[2] = {(((v64 >> 1) & 0x5555555555555555ull) |
                                   ((v64 & 0x5555555555555555ull) << 1)) >> (64u - 2u * L),
                                  ~W.code};
        const uint32_t km = (1u << (2u * K)) - 1u;
        const uint64_t e[2] = {P.ix.kmer[0][(uint32_t)code[0] & km],
                               P.ix.kmer[0][(uint32_t)code[1] & km]};
        // both strands' first rows are read together where they lie in two
        // 16-byte pieces of contexts (almost all do), then both suffixes
        const uint32_t gs = L - K, gm = (uint32_t)win_mask(min(gs, 16u));
        uint4 c[2][2];
        bool near[2];
#pragma unroll
        for (uint32_t t = 0; t < 2u; ++t) {
          const uint32_t k = (uint32_t)e[t], l = (uint32_t)(e[t] >> 32);
          near[t] = k <= l && gs >= 1u && gs <= 16u && (k & 3u) + (l - k) < 8u && l - k < 8u;
          c[t][0] = c[t][1] = opaque4();
          const uint4 *p = reinterpret_cast<const uint4 *>(D.ctx + (k & ~3u));
          if (near[t]) {
            c[t][0] = p[0];
            if ((k & 3u) + (l - k) >= 4u) c[t][1] = p[1];
          }
        }
#pragma unroll
        for (uint32_t t = 0; t < 2u; ++t) {
          const uint32_t k = (uint32_t)e[t], l = (uint32_t)(e[t] >> 32);
          const uint64_t rest = code[t] >> (2u * K);
          if (!near[t]) {
            if (k > l || !win_extend(D, k, l, rest, gs, v[t])) v[t].rows = 0u;
            continue;
          }
          const uint32_t w[8] = {c[t][0].x, c[t][0].y, c[t][0].z, c[t][0].w,
                                 c[t][1].x, c[t][1].y, c[t][1].z, c[t][1].w};
          uint32_t hit = 0u;
#pragma unroll
          for (uint32_t i = 0; i < 8u; ++i) {
            const bool in = i >= (k & 3u) && i - (k & 3u) <= l - k;
            if (in && ((w[i] ^ (uint32_t)rest) & gm) == 0u &&
                win_real(D, (k & ~3u) + i, w[i], gs))
              hit |= 1u << i;
          }
          v[t].rows = (uint32_t)__builtin_popcount(hit);
          v[t].k = (k & ~3u) + (uint32_t)__builtin_ctz(hit | 0x100u);   // the first row before
        }
#pragma unroll
        for (uint32_t t = 0; t < 2u; ++t) {
          if (!near[t]) continue;
          v[t].q = kWinNone;
          if (v[t].rows) v[t].q = D.sa[v[t].k] - gs;
        }
      }
      seed_filter(P.filter, v[0].rows, v[1].rows, rp, rm);
#pragma unroll
      for (uint32_t t = 0; t < 2u; ++t) {
        const uint32_t rows = t ? rm : rp;
        uint2 slot = make_uint2(v[t].k, rows);
        if (rows && v[t].q != kWinNone) {
          if (rows == 1u) slot = make_uint2(v[t].q, kRowKnown);
          else slot.x = D.isa[v[t].q];
        }
        P.slots[2 * g + t] = slot;
      }
    }
    const uint64_t sum = wave_sum((uint64_t)rp + rm);
    if (lane == 0u) put_sum(P, g0 >> 6, sum);
  }
}

struct RowParams {
  DevIndex ix;
  const uint64_t *offsets;
  const uint64_t *seed_base;   // nreads + 1
  const uint64_t *sum_base;    // exclusive scan of the rows of 64 seeds each
  const uint2 *slots;          // as SeedParams
  const uint64_t *koff;        // kcount + 1
  const uint64_t *kstart;
  uint64_t nseeds, nrows;      // rows to write
  uint32_t nreads, seed_len, stride, kcount;
  uint32_t tile;               // rows of a wavefront, a multiple of 64
  fmi_seed_region *out;
};

// The region of one row at text position key.
__device__ __forceinline__ void store_row(const RowParams &P, uint64_t row, uint64_t key,
                                          uint32_t sid, uint32_t read, uint32_t seq_len,
                                          uint32_t strand) {
  const uint64_t seq_start = (uint64_t)sid * P.stride;
  const uint64_t seq_end = seq_start + P.seed_len - 1;
  const uint64_t len = seq_end - seq_start;
  uint64_t lo = 0, size = P.kcount;            // binsearch, search/io.h:43-64
  while (size > 0) {
    const uint64_t w = size / 2;
    if (P.koff[lo + w] <= key) { lo += w + 1; size -= w + 1; }
    else size = w;
  }
  uint64_t start = 0, end = 0;
  uint32_t valid = 0u;
  if (lo >= 1 && key + len <= P.koff[lo]) {
    start = P.kstart[lo - 1] + (key - P.koff[lo - 1]) + 1;
    end = start + len;
    valid = 1u;
  }
  const uint32_t ss = (uint16_t)(strand ? seq_len - seq_end - 1 : seq_start);
  const uint32_t se = (uint16_t)(strand ? seq_len - seq_start - 1 : seq_end);
  uint4 *dst = reinterpret_cast<uint4 *>(P.out + row);
  dst[0] = make_uint4((uint32_t)start, (uint32_t)(start >> 32), (uint32_t)end,
                      (uint32_t)(end >> 32));
  dst[1] = make_uint4((uint32_t)lo, read, ss | (se << 16),
                      (uint32_t)(uint16_t)sid | (strand << 16) | (valid << 24));
}

// Rows row .. end - 1 of out, all of seeds 64 b .. 64 b + 63, shared out among
// the wavefront's lanes 64 at a time (every lane calls it).
__device__ __forceinline__ void block_rows(const RowParams &P, uint64_t b, uint64_t row,
                                           uint64_t end) {
  const DevDir &D = P.ix.d[0];
  const uint32_t lane = threadIdx.x & 63u;
  const uint64_t first = P.sum_base[b], g0 = 64u * b;
  const uint64_t own = wave_owner(P.seed_base, P.nreads, P.nseeds, g0);
  uint4 sl = make_uint4(0u, 0u, 0u, 0u);           // + and - of the lane's seed
  uint32_t seed = 0u, rd = 0u, rlen = 0u;
  if (g0 + lane < P.nseeds) {
    sl = reinterpret_cast<const uint4 *>(P.slots)[g0 + lane];
    rd = (uint32_t)own;
    seed = (uint32_t)(g0 + lane - P.seed_base[own]);
    rlen = (uint32_t)(P.offsets[own + 1] - P.offsets[own]);
  }
  const uint32_t rp = sl.y == kRowKnown ? 1u : sl.y, rm = sl.w == kRowKnown ? 1u : sl.w;
  const uint64_t rows = (uint64_t)rp + rm;
  unsigned long long incl = rows;                  // rows of lanes 0..i
#pragma unroll
  for (uint32_t d = 1u; d < 64u; d <<= 1) {
    const unsigned long long v = __shfl_up(incl, d);
    if (lane >= d) incl += v;
  }
  const unsigned long long excl = incl - rows;
  for (; row < end; row += 64u) {
    const unsigned long long t = row - first + lane;
    uint32_t o = 0u;                               // the first lane whose rows reach past t
#pragma unroll
    for (uint32_t d = 32u; d >= 1u; d >>= 1)
      if (__shfl(incl, (int)(o + d - 1u)) <= t) o += d;
    const int src = (int)min(o, 63u);
    uint64_t j = t - __shfl(excl, src);
    const uint32_t np = __shfl(rp, src);
    const uint32_t strand = j >= np ? 1u : 0u;
    const uint32_t px = __shfl(sl.x, src), py = __shfl(sl.y, src);
    const uint32_t mx = __shfl(sl.z, src), my = __shfl(sl.w, src);
    const uint32_t sid = __shfl(seed, src), read = __shfl(rd, src), seq_len = __shfl(rlen, src);
    if (row + lane >= end) continue;
    if (strand) j -= np;
    const uint32_t x = strand ? mx : px;
    const bool known = (strand ? my : py) == kRowKnown;
    const uint64_t key = known ? x : sa_value(D, P.ix.ratio, P.ix.n, (uint32_t)(x + j));
    store_row(P, row + lane, key, sid, read, seq_len, strand);
  }
}

// A wavefront takes the rows of 64 seeds, which are neighbours in out.  Bound by
// the slots read and the regions written (and a line of SA per row that the
// search did not locate); a thread per row took a binary search over the
// scanned row counts, 27 dependent loads for 94 M slots: 57 M rows in 3.2 ms
// (and 0.6 to scan the counts), 2.0 as below.
// TILED: a wavefront takes `tile` neighbouring rows instead, of as many seeds as
// they are.  A batch is taken so where some 64 seeds bring more than
// kSeedBlockRows rows and 4 times what a wavefront of a full device (8192) has
// on average: the rows of one wavefront are a chain, 0.95 us per 64 (6.5 on a
// compact index), and a single seed of 2 M rows took 29.4 ms (203), 0.10 (0.19)
// by tiles.  Elsewhere tiles look most of the 64 seeds up twice: 1.7 M seeds of
// 18 bases, a row each, on a compact index 1.16 ms, 1.35 by tiles.
template <bool TILED>
__global__ __launch_bounds__(256) void seed_rows_kernel(RowParams P) {
  const uint64_t nsums = (P.nseeds + 63u) / 64u;
  const uint64_t wave = ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const uint64_t waves = (uint64_t)gridDim.x * (blockDim.x >> 6);
  if (!TILED) {
    for (uint64_t b = wave; b < nsums; b += waves) {
      const uint64_t row = P.sum_base[b], end = min(P.sum_base[b + 1u], P.nrows);
      if (row < end) block_rows(P, b, row, end);
    }
    return;
  }
  for (uint64_t at = wave * P.tile; at < P.nrows; at += waves * P.tile) {
    const uint64_t last = min(at + P.tile, P.nrows);
    uint64_t row = at, b = wave_last(P.sum_base, 0u, nsums, at);
    for (;;) {
      const uint64_t end = min(P.sum_base[b + 1u], last);
      block_rows(P, b, row, end);
      if (end == last) break;
      row = end;
      b = P.sum_base[b + 2u] > row ? b + 1u : wave_last(P.sum_base, b + 1u, nsums, row);
    }
  }
}
static_assert(sizeof(fmi_seed_region) == 32 && offsetof(fmi_seed_region, chrom_idx) == 16 &&
                  offsetof(fmi_seed_region, seq_start) == 24 &&
                  offsetof(fmi_seed_region, seed_id) == 28 &&
                  offsetof(fmi_seed_region, strand) == 30 &&
                  offsetof(fmi_seed_region, valid) == 31,
              "fmi_seed_region layout");

// ---------------------------------------------------------------- inexact seeds
// bwt_map_inexact_seeds_seq (bwt.c:3262-3302) + bwt_map_inexact_seed
// (bwt.c:1401-1644):
//   1. windows per read (len / seed_size, plus the remainder when it holds
//      at least min_seed_size bases), exclusive scan -> window numbering
//   2. one lane per window (persistent grid): the vector helper on the +
//      strand then the - strand (final_pos carries over between them), each
//      record turned into regions as it is produced (the reference makes the
//      records first and then walks them in the same order), straight into
//      the caller's slot; then the slot's dedup and reversal in place.

__global__ void win_count_kernel(const uint64_t *offsets, uint32_t nreads, uint32_t seed_size,
                                 uint32_t min_seed_size, uint64_t *cnt) {
  for (uint64_t r = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; r <= nreads;
       r += (uint64_t)gridDim.x * blockDim.x) {
    uint64_t c = 0;
    if (r < nreads) {
      const uint64_t len = offsets[r + 1] - offsets[r];
      c = len / seed_size + (len % seed_size >= min_seed_size ? 1 : 0);
    }
    cnt[r] = c;
  }
}

struct InexactParams {
  DevIndex ix;
  const uint8_t *reads;
  const uint64_t *offsets;
  const uint64_t *win_base;    // nreads + 1
  uint64_t nwin;
  uint32_t nreads, seed_size, rec_cap, region_cap;
  const uint64_t *koff;        // kcount + 1
  const uint64_t *kstart;
  uint32_t kcount;
  uint2 *vscratch;             // lanes * (seed_size + 3)
  uint32_t min_len;            // context_seed_kernel: shorter windows are left
  uint32_t *list, *list_n;     // the list of the windows left
  fmi_inexact_region *out;     // 2 * nwin * region_cap
  uint32_t *nreg;
  uint8_t *status;
};

// What a record says of its error, as the list stores it (no error fields
// without an error): final_pos where it is assigned, the change of the length
// and final_err (bwt.c:1499-1530).
__device__ __forceinline__ void record_errors(const VhRec &r, uint32_t type, int32_t len,
                                              int32_t &final_pos, int32_t &dl,
                                              int32_t &final_err) {
  const uint32_t error = r.nmm ? r.kind : 0u;
  const int32_t pos = r.nmm ? r.err_pos : 0;
  dl = error == FMI_DELETION ? -1 : (error == FMI_INSERTION ? 1 : 0);
  if (error == FMI_DELETION || pos == 0 || pos == len - 1) {
    final_pos = type ? pos : len - 1 - pos;
  } else if (error == FMI_INSERTION) {
    if (type) final_pos = r.dir ? pos : pos + 1;
    else final_pos = r.dir ? len - pos : len - pos - 1;
  }
  // -1 mismatch, SEED_INSERTION 1, SEED_DELETION 2
  final_err = error == FMI_MISMATCH ? -1 : (error == FMI_DELETION ? 1 : 2);
}

// Regions of one strand's records (bwt.c:1490-1588), in record order.
struct RegionSink {
  const InexactParams *P;
  fmi_inexact_region *out;
  uint32_t m, nrec, type, read, aux_s, aux_e, seq_len, seed_id;
  int32_t start, len;
  int32_t *final_pos;
  uint8_t st;
  __device__ __forceinline__ bool full() const { return false; }   // its caps are counted past
  __device__ __forceinline__ void add(const VhRec &r) {
    add(r, (type ? r.dir : !r.dir) ? 1u : 0u, WinIv{r.k, kWinNone, r.l - r.k + 1u});
  }
  // The record's interval on direction dsel: its first row, or that row's
  // suffix, and its rows.
  __device__ __forceinline__ void add(const VhRec &r, uint32_t dsel, const WinIv &iv) {
    if (nrec++ >= P->rec_cap) { st |= 1; return; }   // the reference's list holds 20000
    int32_t dl, final_err;
    record_errors(r, type, len, *final_pos, dl, final_err);
    final_err += start;
    const int64_t len_calc = (int64_t)len + dl;
    const DevDir &D = dir_of(P->ix, dsel);
    const uint32_t rows = iv.rows < 50u ? iv.rows : 2u;    // bwt.c:1539-1547
    const uint32_t k = iv.q != kWinNone && rows > 1u ? D.isa[iv.q] : iv.k;
    const uint64_t size_sa = (uint64_t)P->ix.n + 1;
    for (uint32_t j = 0; j < rows; ++j) {
      const uint64_t sa = iv.q != kWinNone && j == 0u ? iv.q
                                                      : sa_value(D, P->ix.ratio, P->ix.n, k + j);
      const uint64_t key = dsel ? size_sa - sa - (uint64_t)len_calc - 1 : sa;
      uint64_t lo = 0, size = P->kcount;    // binsearch, search/io.h:43-64
      while (size > 0) {
        const uint64_t w = size / 2;
        if (P->koff[lo + w] <= key) { lo += w + 1; size -= w + 1; }
        else size = w;
      }
      if (!(lo >= 1 && key + (uint64_t)len_calc <= P->koff[lo])) continue;
      if (m >= P->region_cap) { st |= 2; continue; }
      fmi_inexact_region R;
      R.start = P->kstart[lo - 1] + (key - P->koff[lo - 1]) + 1;
      R.end = R.start + (uint64_t)len - 1;
      R.chrom_idx = (uint32_t)lo;
      R.read = read;
      R.seq_start = (uint16_t)aux_s;
      R.seq_end = (uint16_t)aux_e;
      R.seq_len = (uint16_t)seq_len;
      R.seed_id = (uint16_t)seed_id;
      R.pos_err = *final_pos;
      R.type_err = final_err;
      R.strand = (uint8_t)(1u - type);
      for (int b = 0; b < 7; ++b) R.pad[b] = 0;
      out[m++] = R;
    }
  }
};

// A lane's m regions at out deduplicated within 10 bp (bwt.c:1593-1615), the
// mark kept in pad[0], and handed over from the last to the first
// (bwt.c:1616-1626), in place; returns how many stay.
__device__ __forceinline__ uint32_t dedup_list(fmi_inexact_region *out, uint32_t m) {
  for (int32_t a1 = (int32_t)m - 1; a1 >= 1; --a1) {
    if (out[a1].pad[0]) continue;
    const uint64_t s1 = out[a1].start;
    const uint32_t c1 = out[a1].chrom_idx;
    for (int32_t a2 = a1 - 1; a2 >= 0; --a2) {
      const int32_t d = (int32_t)(uint32_t)(s1 - out[a2].start);
      const int64_t dist = d < 0 ? -(int64_t)d : (int64_t)d;
      if (c1 == out[a2].chrom_idx && dist < 10 && !out[a2].pad[0]) out[a2].pad[0] = 1;
    }
  }
  uint32_t kept = 0;
  for (uint32_t i = 0; i < m; ++i) {
    if (out[i].pad[0]) continue;
    const fmi_inexact_region R = out[i];
    out[kept++] = R;
  }
  for (uint32_t i = 0; i < kept / 2; ++i) {
    const fmi_inexact_region x = out[i];
    out[i] = out[kept - 1 - i];
    out[kept - 1 - i] = x;
  }
  return kept;
}

// ---- windows by row contexts: the records of a window and strand are kept
// (16 bytes each) and become regions together, one region a lane.
constexpr uint32_t kWinRecs = 64;      // rows of its records that a wavefront takes at once
constexpr uint8_t kWinLeft = 0x80;     // status of a window with more of them

// A kept record: x the first row, or (known) that row's suffix; y its rows (as
// many as it gives regions for) | known << 8 | direction << 9 | (len_calc - len
// + 1) << 10; z pos_err, w type_err.
struct RecordSink {
  uint4 *list;
  uint32_t n, total, nrec, rec_cap, type;
  int32_t start, len;
  int32_t final_pos;
  uint8_t st;
  __device__ __forceinline__ bool full() const { return total > kWinRecs; }
  __device__ __forceinline__ void add(const VhRec &r, uint32_t dsel, const WinIv &iv) {
    if (nrec++ >= rec_cap) { st |= 1; return; }      // the reference's list holds 20000
    int32_t dl, final_err;
    record_errors(r, type, len, final_pos, dl, final_err);
    const uint32_t rows = iv.rows < 50u ? iv.rows : 2u;        // bwt.c:1539-1547
    const bool known = iv.q != kWinNone;
    const uint4 v = make_uint4(known ? iv.q : iv.k,
                               rows | (known ? 1u << 8 : 0u) | (dsel << 9) |
                                   ((uint32_t)(dl + 1) << 10),
                               (uint32_t)final_pos, (uint32_t)(final_err + start));
    if (n < kWinRecs) list[n] = v;
    n++;
    total += rows;
  }
};

// The region of row j of a kept record: its start and contig, or contig 0
// where the occurrence crosses a contig's end.
__device__ __forceinline__ void record_region(const InexactParams &P, const uint4 &rec, uint32_t j,
                                              int32_t len, uint64_t &start, uint32_t &chrom) {
  const uint32_t dsel = (rec.y >> 9) & 1u, rows = rec.y & 0xFFu;
  const bool known = ((rec.y >> 8) & 1u) != 0u;
  const DevDir &D = dir_of(P.ix, dsel);
  const uint64_t len_calc = (uint64_t)((int64_t)len + (int64_t)((rec.y >> 10) & 3u) - 1);
  uint32_t sa;
  if (known && j == 0u) sa = rec.x;
  else sa = D.sa[(known && rows > 1u ? D.isa[rec.x] : rec.x) + j];
  const uint64_t key = dsel ? (uint64_t)P.ix.n + 1u - sa - len_calc - 1u : (uint64_t)sa;
  uint64_t lo = 0, size = P.kcount;        // binsearch, search/io.h:43-64
  while (size > 0) {
    const uint64_t w = size / 2;
    if (P.koff[lo + w] <= key) { lo += w + 1; size -= w + 1; }
    else size = w;
  }
  chrom = 0u;
  start = 0ull;
  if (lo >= 1 && key + len_calc <= P.koff[lo]) {
    chrom = (uint32_t)lo;
    start = P.kstart[lo - 1] + (key - P.koff[lo - 1]) + 1;
  }
}

struct WinOf {                       // what a window's regions have in common
  uint32_t read, aux_s, aux_e, seq_len, seed_id, strand;
  int32_t len;
};

// A region as three 16-byte pieces.
__device__ __forceinline__ void store_region(fmi_inexact_region *dst, const WinOf &w,
                                             uint64_t start, uint32_t chrom, const uint4 &rec,
                                             uint32_t mark) {
  const uint64_t end = start + (uint64_t)(int64_t)w.len - 1u;
  uint4 *d = reinterpret_cast<uint4 *>(dst);
  d[0] = make_uint4((uint32_t)start, (uint32_t)(start >> 32), (uint32_t)end, (uint32_t)(end >> 32));
  d[1] = make_uint4(chrom, w.read, w.aux_s | (w.aux_e << 16), w.seq_len | (w.seed_id << 16));
  d[2] = make_uint4(rec.z, rec.w, w.strand | (mark << 8), 0u);
}
static_assert(sizeof(fmi_inexact_region) == 48 && offsetof(fmi_inexact_region, chrom_idx) == 16 &&
                  offsetof(fmi_inexact_region, seq_start) == 24 &&
                  offsetof(fmi_inexact_region, pos_err) == 32 &&
                  offsetof(fmi_inexact_region, strand) == 40,
              "fmi_inexact_region layout");

__device__ __forceinline__ uint32_t lane_value(uint32_t v, int src) {
  return (uint32_t)__builtin_amdgcn_readlane((int)v, src);
}

// Turns every lane's kept records (n of them with `total` rows, at most
// kWinRecs; n = 0: none) into its slot's list: the regions in record and row
// order, the dedup, the hand-over from the last to the first.  A lane with one
// row does it alone, all such lanes together; any other list is taken by the
// whole wavefront, a row a lane, and leaves the registers once.  Slots past
// the list hold what the list held there before the hand-over, marked in
// pad[0] where it was dropped.  Every lane of the wavefront calls it; returns
// the regions kept.
__device__ __forceinline__ uint32_t regions_of(const InexactParams &P, const RecordSink &S,
                                               uint32_t n, const WinOf &w,
                                               fmi_inexact_region *out, uint8_t &st) {
  const uint32_t lane = threadIdx.x & 63u;
  uint32_t kept = 0u;
  if (n == 1u && S.total == 1u) {
    uint64_t start;
    uint32_t chrom;
    const uint4 rec = S.list[0];
    record_region(P, rec, 0u, w.len, start, chrom);
    if (chrom) {
      store_region(out, w, start, chrom, rec, 0u);
      kept = 1u;
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");   // the lists, read by other lanes
  for (uint64_t todo = __ballot(n > 0u && S.total > 1u); todo; todo &= todo - 1ull) {
    const int src = (int)__builtin_ctzll(todo);
    const uint4 *list = reinterpret_cast<const uint4 *>(
        ((uint64_t)lane_value((uint32_t)((uintptr_t)S.list >> 32), src) << 32) |
        lane_value((uint32_t)(uintptr_t)S.list, src));
    fmi_inexact_region *dst = reinterpret_cast<fmi_inexact_region *>(
        ((uint64_t)lane_value((uint32_t)((uintptr_t)out >> 32), src) << 32) |
        lane_value((uint32_t)(uintptr_t)out, src));
    const uint32_t nr = lane_value(n, src);
    const WinOf ws{lane_value(w.read, src),    lane_value(w.aux_s, src),
                   lane_value(w.aux_e, src),   lane_value(w.seq_len, src),
                   lane_value(w.seed_id, src), lane_value(w.strand, src),
                   (int32_t)lane_value((uint32_t)w.len, src)};
    uint4 rec = make_uint4(0u, 0u, 0u, 0u);
    if (lane < nr) rec = list[lane];
    uint32_t incl = rec.y & 0xFFu;             // rows of records 0..lane
    const uint32_t own = incl;
#pragma unroll
    for (uint32_t d = 1u; d < 64u; d <<= 1) {
      const uint32_t v = __shfl_up(incl, d);
      if (lane >= d) incl += v;
    }
    uint32_t ri = 0u;                          // the record of row `lane`
#pragma unroll
    for (uint32_t d = 32u; d >= 1u; d >>= 1)
      if (__shfl(incl, (int)(ri + d - 1u)) <= lane) ri += d;
    const uint32_t rows = lane_value(incl, 63);
    const int at = (int)min(ri, 63u);
    const uint32_t first = __shfl(incl - own, at);
    const uint4 mine = make_uint4(__shfl(rec.x, at), __shfl(rec.y, at), __shfl(rec.z, at),
                                  __shfl(rec.w, at));
    uint64_t start = 0ull;
    uint32_t chrom = 0u;
    if (lane < rows) record_region(P, mine, lane - first, ws.len, start, chrom);
    const uint64_t below = (1ull << lane) - 1ull;
    const uint64_t valid = __ballot(chrom != 0u);
    const uint32_t rank = (uint32_t)__popcll(valid & below);
    const bool in = chrom != 0u && rank < P.region_cap;
    const uint64_t all = __ballot(in);
    // within 10 bp (bwt.c:1593-1615): from the last region to the first, one
    // not yet dropped drops every earlier one of its chromosome that near
    bool gone = !in;
    for (uint64_t left = all; left;) {
      const int a = 63 - (int)__builtin_clzll(left);
      left ^= 1ull << a;
      if (!((__ballot(!gone) >> a) & 1ull)) continue;
      const uint64_t s1 = ((uint64_t)lane_value((uint32_t)(start >> 32), a) << 32) |
                          lane_value((uint32_t)start, a);
      const int32_t d = (int32_t)(uint32_t)(s1 - start);
      const int64_t dist = d < 0 ? -(int64_t)d : (int64_t)d;
      if ((int)lane < a && lane_value(chrom, a) == chrom && dist < 10) gone = true;
    }
    const uint64_t stay = __ballot(!gone);
    const uint32_t k = (uint32_t)__popcll(stay);
    if (in && rank >= k) store_region(dst + rank, ws, start, chrom, mine, gone ? 1u : 0u);
    if (!gone)
      store_region(dst + (k - 1u - (uint32_t)__popcll(stay & below)), ws, start, chrom, mine, 0u);
    if ((int)lane == src) {
      kept = k;
      if ((uint32_t)__popcll(valid) > P.region_cap) st |= 2;
    }
  }
  return kept;
}

// Held to 128 VGPRs for 4 waves per SIMD (157 unbounded: 3 waves): a lane's
// windows are chains of dependent loads, so a fourth wave to hide them pays
// for the few registers spilled (83.3 -> 76.7 ms on 8 M windows of 18 bases
// over 64 Mbp).  REGS (seed_size <= 32): the window's bases are packed into
// registers once (vh_regs) for both strands, so the helper's LF steps and
// comparisons read no read bytes from memory.
// kWinsLeft: only the windows that context_seed_kernel left for their rows
// (kWinLeft), by their contexts too: with LF steps the longest of them took 0.6 ms
// more of 5.7 for 2 M windows over 64 Mbp.
// kWinsListed: P.list[0 .. *P.list_n), by LF steps: the windows left where some
// have fewer than min_len bases, in one launch with those (each kind is a few
// long chains, and launches one after the other take their sum).
enum : int { kWinsAll, kWinsLeft, kWinsListed };

template <bool REGS, int WHICH>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void inexact_seed_kernel(InexactParams P) {
  constexpr bool LEFT = WHICH == kWinsLeft, LISTED = WHICH == kWinsListed;
  __shared__ uint32_t words[LEFT ? kWinWords * 256u : 1u];
  const uint64_t lane = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  uint2 *vb = P.vscratch + lane * (uint64_t)(P.seed_size + 3);
  const uint64_t wlane = lane & 63u, count = LISTED ? (uint64_t)*P.list_n : P.nwin;
  // a wavefront's lanes take consecutive windows and go on together
  for (uint64_t g0 = lane - wlane; g0 < count; g0 += (uint64_t)gridDim.x * blockDim.x) {
    uint64_t g = g0 + wlane, rd = 0;
    if (!LISTED) rd = wave_owner(P.win_base, P.nreads, P.nwin, g0);
    if (g >= count || (LEFT && P.status[2 * g] != kWinLeft)) continue;
    if (LISTED) {
      g = P.list[g];
      rd = owner(P.win_base, P.nreads, g);
    }
    const uint64_t off = P.offsets[rd];
    const int32_t len = (int32_t)(P.offsets[rd + 1] - off);
    const int32_t w = (int32_t)(g - P.win_base[rd]);
    const int32_t num_seeds = len / (int32_t)P.seed_size;
    const int32_t ws = w * (int32_t)P.seed_size;
    const int32_t we = w < num_seeds ? ws + (int32_t)P.seed_size - 1 : len - 1;
    const bool run = we - ws >= 2;
    int32_t final_pos = 0;
    VhRegs WR{0ull, 0u, ws};
    if (REGS && run) WR = vh_regs(P.reads + off, ws, (uint32_t)(we - ws + 1));
    for (uint32_t s = 0; s < 2; ++s) {
      const uint32_t type = 1u - s;          // bwt.c:1460: type 1 (+) first
      const uint64_t slot = 2 * g + s;
      RegionSink S{&P, P.out + slot * P.region_cap, 0u, 0u, type, (uint32_t)rd,
                   type ? (uint32_t)ws : (uint32_t)(len - we - 1),
                   type ? (uint32_t)we : (uint32_t)(len - ws - 1), (uint32_t)len, (uint32_t)w,
                   ws, we - ws + 1, &final_pos, 0};
      if (run) {
        if (LEFT) win_run(P.ix, WR, ws, we, s, vb, words + threadIdx.x, S);
        else if (REGS) vh_run(P.ix, WR, ws, we, s, 0u, vb, S);
        else vh_run(P.ix, VhBytes{P.reads + off}, ws, we, s, 0u, vb, S);
      }
      P.nreg[slot] = dedup_list(S.out, S.m);
      P.status[slot] = S.st;
    }
  }
}

// The same windows on an index with row contexts, seed_size <= kWinMax: they go
// by their rows' contexts and the k-mer table instead of an LF step per base
// and branch (win_run), and their records become regions a wavefront at a time
// (regions_of).  A window with more than kWinRecs rows on a strand, or of fewer
// than min_len bases, is left to inexact_seed_kernel.  vscratch: per lane seed_size + 3 intervals and kWinRecs
// records.  At 4 waves per SIMD 31 registers spill; 3 waves (none) took 8.6 ms
// where 4 took 7.6, 5 waves 10.0 (before the loops were parted).
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void context_seed_kernel(InexactParams P) {
  __shared__ uint32_t words[kWinWords * 256u];
  const uint64_t lane = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const uint64_t lanes = (uint64_t)gridDim.x * blockDim.x;
  uint4 *list = reinterpret_cast<uint4 *>(P.vscratch) + lane * kWinRecs;
  uint2 *vb = reinterpret_cast<uint2 *>(reinterpret_cast<uint4 *>(P.vscratch) + lanes * kWinRecs) +
              lane * (uint64_t)(P.seed_size + 3);
  const uint64_t wlane = lane & 63u;
  // a wavefront's lanes take consecutive windows and go on together
  for (uint64_t g0 = lane - wlane; g0 < P.nwin; g0 += lanes) {
    const uint64_t rd0 = wave_owner(P.win_base, P.nreads, P.nwin, g0);
    const bool mine = g0 + wlane < P.nwin;
    const uint64_t g = mine ? g0 + wlane : P.nwin - 1u, rd = mine ? rd0 : P.nreads - 1u;
    const uint64_t off = P.offsets[rd];
    const int32_t len = (int32_t)(P.offsets[rd + 1] - off);
    const int32_t w = (int32_t)(g - P.win_base[rd]);
    const int32_t num_seeds = len / (int32_t)P.seed_size;
    const int32_t ws = w * (int32_t)P.seed_size;
    const int32_t we = w < num_seeds ? ws + (int32_t)P.seed_size - 1 : len - 1;
    const bool any = mine && we - ws >= 2, run = any && (uint32_t)(we - ws + 1) >= P.min_len;
    int32_t final_pos = 0;
    bool left = any && !run;
    VhRegs WR{0ull, 0u, ws};
    if (run) WR = vh_regs(P.reads + off, ws, (uint32_t)(we - ws + 1));
    for (uint32_t s = 0; s < 2; ++s) {
      const uint32_t type = 1u - s;          // bwt.c:1460: type 1 (+) first
      const uint64_t slot = 2 * g + s;
      RecordSink S{list, 0u, 0u, 0u, P.rec_cap, type, ws, we - ws + 1,
                   final_pos, 0};
      if (run) win_run(P.ix, WR, ws, we, s, vb, words + threadIdx.x, S);
      final_pos = S.final_pos;
      left |= S.full();
      const WinOf wo{(uint32_t)rd,
                     (uint32_t)(uint16_t)(type ? ws : len - we - 1),
                     (uint32_t)(uint16_t)(type ? we : len - ws - 1),
                     (uint32_t)(uint16_t)len,
                     (uint32_t)(uint16_t)w,
                     s,
                     we - ws + 1};
      uint8_t st = S.st;
      const uint32_t kept =
          regions_of(P, S, left ? 0u : S.n, wo, P.out + slot * P.region_cap, st);
      if (mine) {
        P.nreg[slot] = kept;
        P.status[slot] = st;
      }
    }
    if (left) P.status[2 * g] = kWinLeft;
  }
}

// The windows that context_seed_kernel left, in the order of their numbers within
// a group's 4096: appended to list with an atomic per group.
__global__ __launch_bounds__(256) void left_windows_kernel(InexactParams P) {
  __shared__ uint32_t waves[4], base;
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  const uint64_t g0 = (uint64_t)blockIdx.x * 4096u + 16u * threadIdx.x;
  uint32_t marks = 0u;
  for (uint32_t j = 0; j < 16u; ++j)
    if (g0 + j < P.nwin && P.status[2 * (g0 + j)] == kWinLeft) marks |= 1u << j;
  const uint32_t own = (uint32_t)__builtin_popcount(marks);
  uint32_t incl = own;
#pragma unroll
  for (uint32_t d = 1u; d < 64u; d <<= 1) {
    const uint32_t v = __shfl_up(incl, d);
    if (lane >= d) incl += v;
  }
  if (lane == 63u) waves[wave] = incl;
  __syncthreads();
  const uint32_t w0 = waves[0], w1 = waves[1], w2 = waves[2], all = w0 + w1 + w2 + waves[3];
  if (threadIdx.x == 0u && all) base = atomicAdd(P.list_n, all);
  __syncthreads();
  if (!own) return;
  uint32_t at = base + incl - own;
  at += (wave > 0u ? w0 : 0u) + (wave > 1u ? w1 : 0u) + (wave > 2u ? w2 : 0u);
  for (; marks; marks &= marks - 1u) P.list[at++] = (uint32_t)g0 + (uint32_t)__builtin_ctz(marks);
}

inline dim3 grid_for(uint64_t m) {
  uint64_t g = (m + 255) / 256;
  if (g > 65536ull * 4) g = 65536ull * 4;
  if (g == 0) g = 1;
  return dim3((uint32_t)g);
}

#define SEED_TRY(expr)                                            \
  do {                                                            \
    hipError_t e_ = (expr);                                       \
    if (e_ != hipSuccess) {                                       \
      *err = std::string(#expr) + ": " + hipGetErrorString(e_);   \
      rc = FMI_EDEVICE;                                           \
      goto done;                                                  \
    }                                                             \
  } while (0)

}  // namespace

int seed_map(const fmi_index *ix, const uint8_t *reads, const uint64_t *offsets, uint32_t nreads,
             uint32_t seed_len, uint32_t stride, uint32_t filter, fmi_seed_info *info,
             uint64_t info_cap, fmi_seed_region *regions, uint64_t region_cap, uint64_t *nseeds_out,
             uint64_t *nrows_out, void *stream, std::string *err) {
  hipStream_t s = static_cast<hipStream_t>(stream);
  int rc = FMI_OK;
  uint64_t *cnt = nullptr, *base = nullptr, *sums = nullptr;
  uint2 *slots = nullptr;
  void *tmp = nullptr;
  size_t tmp_bytes = 0, need = 0;
  uint64_t nseeds = 0, nsums = 0, totals[2] = {0, 0};   // rows; the most of 64 seeds
  *nseeds_out = 0;
  *nrows_out = 0;
  SEED_TRY(hipMalloc(&cnt, (uint64_t)(nreads + 1) * 8));
  SEED_TRY(hipMalloc(&base, (uint64_t)(nreads + 1) * 8));
  seed_count_kernel<<<grid_for(nreads + 1), 256, 0, s>>>(offsets, nreads, seed_len, stride, cnt);
  SEED_TRY(rocprim::exclusive_scan(nullptr, need, cnt, base, (uint64_t)0, (uint64_t)nreads + 1,
                                   rocprim::plus<uint64_t>(), s));
  tmp_bytes = need;
  SEED_TRY(hipMalloc(&tmp, tmp_bytes));
  SEED_TRY(rocprim::exclusive_scan(tmp, need, cnt, base, (uint64_t)0, (uint64_t)nreads + 1,
                                   rocprim::plus<uint64_t>(), s));
  SEED_TRY(hipMemcpyAsync(&nseeds, base + nreads, 8, hipMemcpyDeviceToHost, s));
  SEED_TRY(hipStreamSynchronize(s));
  *nseeds_out = nseeds;
  if (nseeds == 0) goto done;
  nsums = (nseeds + 63) / 64;
  SEED_TRY(hipMalloc(&slots, 2 * nseeds * sizeof(uint2)));
  SEED_TRY(hipMalloc(&sums, (nsums + 2) * 8));
  SEED_TRY(launch_zero(reinterpret_cast<uint32_t *>(sums + nsums + 1), 2, s));
  {
    SeedParams P{ix->dev, reads, offsets, base, nseeds, nreads, seed_len, stride,
                 (int32_t)(filter > (uint32_t)INT32_MAX ? INT32_MAX : filter), info, info_cap,
                 slots, sums, reinterpret_cast<unsigned long long *>(sums + nsums + 1)};
    const uint32_t K = ix->dev.kmer_k;
    if (!info && ix->dev.d[0].ctx && K && seed_len >= K && seed_len <= 32u)
      seed_context_kernel<<<grid_for(nseeds), 256, 0, s>>>(P);
    else if (seed_len <= 32u) seed_search_kernel<true><<<grid_for(nseeds), 256, 0, s>>>(P);
    else seed_search_kernel<false><<<grid_for(nseeds), 256, 0, s>>>(P);
  }
  SEED_TRY(hipGetLastError());
  // in place, one sum more (any value): the last entry is then the total
  SEED_TRY(rocprim::exclusive_scan(nullptr, need, sums, sums, (uint64_t)0, nsums + 1,
                                   rocprim::plus<uint64_t>(), s));
  if (need > tmp_bytes) {
    SEED_TRY(hipFree(tmp));
    tmp = nullptr;
    tmp_bytes = need;
    SEED_TRY(hipMalloc(&tmp, tmp_bytes));
  }
  SEED_TRY(rocprim::exclusive_scan(tmp, need, sums, sums, (uint64_t)0, nsums + 1,
                                   rocprim::plus<uint64_t>(), s));
  SEED_TRY(hipMemcpyAsync(totals, sums + nsums, 16, hipMemcpyDeviceToHost, s));
  SEED_TRY(hipStreamSynchronize(s));
  *nrows_out = totals[0];
  if (totals[0] && region_cap && regions) {
    // tiles of 512 rows (128 on a compact index, whose rows take 7 times as
    // long: 1.12 ms for 18 M of few seeds, 1.39 at 512), smaller where they
    // would be fewer wavefronts than fill the device twice
    const uint64_t rows = std::min(totals[0], region_cap);
    const uint32_t tile = (uint32_t)std::clamp<uint64_t>(rows / 16384 / 64 * 64, 64,
                                                         ix->dev.d[0].sa ? 512 : 128);
    RowParams R{ix->dev, offsets, base, sums, slots, ix->d_koffset, ix->d_kstart, nseeds,
                rows, nreads, seed_len, stride, (uint32_t)ix->kstart.size(), tile, regions};
    if (totals[1] > rows / 2048)
      seed_rows_kernel<true><<<grid_for((rows + tile - 1) / tile * 64), 256, 0, s>>>(R);
    else
      seed_rows_kernel<false><<<grid_for(nseeds), 256, 0, s>>>(R);
    SEED_TRY(hipGetLastError());
  }
done:
  if (rc == FMI_OK) {
    hipError_t e = hipStreamSynchronize(s);
    if (e != hipSuccess) { *err = hipGetErrorString(e); rc = FMI_EDEVICE; }
  }
  (void)hipFree(cnt);
  (void)hipFree(base);
  (void)hipFree(sums);
  (void)hipFree(slots);
  (void)hipFree(tmp);
  return rc;
}

int map_inexact_seeds(const fmi_index *ix, const uint8_t *reads, const uint64_t *offsets,
                      uint32_t nreads, uint32_t seed_size, uint32_t min_seed_size,
                      uint32_t rec_cap, uint32_t region_cap, uint64_t windows_cap,
                      fmi_inexact_region *regions, uint32_t *nregions, uint8_t *status,
                      uint64_t *nwindows, void *stream, std::string *err) {
  hipStream_t s = static_cast<hipStream_t>(stream);
  int rc = FMI_OK;
  uint64_t *cnt = nullptr, *base = nullptr;
  uint2 *vscr = nullptr;
  void *tmp = nullptr;
  size_t need = 0;
  uint64_t nwin = 0;
  *nwindows = 0;
  SEED_TRY(hipMalloc(&cnt, (uint64_t)(nreads + 1) * 8));
  SEED_TRY(hipMalloc(&base, (uint64_t)(nreads + 1) * 8));
  win_count_kernel<<<grid_for(nreads + 1), 256, 0, s>>>(offsets, nreads, seed_size,
                                                        min_seed_size, cnt);
  SEED_TRY(hipGetLastError());
  SEED_TRY(rocprim::exclusive_scan(nullptr, need, cnt, base, (uint64_t)0, (uint64_t)nreads + 1,
                                   rocprim::plus<uint64_t>(), s));
  SEED_TRY(hipMalloc(&tmp, need));
  SEED_TRY(rocprim::exclusive_scan(tmp, need, cnt, base, (uint64_t)0, (uint64_t)nreads + 1,
                                   rocprim::plus<uint64_t>(), s));
  SEED_TRY(hipMemcpyAsync(&nwin, base + nreads, 8, hipMemcpyDeviceToHost, s));
  SEED_TRY(hipStreamSynchronize(s));
  *nwindows = nwin;
  if (nwin > windows_cap) {
    *err = "the batch has " + std::to_string(nwin) + " windows, more than windows_cap";
    rc = FMI_ERANGE;
    goto done;
  }
  if (nwin == 0) goto done;
  {
    uint64_t lanes = (nwin + 255) / 256 * 256;
    const uint64_t per = (uint64_t)(seed_size + 3) * sizeof(uint2);
    const uint64_t max_lanes = std::min<uint64_t>(1ull << 19, ((1ull << 30) / per) / 256 * 256);
    if (lanes > max_lanes) lanes = max_lanes;
    // Windows by context where the table holds the first bases of their strings
    // (a base shorter than the window) and a string occurs in few places by
    // chance: at 1/16 row a string, or 1/256 where the table holds fewer than
    // log4 n bases.  By LF steps and by contexts, 100 K windows of 15 and 16 bases
    // over 64 Mbp: k = 15 1.98, 2.34 and 1.61, 1.10 ms; k = 12 1.99, 1.51 and
    // 1.60, 1.14; no table 1.97, 2.31 and 1.61, 1.81, and 1.29, 1.13 of 18 bases.
    const uint32_t K = ix->dev.kmer_k;
    uint32_t once = 0u;
    while ((1ull << (2u * once)) < ix->n) ++once;
    const uint32_t min_len = std::max(K + 1u, once + (K + 1u >= once ? 2u : 4u));
    // as many lanes as are resident (4 waves per SIMD), each with its record list
    // too, then the list of the windows left (numbers of 32 bits)
    bool ctx = ix->dev.d[0].ctx && seed_size <= kWinMax && seed_size >= min_len &&
               nwin < (1ull << 32);
    const bool some_short = ctx && min_seed_size < min_len;
    const uint64_t ctx_lanes = std::min<uint64_t>(lanes, 1ull << 18);
    const uint64_t lane_bytes =
        std::max<uint64_t>(lanes * per, ctx ? ctx_lanes * (per + kWinRecs * 16ull) : 0ull);
    hipError_t got = hipMalloc(&vscr, lane_bytes + (some_short ? 64ull + 4ull * nwin : 0ull));
    if (got != hipSuccess && ctx) {              // LF steps need 88 MB of the 310
      (void)hipGetLastError();
      ctx = false;
      got = hipMalloc(&vscr, lanes * per);
    }
    SEED_TRY(got);
    uint32_t *list = reinterpret_cast<uint32_t *>(reinterpret_cast<char *>(vscr) + lane_bytes);
    InexactParams P{ix->dev, reads, offsets, base, nwin, nreads, seed_size, rec_cap, region_cap,
                    ix->d_koffset, ix->d_kstart, (uint32_t)ix->kstart.size(), vscr, min_len,
                    list + 16, list, regions, nregions, status};
    // windows are at most seed_size bases (the remainder window is shorter)
    const dim3 grid((uint32_t)(lanes / 256));
    if (ctx) {
      context_seed_kernel<<<dim3((uint32_t)(ctx_lanes / 256)), 256, 0, s>>>(P);
      if (some_short) {
        SEED_TRY(launch_zero(list, 1, s));
        left_windows_kernel<<<dim3((uint32_t)((nwin + 4095) / 4096)), 256, 0, s>>>(P);
        inexact_seed_kernel<true, kWinsListed><<<grid, 256, 0, s>>>(P);
      } else {
        inexact_seed_kernel<true, kWinsLeft><<<grid, 256, 0, s>>>(P);
      }
    } else if (seed_size <= 32u) {
      inexact_seed_kernel<true, kWinsAll><<<grid, 256, 0, s>>>(P);
    } else {
      inexact_seed_kernel<false, kWinsAll><<<grid, 256, 0, s>>>(P);
    }
    SEED_TRY(hipGetLastError());
  }
done:
  if (rc == FMI_OK) {
    hipError_t e = hipStreamSynchronize(s);
    if (e != hipSuccess) { *err = hipGetErrorString(e); rc = FMI_EDEVICE; }
  }
  (void)hipFree(cnt);
  (void)hipFree(base);
  (void)hipFree(vscr);
  (void)hipFree(tmp);
  return rc;
}

}  // namespace fmi
