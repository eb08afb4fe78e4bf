// fmi_rows.h -- an exact search narrowed to a few rows' suffixes on an expanded
// index, shared by the kernels that go on with a read on the text.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "fmi_device.h"
#include "fmi_internal.h"
#include "fmi_window.h"

namespace fmi {

// The read's bases: from the thread's LDS slot (STAGED) or its bytes.
template <bool STAGED>
struct ReadBases {
  const uint8_t *W;
  const uint32_t *slot;
  __device__ __forceinline__ uint32_t at(int32_t p) const {
    return STAGED ? lds_base(slot, p) : (uint32_t)W[p];
  }
  // W[p], W[p + d], ... (cnt <= 16 of them) as 2-bit symbols, complemented
  // when comp is set; false when one is an N.
  __device__ __forceinline__ bool code(int32_t p, int32_t d, int32_t cnt, uint32_t comp,
                                       uint32_t &c) const {
    uint32_t bad = 0u;
    if (STAGED) {
      uint64_t w;
      uint32_t nb;
      lds_window(slot, p, d, w, nb);
      c = (uint32_t)w;
      bad = nb & ((1u << (uint32_t)cnt) - 1u);
    } else {
      c = 0u;
      for (int32_t j = 0; j < cnt; ++j) {
        const uint32_t s = W[p + j * d];
        bad |= s > 3u ? 1u : 0u;
        c |= (s & 3u) << (2u * (uint32_t)j);
      }
    }
    if (comp) c = ~c;
    c &= (uint32_t)win_mask((uint32_t)cnt);
    return bad == 0u;
  }
  // How many of the cnt bases W[p], W[p + d], ... equal the text before
  // suffix q.
  __device__ __forceinline__ int32_t match(const DevIndex &ix, uint32_t dsel, uint32_t comp,
                                           uint32_t q, int32_t p, int32_t d, int32_t cnt) const {
    int32_t done = 0;
    while (done < cnt) {
      const uint32_t lim = min(min((uint32_t)(cnt - done), STAGED ? 32u : 16u), q);
      if (lim == 0u) break;
      const uint32_t m = STAGED ? text_match32(ix, dsel, comp, q, slot, p + done * d, d, lim)
                                : text_match(ix, dsel, comp, q, W, p + done * d, d, lim);
      done += (int32_t)m;
      q -= m;
      if (m < lim) break;
    }
    return done;
  }
};

// An interval of more than kManyRows rows 8 bases past those that occur once by
// chance is that of a repeat of many alike copies: its reads are mostly searched
// elsewhere in the end, and every further step (an LF query) is in vain.
// 100 K reads of a repeat of 3000 exact copies: 42 us where they end here, 139
// with no end.  Fewer rows mostly narrow: of 4000 copies 10% apart, 411 us a
// call; 936 with an end at 64 rows, whose reads go the long way.
constexpr uint32_t kManyRows = 1024;

inline int32_t rows_wide_m(uint32_t n) {
  int32_t m = 8;
  for (uint64_t s = 1; s < n; s *= 4) ++m;
  return m;
}

enum : uint32_t { kRowsNone = 0u, kRowsFew = 1u, kRowsMany = 2u, kRowsCut = 3u };

// The search for the m0 bases W[p0], W[p0 + d], ... from the whole index:
// kRowsNone when they occur nowhere, kRowsFew with their rows' suffixes in R,
// kRowsMany when they have more than kTextRows rows (k..l).  The first bases
// come from the longest table they fill.  Then an interval of one row, or few
// without contexts, is compared with the text; one of up to kWinRows rows
// goes by its rows' contexts, 16 bases a look, which leaves few of a repeat's
// rows (and none of the rows that a k-mer has by chance) without a look at
// their suffixes; a wider one takes an LF step.  wide_m (rows_wide_m, for
// callers that do without such rows): a step to that many bases or more that
// leaves more than kManyRows rows ends the search with kRowsCut.
template <bool STAGED>
__device__ __forceinline__ uint32_t search_rows(const DevIndex &ix, uint32_t dsel, uint32_t comp,
                                                const ReadBases<STAGED> &rd, int32_t p0, int32_t d,
                                                int32_t m0, TextRows &R, uint32_t &k, uint32_t &l,
                                                int32_t wide_m = INT32_MAX) {
  const DevDir &D = dir_of(ix, dsel);
  const int32_t K = (int32_t)ix.kmer_k <= m0
                        ? (int32_t)ix.kmer_k
                        : ((int32_t)ix.kmer2_k <= m0 ? (int32_t)ix.kmer2_k : 0);
  k = 0u;
  l = ix.n;
  int32_t m = 0;
  if (K) {
    uint32_t c;
    if (!rd.code(p0, d, K, comp, c)) return kRowsNone;
    const uint64_t e = (K == (int32_t)ix.kmer_k ? (dsel ? ix.kmer[1] : ix.kmer[0])
                                                : (dsel ? ix.kmer2[1] : ix.kmer2[0]))[c];
    k = (uint32_t)e;
    l = (uint32_t)(e >> 32);
    if (k > l) return kRowsNone;
    m = K;
  }
  while (m < m0) {
    const uint32_t rows = l - k + 1u;
    if (rows == 1u || (rows <= kTextRows && D.ctx == nullptr)) break;
    const int32_t g = min(m0 - m, 16);
    if (rows <= kWinRows && D.ctx != nullptr) {
      uint32_t c;
      if (!rd.code(p0 + m * d, d, g, comp, c)) return kRowsNone;
      const uint32_t mask = (uint32_t)win_mask((uint32_t)g);
      uint32_t cnt = 0u, r0 = 0u, r1 = 0u, r2 = 0u, r3 = 0u;
      win_rows<2>(D, k, rows, [&](uint32_t i, uint32_t t) {
        if (((t ^ c) & mask) != 0u || !win_real(D, k + i, t, (uint32_t)g)) return;
        if (cnt == 0u) r0 = i;
        else if (cnt == 1u) r1 = i;
        else if (cnt == 2u) r2 = i;
        else if (cnt == 3u) r3 = i;
        ++cnt;
      });
      if (cnt == 0u) return kRowsNone;
      m += g;
      if (cnt <= kTextRows) {
        const uint32_t ug = (uint32_t)g;
        R.n = cnt;
        R.q[0] = D.sa[k + r0] - ug;
        R.q[1] = cnt > 1u ? D.sa[k + r1] - ug : 0u;
        R.q[2] = cnt > 2u ? D.sa[k + r2] - ug : 0u;
        R.q[3] = cnt > 3u ? D.sa[k + r3] - ug : 0u;
        text_feed<STAGED>(ix, dsel, comp, rd.slot, rd.W, p0 + m * d, d, m0 - m, R);
        return R.n ? kRowsFew : kRowsNone;
      }
      k = D.isa[D.sa[k + r0] - (uint32_t)g];
      l = k + cnt - 1u;
      continue;
    }
    uint32_t a, b;
    if (lf_sym(D, k, l, rd.at(p0 + m * d), comp, a, b) > 3u || a > b) return kRowsNone;
    k = a;
    l = b;
    ++m;
    if (m >= wide_m && l - k >= kManyRows) return kRowsCut;
  }
  if (l - k >= kTextRows) return kRowsMany;
  R = text_rows(D, k, l);
  text_feed<STAGED>(ix, dsel, comp, rd.slot, rd.W, p0 + m * d, d, m0 - m, R);
  return R.n ? kRowsFew : kRowsNone;
}

// The suffixes of a node's nine strings: the rows run[j] >= a of R stand at
// its length, p is the place of its base, and c1 bases follow it to the
// search's end (fmi_window.h numbers the strings: the deletion, then per base
// the insertion, bit 1 + 2b, and the mismatch, bit 2 + 2b).  bit: a string's
// rows are in cnts, 3 bits each, and q holds its first row's suffix.
struct NodeStrings {
  uint32_t live, cnts;
  uint32_t q[9];
};

template <bool STAGED, bool MM_ONLY>
__device__ __forceinline__ NodeStrings node_strings(const DevIndex &ix, uint32_t dsel,
                                                    uint32_t comp, const ReadBases<STAGED> &rd,
                                                    const TextRows &R,
                                                    const int32_t (&run)[kTextRows], int32_t a,
                                                    int32_t p, int32_t d, int32_t c1) {
  NodeStrings S;
  S.live = 0u;
  S.cnts = 0u;
  const uint32_t w = rd.at(p), sm = w > 3u ? 4u : (comp ? 3u - w : w);
#pragma unroll
  for (uint32_t j = 0; j < kTextRows; ++j) {
    if (run[j] < a) continue;
    const uint32_t qa = R.q[j] - (uint32_t)a;
    auto put = [&](uint32_t bit, uint32_t x) {
#pragma unroll
      for (uint32_t i = 0; i < 9u; ++i)
        if (i == bit && !((S.live >> i) & 1u)) S.q[i] = x;
      S.live |= 1u << bit;
      S.cnts += 1u << (3u * bit);
    };
    if (!MM_ONLY && rd.match(ix, dsel, comp, qa, p + d, d, c1) == c1) put(0u, qa - (uint32_t)c1);
    if (qa == 0u) continue;
    const uint32_t b = (uint32_t)text_window32(ix, dsel, qa) & 3u, lb = comp ? 3u - b : b;
    if (b != sm && rd.match(ix, dsel, comp, qa - 1u, p + d, d, c1) == c1)
      put(2u * lb + 2u, qa - 1u - (uint32_t)c1);
    if (!MM_ONLY && rd.match(ix, dsel, comp, qa - 1u, p, d, c1 + 1) == c1 + 1)
      put(2u * lb + 1u, qa - 2u - (uint32_t)c1);
  }
  return S;
}

}  // namespace fmi
