// fmi_window.h -- BWSearch1VectorHelper (search/search.c:1491-1709) on a short
// window (3 to kWinMax bases) of an expanded index with row contexts.
//
// The helper's vectors are the intervals of the window's suffixes (backward
// half) and prefixes (forward half), and its records are the window with one
// base left out, put in or replaced at the vector's end, searched to the
// window's other end.  Feeding the window's bases s[0], s[1], ... in a half's
// direction, node m is the interval of s[0 .. m-1]; it has records when the
// step to m + 1 changes its size, and its nine strings are
//   deletion     s[0 .. m-1]    s[m+1 .. L-1]
//   insertion b  s[0 .. m-1] b  s[m .. L-1]
//   mismatch b   s[0 .. m-1] b  s[m+1 .. L-1]
// An LF step per base of each costs a few hundred dependent block reads a
// window and strand.  Here:
//   - from the first length with at most kWinRows rows on, the rows' contexts
//     say for every row how far the window's bases extend it (so, which nodes
//     exist) and which of a node's strings it goes on with: one or a few lines
//     for all nodes and strings, no LF step;
//   - a wider node's strings are looked up in the k-mer table (most of them
//     are absent from the text), and what remains of a string after the
//     table's k bases comes from its rows' contexts.
// A string's rows are the base interval's rows that extend with it, in the
// same order, so its interval starts at the row of the first one's suffix and
// holds as many rows as there are.
//
// 2 M windows of 18 bases over 64 Mbp: 18.1 ms by LF steps, 5.0 ms.  190 M
// lines of 64 bytes at 2.4 TB/s, of 3.0-3.5 that random lines reach on this
// memory: the wide nodes' lookups (72 M), the contexts (40 M) and the short
// intervals' table rows.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "../../include/fmi.h"
#include "fmi_device.h"
#include "fmi_internal.h"
#include "fmi_vhelper.h"

namespace fmi {

// The longest window: the last string has L + 1 bases, the shortest node of
// the forward half (L - 1) / 2, and a context holds 16 of the rest.
constexpr uint32_t kWinMax = 29;
// Rows below which an interval goes by its rows' contexts.  A row costs a few
// instructions and a quarter of a 16-byte load, a wider node's nine lookups a
// line each: on 2 M windows of 18 bases over 64 Mbp the intervals have 977,
// 244, 61, 15, 4 rows at lengths 8 to 12, and 64 rows took 7.8 ms where 32
// took 8.4 and 16 took 9.2 (before the nodes' loops were parted).
constexpr uint32_t kWinRows = 64;
constexpr uint32_t kWinNone = 0xFFFFFFFFu;
// A lane's words in LDS: a wide node's nine intervals, then the contexts of the
// first rows that have a part in a record (a repeat's window goes over them
// once per node).  In registers the intervals cost 38 spilled ones and 3.6
// times the stores: 7.5 ms against 5.8 for 2 M windows.
constexpr uint32_t kWinKept = 14;
constexpr uint32_t kWinWords = 18u + kWinKept;

__device__ __forceinline__ uint64_t win_mask(uint32_t x) {
  return x >= 32u ? ~0ull : (1ull << (2u * x)) - 1ull;
}

// Whether the first x context bases of a row are all text: the bases past the
// text's start are 0 in a context, so only one that ends in zeros from base
// x - 1 on has to look at its suffix.
__device__ __forceinline__ bool win_real(const DevDir &D, uint32_t row, uint32_t t, uint32_t x) {
  return x == 0u || (t >> (2u * (x - 1u))) != 0u || D.sa[row] >= x;
}

// f(i, context) for rows k .. k + rows - 1, in order, from 16-byte pieces, U of
// them a round of loads (the last piece may reach past the rows, not past the
// array, which is padded to 256 bytes).  A piece that holds none of the rows
// is not read: a load costs a request per lane, needed or not.
template <uint32_t U, class F>
__device__ __forceinline__ void win_rows(const DevDir &D, uint32_t k, uint32_t rows, F f) {
  const uint4 *c = reinterpret_cast<const uint4 *>(D.ctx + (k & ~3u));
  const uint32_t off = k & 3u, end = off + rows;
  for (uint32_t b = 0; b < end; b += 4u * U) {
    uint4 v[U];
    v[0] = c[b >> 2];
#pragma unroll
    for (uint32_t u = 1; u < U; ++u) {
      v[u] = opaque4();
      if (b + 4u * u < end) v[u] = c[(b >> 2) + u];
    }
#pragma unroll
    for (uint32_t u = 0; u < U; ++u) {
      const uint32_t w[4] = {v[u].x, v[u].y, v[u].z, v[u].w};
#pragma unroll
      for (uint32_t e = 0; e < 4u; ++e) {
        const uint32_t x = b + 4u * u + e;
        if (x >= off && x < end) f(x - off, w[e]);
      }
    }
  }
}

// An interval of a record: its rows, and the first row's suffix q when that is
// known (then k is not: the caller reads isa[q] where it needs it).
struct WinIv {
  uint32_t k, q, rows;
};

// The first K-mer table row of the strings that start with the m fed bases of
// code, m < K, K - m <= 3: the entries of those bases behind K - m others are
// neighbours, in row order.  False where the text ends within those others
// (the interval has a row that no entry holds).
__device__ __forceinline__ bool win_range(const uint64_t *tab, uint32_t K, uint64_t tail,
                                          uint64_t code, uint32_t m, uint32_t &k, uint32_t &l) {
  const uint32_t t = K - m;
  const uint64_t mm = win_mask(m), c = code & mm;
  for (uint32_t u = 0; u < t; ++u)
    if (((tail >> (2u * u)) & mm) == c) return false;
  uint32_t a = (uint32_t)(c << (2u * t)), b = a + (1u << (2u * t)) - 1u;
  uint64_t ea = tab[a], eb = tab[b];
  while ((uint32_t)ea > (uint32_t)(ea >> 32) && a < b) ea = tab[++a];
  if ((uint32_t)ea > (uint32_t)(ea >> 32)) { k = 1u; l = 0u; return true; }
  while ((uint32_t)eb > (uint32_t)(eb >> 32)) eb = tab[--b];
  k = (uint32_t)ea;
  l = (uint32_t)(eb >> 32);
  return true;
}

// One LF step of physical symbol s; false when it empties.
__device__ __forceinline__ bool win_lf(const DevDir &D, uint32_t s, uint32_t &k, uint32_t &l) {
  uint32_t a, b;
  lf_sym(D, k, l, s, 0u, a, b);
  k = a;
  l = b;
  return a <= b;
}

// The g bases of code fed to [k, l]: by LF steps while it is wide, then from
// its rows' contexts; false when nothing is left.
__device__ __forceinline__ bool win_extend(const DevDir &D, uint32_t k, uint32_t l, uint64_t code,
                                           uint32_t g, WinIv &iv) {
  while (g > 0u && (g > 16u || l - k >= kWinRows)) {
    if (!win_lf(D, (uint32_t)code & 3u, k, l)) return false;
    code >>= 2;
    --g;
  }
  iv.k = k;
  iv.q = kWinNone;
  iv.rows = l - k + 1u;
  if (g == 0u) return true;
  uint32_t cnt = 0u, first = 0u;
  const uint32_t want = (uint32_t)code, mask = (uint32_t)win_mask(g);
  win_rows<2>(D, k, l - k + 1u, [&](uint32_t i, uint32_t t) {
    if (((t ^ want) & mask) == 0u && win_real(D, k + i, t, g)) {
      if (cnt == 0u) first = i;
      ++cnt;
    }
  });
  if (cnt == 0u) return false;
  iv.q = D.sa[k + first] - g;
  iv.rows = cnt;
  return true;
}

// One half: dir 0 the backward vector's nodes and the exact record, dir 1 the
// forward vector's.  s, nf: the window's L bases in the half's feed order as
// physical symbols, and their N flags; vb: L intervals of scratch; lds:
// kWinWords words in LDS, word i at lds[i * 256].  Records
// go to S.add(r, dsel, iv) in the helper's order, until S.full(); r carries the
// record state (its k, l are not used).
template <class Sink>
__device__ __forceinline__ void win_half(const DevIndex &ix, uint32_t dir, uint32_t strand,
                                         uint64_t s, uint32_t nf, uint32_t L, int32_t start,
                                         int32_t end, uint2 *vb, uint32_t *lds, VhRec &r, Sink &S) {
  const uint32_t dsel = dir ^ strand;
  const DevDir &D = dir_of(ix, dsel);
  const uint32_t K = ix.kmer_k, K2 = ix.kmer2_k;
  const uint64_t *tabK = dsel ? ix.kmer[1] : ix.kmer[0];
  const uint64_t *tab2 = dsel ? ix.kmer2[1] : ix.kmer2[0];
  const uint32_t m0 = dir ? (L - 1u) / 2u : L - (L - 1u) / 2u;   // the shortest node
  const uint32_t fn = nf ? (uint32_t)__builtin_ctz(nf) : L;      // bases before the first N
  if (fn < m0) return;
  // ---- the interval at a length m <= m0, or the first narrow one
  const uint64_t tail = text_window32(ix, dsel, ix.n);           // the text's last bases
  uint32_t k = 0u, l = ix.n, m = 0u;
  if (K && K <= m0) {
    const uint64_t e = tabK[(uint32_t)(s & win_mask(K))];
    k = (uint32_t)e; l = (uint32_t)(e >> 32); m = K;
  } else if (K2 && K2 <= m0) {
    const uint64_t e = tab2[(uint32_t)(s & win_mask(K2))];
    k = (uint32_t)e; l = (uint32_t)(e >> 32); m = K2;
  } else if (K2 && K2 - m0 <= 3u) {
    if (win_range(tab2, K2, tail, s, m0, k, l)) m = m0;
  } else if (!K2 && K && K - m0 <= 3u) {
    if (win_range(tabK, K, tail, s, m0, k, l)) m = m0;
  }
  if (k > l) return;
  for (; m < m0 && (l - k >= kWinRows || L + 1u - m > 16u); ++m)
    if (!win_lf(D, (uint32_t)(s >> (2u * m)) & 3u, k, l)) return;
  // ---- wide nodes, kept until the narrow ones are done
  uint32_t wide = 0u;
  bool dead = false;
  while (m < L && l - k >= kWinRows) {
    uint32_t a = k, b = l;
    bool live = m < fn;
    if (live) {
      bool done = false;
      if (K2 && m + 1u <= K2 && K2 - (m + 1u) <= 3u) {
        if (m + 1u == K2) {
          const uint64_t e = tab2[(uint32_t)(s & win_mask(K2))];
          a = (uint32_t)e; b = (uint32_t)(e >> 32);
          done = true;
        } else {
          done = win_range(tab2, K2, tail, s, m + 1u, a, b);
        }
      }
      live = done ? a <= b : win_lf(D, (uint32_t)(s >> (2u * m)) & 3u, a, b);
    }
    if (!live || b - a != l - k) {
      vb[m] = make_uint2(k, l);
      wide |= 1u << m;
    }
    if (!live) { dead = true; break; }
    k = a;
    l = b;
    ++m;
  }
  // ---- narrow nodes, from one look at every row.  Against the N = L - mb
  // bases left, a row's context differs from them at the bits of x0, from
  // them less the first at those of xd, and less its own first base at those
  // of xi (one bit per base, an N always differs).  The row ends at the
  // length of its first difference, a node (bit L: it reaches the window's
  // end), and has a part in node a's strings only if it agrees with the
  // first a bases and then
  //   mismatch   x0 holds a alone
  //   deletion   xd is empty from a on
  //   insertion  xi is empty from a on
  // Few rows have any: cand.
  const uint32_t mb = m;
  uint32_t nodes = wide;
  uint64_t cand = 0ull;
  uint32_t nc = 0u;
  uint32_t *kept = lds + 18u * 256u;               // the first of their contexts
  if (!dead) {
    if (m == L) {
      nodes |= 1u << L;
    } else {
      const uint32_t N = L - m;
      const uint32_t want = (uint32_t)(s >> (2u * m));
      uint32_t ns = (nf >> m) & 0xFFFFu;           // N of base i -> bit 2i
      ns = (ns | (ns << 8)) & 0x00FF00FFu;
      ns = (ns | (ns << 4)) & 0x0F0F0F0Fu;
      ns = (ns | (ns << 2)) & 0x33333333u;
      ns = (ns | (ns << 1)) & 0x55555555u;
      const uint32_t mN = (uint32_t)win_mask(N), mN1 = mN >> 2;
      uint32_t at = 0u;
      win_rows<4>(D, k, l - k + 1u, [&](uint32_t i, uint32_t t) {
        auto fold = [](uint32_t x) { return (x | (x >> 1)) & 0x55555555u; };
        const uint32_t x0 = (fold(t ^ want) | ns) & mN;
        const uint32_t xd = (fold(t ^ (want >> 2)) | (ns >> 2)) & mN1;
        const uint32_t xi = (fold((t >> 2) ^ want) | ns) & mN;
        // the bits of xd, xi from the row's first difference on are clear
        // exactly when a string goes on from some node up to it
        const uint32_t low = x0 & (0u - x0);       // its first difference
        const uint32_t run = x0 ? (uint32_t)__builtin_ctz(x0) >> 1 : N;
        const uint32_t up = x0 ? ~(low - 1u) : 0u; // bits at it and above
        if ((x0 & (x0 - 1u)) == 0u || (xd & up) == 0u || (xi & up) == 0u) {
          cand |= 1ull << i;
          if (nc < kWinKept) kept[nc * 256u] = t;
          ++nc;
        }
        uint32_t end_at = run;
        if (!win_real(D, k + i, t, run)) end_at = min(run, D.sa[k + i]);
        at |= 1u << (m + end_at);
      });
      nodes |= at & ~((1u << m0) - 1u);
    }
  }
  if (dir) nodes &= ~(1u << L);
  // ---- the records, longest node first: the narrow ones, then the wide (in
  // loops of their own, so that the lanes of a wavefront, whose windows have
  // different numbers of narrow nodes, come to the wide ones together)
  // The order of a node's records: number 0 the deletion, then per base the
  // insertion and the mismatch (at the last base the mismatch first).
  auto emit = [&](uint32_t bit, bool last, const WinIv &iv) {
    const bool del = bit == 0u, isins = !del && ((bit & 1u) != 0u) == !last;
    const uint32_t b = (bit - 1u) >> 1;
    r.pos = last ? -1 : (dir ? end + 1 : start - 1);
    r.kind = del ? FMI_DELETION : (isins ? FMI_INSERTION : FMI_MISMATCH);
    r.base = del ? 0xFFu : b;
    if (isins && last && dir == 0u) {
      // search.c:1556 stores kind 3, base INSERTION (3), position b
      r.base = FMI_INSERTION;
      r.err_pos = (int32_t)b;
    }
    S.add(r, dsel, iv);
  };
  if (mb == L && (nodes >> L)) {                   // the window itself is wide
    r.pos = -1;
    S.add(r, dsel, WinIv{k, kWinNone, l - k + 1u});
    nodes ^= 1u << L;
  }
  for (nodes &= ~wide; nodes && !S.full();) {
    m = 31u - (uint32_t)__builtin_clz(nodes);
    nodes ^= 1u << m;
    const bool exact = m == L, last = m == L - 1u;
    // what follows the node's base, with the base (G) and without (F)
    const uint32_t c1 = exact ? 0u : L - 1u - m, a = m - mb;
    const uint32_t f32 = (uint32_t)(s >> (2u * (m + 1u))), g32 = (uint32_t)(s >> (2u * m));
    const uint32_t sm = g32 & 3u;
    const bool smn = exact || ((nf >> m) & 1u) != 0u;
    const bool okf = exact || (nf >> (m + 1u)) == 0u, okg = okf && !smn;
    const uint32_t insbit = last ? 2u : 1u, mmbit = last ? 1u : 2u;
    const uint32_t pre = (uint32_t)(s >> (2u * mb)), pm = (uint32_t)win_mask(a);
    const uint32_t mf = (uint32_t)win_mask(c1), mg = (uint32_t)win_mask(c1 + 1u);
    uint32_t live = 0u;
    uint64_t cnts = 0ull, firsts = 0ull;           // per string: 7 and 6 bits
    uint32_t c = 0u;
    for (uint64_t left = cand; left; left &= left - 1ull, ++c) {
      const uint32_t i = (uint32_t)__builtin_ctzll(left);
      const uint32_t t = c < kWinKept ? kept[c * 256u] : D.ctx[k + i];
      if (((t ^ pre) & pm) != 0u) continue;
      const uint32_t u = a >= 16u ? 0u : t >> (2u * a), b = u & 3u, v = u >> 2;
      auto put = [&](uint32_t bit, uint32_t x) {
        if (!win_real(D, k + i, t, x)) return;
        if (!((live >> bit) & 1u)) firsts |= (uint64_t)i << (6u * bit);
        live |= 1u << bit;
        cnts += 1ull << (7u * bit);
      };
      if (okf && ((u ^ f32) & mf) == 0u) put(0u, a + c1);
      if (exact) continue;
      const uint32_t lb = strand ? 3u - b : b;
      if (okf && (smn || b != sm) && ((v ^ f32) & mf) == 0u) put(2u * lb + mmbit, a + c1 + 1u);
      if (okg && ((v ^ g32) & mg) == 0u) put(2u * lb + insbit, a + c1 + 2u);
    }
    if (!exact) {
      r.nmm = 1u;
      r.err_pos = dir ? start + (int32_t)m : end - (int32_t)m;
    }
    while (live) {
      const uint32_t bit = (uint32_t)__builtin_ctz(live);
      live &= live - 1u;
      const bool isins = bit != 0u && ((bit & 1u) != 0u) == !last;
      const uint32_t first = (uint32_t)(firsts >> (6u * bit)) & 63u;
      const WinIv iv{0u, D.sa[k + first] - (a + c1 + (bit == 0u ? 0u : (isins ? 2u : 1u))),
                     (uint32_t)(cnts >> (7u * bit)) & 127u};
      if (exact) {
        r.pos = -1;
        S.add(r, dsel, iv);
      } else {
        emit(bit, last, iv);
      }
    }
  }
  while (wide && !S.full()) {
    m = 31u - (uint32_t)__builtin_clz(wide);
    wide ^= 1u << m;
    const bool last = m == L - 1u;
    const uint32_t c1 = L - 1u - m;
    const uint64_t F = s >> (2u * (m + 1u)), G = s >> (2u * m);
    const uint32_t sm = (uint32_t)G & 3u;
    const bool smn = ((nf >> m) & 1u) != 0u;
    const bool okf = (nf >> (m + 1u)) == 0u, okg = okf && !smn;
    const uint2 w = vb[m];
    auto base = [&](uint32_t b) -> uint32_t { return strand ? 3u - b : b; };
    // string i's interval after the node's bases and its own base, or after
    // the first K bases of all of it
    const bool table = K && m < K && L - 1u >= K;
    uint32_t live = 0u;
    uint2 e[9];
    if (table) {
      const uint64_t low = s & win_mask(m);
      const uint32_t km = (uint32_t)win_mask(K);
#pragma unroll
      for (uint32_t i = 0; i < 9u; ++i) {
        const uint32_t b = (i - 1u) >> 1;
        const bool isins = i != 0u && ((i & 1u) != 0u) == !last;
        e[i] = make_uint2(1u, 0u);
        if (isins ? okg : (okf && (i == 0u || smn || base(b) != sm))) {
          const uint64_t rest = i == 0u ? F : ((uint64_t)base(b) | ((isins ? G : F) << 2));
          const uint64_t x = tabK[(uint32_t)(low | (rest << (2u * m))) & km];
          e[i] = make_uint2((uint32_t)x, (uint32_t)(x >> 32));
        }
      }
    } else {
      uint32_t pk[4], pl[4];
      lf_four(D, w.x, w.y, pk, pl);
#pragma unroll
      for (uint32_t i = 0; i < 9u; ++i) {
        const uint32_t b = (i - 1u) >> 1;
        const bool isins = i != 0u && ((i & 1u) != 0u) == !last;
        e[i] = make_uint2(1u, 0u);
        if (isins ? okg : (okf && (i == 0u || smn || base(b) != sm)))
          e[i] = i == 0u ? w : make_uint2(pick4(pk, base(b)), pick4(pl, base(b)));
      }
    }
#pragma unroll
    for (uint32_t i = 0; i < 9u; ++i) {            // all read before the first is kept
      lds[2u * i * 256u] = e[i].x;
      lds[(2u * i + 1u) * 256u] = e[i].y;
      if (e[i].x <= e[i].y) live |= 1u << i;
    }
    r.nmm = 1u;
    r.err_pos = dir ? start + (int32_t)m : end - (int32_t)m;
    while (live) {
      const uint32_t bit = (uint32_t)__builtin_ctz(live);
      live &= live - 1u;
      const bool isins = bit != 0u && ((bit & 1u) != 0u) == !last;
      // the string's bases after those already in its interval
      const uint32_t have = table ? K - m - (bit == 0u ? 0u : 1u) : 0u;
      WinIv iv;
      if (win_extend(D, lds[2u * bit * 256u], lds[(2u * bit + 1u) * 256u],
                     (isins ? G : F) >> (2u * have), (isins ? c1 + 1u : c1) - have, iv))
        emit(bit, last, iv);
    }
  }
}

// The helper over the window W of L = 3 .. kWinMax bases at start..end on
// strand 0 (backward, forward) or 1 (forward_rev, backward_rev).
template <class Sink>
__device__ __forceinline__ void win_run(const DevIndex &ix, const VhRegs &W, int32_t start,
                                        int32_t end, uint32_t strand, uint2 *vb, uint32_t *lds,
                                        Sink &S) {
  const uint32_t L = (uint32_t)(end - start + 1);
  const uint64_t code = (W.code ^ (strand ? ~0ull : 0ull)) & win_mask(L);
  const uint32_t nf = W.nfl & ((1u << L) - 1u);
  const uint64_t v = __builtin_bitreverse64(code);
  const uint64_t rev = (((v >> 1) & 0x5555555555555555ull) | ((v & 0x5555555555555555ull) << 1)) >>
                       (64u - 2u * L);
  const uint32_t rnf = __builtin_bitreverse32(nf) >> (32u - L);
  VhRec r{0, 0, -1, 0, 0, 0, 0, 0};
  for (uint32_t dir = 0; dir < 2u; ++dir) {
    r.dir = dir;
    if (!S.full())
      win_half(ix, dir, strand, dir ? code : rev, dir ? nf : rnf, L, start, end, vb, lds, r, S);
  }
}

}  // namespace fmi
