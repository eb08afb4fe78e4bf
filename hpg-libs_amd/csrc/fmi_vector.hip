// fmi_vector.hip -- the mapping layer's 1-error search (fmi_search1_vector_batch):
// BWSearch1VectorHelper (search/search.c:1491-1709) over the interval vectors
// of bwt.c:1940-1950 (or, for a seed window, bwt.c:1447-1457).
//
// On an expanded index vector_text_kernel, a thread per (read, strand), runs
// the helper on the text: the vectors' entries that have records lie past
// half the window, where a read's interval has a row or a few, so a half is a
// table read, the rows' suffixes and a comparison with the text before each,
// and a node's nine strings are three more comparisons a row.  What it cannot
// hold (more than kTextRows rows at half the window) and short windows are
// marked in counts and left to vhelper_kernel, whose lanes have scratch for
// the vectors: short windows by their rows' contexts (win_run), the rest by LF
// steps (vh_task).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "../../include/fmi.h"
#include "fmi_device.h"
#include "fmi_internal.h"
#include "fmi_kernels.h"
#include "fmi_rows.h"
#include "fmi_vhelper.h"
#include "fmi_window.h"

namespace fmi {

namespace {

struct VhParams {
  DevIndex ix;
  const uint8_t *reads;
  const uint64_t *offsets;
  const int16_t *bounds;    // NULL or [start, end] per read, relative to the read
  fmi_hit *hits;
  uint32_t *counts;
  uint2 *scratch;           // lanes * (kMaxReadLen + 3) intervals
  uint32_t nreads, cap, strand_mask, mm_only;
  int32_t wide_m;           // rows_wide_m
};

// The count of a (read, strand) that waits for vhelper_kernel.
constexpr uint32_t kVhWaits = 0xFFFFFFFFu;

// VhSink for intervals that may be known by their first row's suffix.
struct VtSink : VhSink {
  const DevIndex *ix;
  using VhSink::add;
  __device__ __forceinline__ bool full() const { return false; }   // it counts them all
  __device__ __forceinline__ void add(VhRec &r, uint32_t dsel, const WinIv &iv) {
    if (mm_only && r.nmm && r.kind != FMI_MISMATCH) return;
    r.k = cnt >= cap || iv.q == kWinNone ? iv.k : dir_of(*ix, dsel).isa[iv.q];
    r.l = r.k + iv.rows - 1u;
    VhSink::add(r);
  }
};

// A task's window; false when it has no records (then its count is written).
__device__ __forceinline__ bool vh_window(const VhParams &P, uint32_t t, const uint8_t *&W,
                                          int32_t &len, int32_t &start, int32_t &end) {
  const uint32_t rd = t >> 1, strand = t & 1u;
  const uint64_t off = P.offsets[rd];
  const uint64_t len64 = P.offsets[rd + 1] - off;
  len = len64 > kMaxReadLen ? -1 : (int32_t)len64;
  W = P.reads + off;
  start = 0;
  end = len - 1;
  if (P.bounds) { start = P.bounds[2 * rd]; end = P.bounds[2 * rd + 1]; }
  return (P.strand_mask & (1u << strand)) && len >= 0 && start >= 0 && end < len &&
         end - start >= 2;
}

// One half (dir 0: the backward vector's nodes and the exact record; dir 1:
// the forward vector's), numbered as in fmi_window.h; false when its interval
// has more than kTextRows rows at the shortest node.
template <bool STAGED>
__device__ __forceinline__ bool vt_half(const DevIndex &ix, uint32_t dir, uint32_t strand,
                                        const ReadBases<STAGED> &rd, int32_t start, int32_t end,
                                        int32_t wide_m, VhRec &r, VtSink &S) {
  const uint32_t dsel = dir ^ strand, comp = strand;
  const int32_t L = end - start + 1, d = dir ? 1 : -1, p0 = dir ? start : end;
  const int32_t m0 = dir ? (L - 1) / 2 : L - (L - 1) / 2;
  TextRows R;
  uint32_t k, l;
  const uint32_t found = search_rows<STAGED>(ix, dsel, comp, rd, p0, d, m0, R, k, l, wide_m);
  if (found != kRowsFew) return found == kRowsNone;   // without rows no node is alive
  // how far each row goes on with the window: it ends at a node
  const int32_t N = L - m0;
  int32_t run[kTextRows] = {-1, -1, -1, -1};
#pragma unroll
  for (uint32_t j = 0; j < kTextRows; ++j)
    if (j < R.n) run[j] = rd.match(ix, dsel, comp, R.q[j], p0 + m0 * d, d, N);
  if (dir == 0u) {
    uint32_t first = kWinNone, rows = 0u;
#pragma unroll
    for (uint32_t j = 0; j < kTextRows; ++j)
      if (run[j] == N) {
        if (rows++ == 0u) first = R.q[j] - (uint32_t)N;
      }
    if (rows) {
      r.pos = -1;
      S.add(r, dsel, WinIv{0u, first, rows});
    }
  }
  r.nmm = 1u;
  // the nodes, longest first
  for (int32_t cur = N;;) {
    int32_t a = -1;
#pragma unroll
    for (uint32_t j = 0; j < kTextRows; ++j)
      if (run[j] < cur) a = max(a, run[j]);
    if (a < 0) break;
    cur = a;
    const int32_t c1 = N - 1 - a, p = p0 + (m0 + a) * d;
    const bool last = c1 == 0;
    r.err_pos = p;
    const NodeStrings T = node_strings<STAGED, false>(ix, dsel, comp, rd, R, run, a, p, d, c1);
#pragma unroll
    for (uint32_t i = 0; i < 9u; ++i) {
      // at the last base the mismatch comes before the insertion
      auto add = [&](uint32_t bit) {
        if (!((T.live >> bit) & 1u)) return;
        const bool isins = (bit & 1u) != 0u;
        r.pos = last ? -1 : (dir ? end + 1 : start - 1);
        r.kind = bit == 0u ? FMI_DELETION : (isins ? FMI_INSERTION : FMI_MISMATCH);
        r.base = bit == 0u ? 0xFFu : (bit - 1u) >> 1;
        if (isins && last && dir == 0u) {
          // search.c:1556 stores kind 3, base INSERTION (3), position b
          r.base = FMI_INSERTION;
          r.err_pos = (int32_t)((bit - 1u) >> 1);
        }
        S.add(r, dsel, WinIv{0u, T.q[bit], (T.cnts >> (3u * bit)) & 7u});
      };
      if (i == 0u || !last) add(i);
      else add(((i - 1u) ^ 1u) + 1u);
    }
  }
  return true;
}

template <bool STAGED>
__device__ __forceinline__ uint32_t vt_task(const VhParams &P, uint32_t t, const uint8_t *W,
                                            const uint32_t *slot, int32_t start, int32_t end) {
  const uint32_t strand = t & 1u;
  VtSink S;
  S.out = P.hits + (uint64_t)t * P.cap;
  S.cap = P.cap;
  S.cnt = 0u;
  S.mm_only = P.mm_only;
  S.strand = strand;
  S.start = (int16_t)start;
  S.end = (int16_t)end;
  S.ix = &P.ix;
  const ReadBases<STAGED> rd{W, slot};
  VhRec r{0, 0, -1, 0, 0, 0, 0, 0};
  for (uint32_t dir = 0; dir < 2u; ++dir) {
    r.dir = dir;
    if (!vt_half<STAGED>(P.ix, dir, strand, rd, start, end, P.wide_m, r, S)) return kVhWaits;
  }
  return S.cnt;
}

// A thread per (read, strand), the read packed into its LDS slot (24 KB a
// workgroup; longer reads from their bytes).  Bound by the latency of a
// half's chain -- a table entry, the rows' suffixes, the text under them --
// with 16 wavefronts a CU (held to 128 registers) to hide it.  250 K reads of
// 150 bases over 64 Mbp: 175 us, where an LF step per base of both vectors on 64 K
// lanes (their scratch allows no more) took 6.6 ms.
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void vector_text_kernel(VhParams P) {
  __shared__ uint32_t slots[kReadRecordWords * 256u];
  const uint64_t t64 = (uint64_t)blockIdx.x * 256u + threadIdx.x;
  if (t64 >= 2ull * P.nreads) return;
  const uint32_t t = (uint32_t)t64;
  const uint8_t *W;
  int32_t len, start, end;
  if (!vh_window(P, t, W, len, start, end)) {
    P.counts[t] = 0;
    return;
  }
  if (end - start + 1 <= (int32_t)kWinMax && P.ix.d[0].ctx != nullptr) {
    P.counts[t] = kVhWaits;
    return;
  }
  uint32_t *slot = slots + threadIdx.x;
  if (len <= (int32_t)kStagedMaxLen) {
    stage_read(W, (uint32_t)len, slot);
    P.counts[t] = vt_task<true>(P, t, W, slot, start, end);
  } else {
    P.counts[t] = vt_task<false>(P, t, W, slot, start, end);
  }
}

// The lanes stride over the tasks (WAITING: those whose count says so), and
// each owns a vector scratch slice of kMaxReadLen + 3 intervals, so the
// scratch is sized by the lane count alone (no read of the offsets on the
// host).
template <bool WAITING>
__global__ __launch_bounds__(256) void vhelper_kernel(VhParams P) {
  __shared__ uint32_t words[WAITING ? kWinWords * 256u : 1u];
  const uint32_t lane = blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t lanes = gridDim.x * blockDim.x;
  uint2 *vb = P.scratch + (uint64_t)lane * (kMaxReadLen + 3u);
  for (uint32_t t = lane; t < 2u * P.nreads; t += lanes) {
    if (WAITING && P.counts[t] != kVhWaits) continue;
    const uint8_t *W;
    int32_t len, start, end;
    if (!vh_window(P, t, W, len, start, end)) {
      P.counts[t] = 0;
      continue;
    }
    const uint32_t strand = t & 1u;
    fmi_hit *out = P.hits + (uint64_t)t * P.cap;
    if (WAITING && end - start + 1 <= (int32_t)kWinMax && P.ix.d[0].ctx != nullptr) {
      VtSink S;
      S.out = out;
      S.cap = P.cap;
      S.cnt = 0u;
      S.mm_only = P.mm_only;
      S.strand = strand;
      S.start = (int16_t)start;
      S.end = (int16_t)end;
      S.ix = &P.ix;
      win_run(P.ix, vh_regs(W, start, (uint32_t)(end - start + 1)), start, end, strand, vb,
              words + threadIdx.x, S);
      P.counts[t] = S.cnt;
    } else {
      P.counts[t] = vh_task(P.ix, W, start, end, strand, P.mm_only, vb, out, P.cap);
    }
  }
}

}  // namespace

uint32_t vhelper_lanes(uint32_t nreads) {
  const uint64_t want = (2ull * nreads + 255) / 256 * 256;
  return (uint32_t)std::min<uint64_t>(want, kVhelperMaxLanes);
}

uint64_t vhelper_scratch_bytes(uint32_t lanes) {
  return (uint64_t)lanes * (kMaxReadLen + 3u) * sizeof(uint2);
}

hipError_t launch_vhelper(const DevIndex &ix, bool mm_only, uint32_t strand_mask,
                          const uint8_t *reads, const uint64_t *offsets, const int16_t *bounds,
                          uint32_t nreads, uint32_t cap, fmi_hit *hits, uint32_t *counts,
                          void *scratch, uint32_t lanes, hipStream_t s) {
  VhParams P{ix, reads, offsets, bounds, hits, counts, static_cast<uint2 *>(scratch), nreads, cap,
             strand_mask, mm_only ? 1u : 0u, rows_wide_m(ix.n)};
  if (nreads == 0 || lanes == 0) return hipSuccess;
  if (ix.text != nullptr) {
    const uint32_t grid = (uint32_t)((2ull * nreads + 255) / 256);
    hipLaunchKernelGGL(vector_text_kernel, dim3(grid), dim3(256), 0, s, P);
    hipLaunchKernelGGL(vhelper_kernel<true>, dim3(lanes / 256), dim3(256), 0, s, P);
  } else {
    hipLaunchKernelGGL(vhelper_kernel<false>, dim3(lanes / 256), dim3(256), 0, s, P);
  }
  return hipGetLastError();
}

}  // namespace fmi
