// fmi_ingest.hip -- reads in the reference's fastq_batch_t layout
// (bioformats/fastq/fastq_batch.h:24-34: the sequences one after another in
// `seq`, each followed by a NUL, and int data_indices[num_reads + 1] with
// the start of each) turned into the engine's read batch on the device: the
// base codes of encode_bases (bwt_commons.c:99-102, alphabet "ACGT"; any
// other byte is N, code 4), without the NULs, and uint64 offsets; and,
// optionally, the codes packed 2 bits per base with a 1-bit N mask.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "../../include/fmi.h"
#include "fmi_kernels.h"

namespace fmi {

namespace {

// Four bytes of text as codes: A/C/G/T in either case 0..3, anything else 4.
// Bits 1-2 of a letter give its code (A 00, C 01, T 10, G 11, so x ^ x >> 1);
// the code's letter is compared back with the byte to find the others.
__device__ __forceinline__ uint32_t encode4(uint32_t v) {
  uint32_t out = 0u;
#pragma unroll
  for (uint32_t j = 0; j < 4u; ++j) {
    const uint32_t c = (v >> (8u * j)) & 0xDFu;
    uint32_t x = (c >> 1) & 3u;
    x ^= x >> 1;
    out |= (((0x54474341u >> (8u * x)) & 0xFFu) == c ? x : 4u) << (8u * j);
  }
  return out;
}

// The last r in [0, n) with di[r] <= at, found by the whole wavefront: 64
// probes a round (4 rounds for 16 M reads, where a lane alone takes 24
// dependent loads).  All lanes of the wavefront call it with the same
// arguments.
__device__ __forceinline__ uint32_t wave_owner(const int32_t *di, uint32_t n, int64_t at) {
  const uint32_t lane = threadIdx.x & 63u;
  uint32_t lo = 0, hi = n;
  while (hi - lo > 1u) {
    const uint32_t step = (hi - lo + 63u) / 64u;
    const uint64_t idx = (uint64_t)lo + (uint64_t)lane * step;
    const uint64_t yes = __ballot(lane == 0u || (idx < hi && (int64_t)di[idx] <= at));
    lo += (63u - (uint32_t)__builtin_clzll(yes)) * step;
    hi = min(lo + step, hi);
  }
  return lo;
}

// The bytes seq[data_indices[0] + p], p < nbytes = data_indices[nreads] -
// data_indices[0] (data_indices index seq, as the reference's
// batch->seq[batch->data_indices[r]]), in tiles of TILE aligned bytes:
// every NUL terminator is dropped, every other byte p of read r goes to
// codes[base_off + p - r].  Threads also write offsets[read_off + i] =
// data_indices[i] - data_indices[0] - i, i <= nreads (from 0: a caller
// placing several batches side by side adds each one's base_off afterwards).
// Indices that are not increasing by at least one per read give wrong codes
// but no write outside codes[base_off .. base_off + nbytes - nreads).
//
// Bound by its bytes (each read and written once).  A thread per byte, each
// with its own binary search of the read starts and a one-byte store, spent
// 20 dependent loads per byte: 519 us for 50.5 MB of 100-base reads.  Here
// two wavefronts find the reads of a tile's first and last byte, a
// thread takes 16 bytes with one short search among the tile's reads, and
// the tile's codes leave through LDS, laid out like their 16-byte pieces in
// codes, as whole 16-byte stores: 59 us, 1.7 TB/s.
template <uint32_t TILE>
__global__ __launch_bounds__(256) void fastq_encode_kernel(const char *seq, const int32_t *di,
                                                           uint32_t nreads, uint64_t nbytes,
                                                           uint64_t ntiles, uint64_t base_off,
                                                           uint64_t read_off, uint8_t *codes,
                                                           uint64_t *offsets) {
  constexpr uint32_t kEnds = TILE / 8u;            // reads of a tile whose ends fit in LDS
  __shared__ __align__(16) uint8_t out[TILE + 32u];
  __shared__ int64_t ends[kEnds];
  __shared__ uint32_t bounds[2];
  const int64_t d0 = di[0];
  for (uint64_t p = (uint64_t)blockIdx.x * 256u + threadIdx.x; p <= nreads;
       p += (uint64_t)gridDim.x * 256u)
    offsets[read_off + p] = (uint64_t)((int64_t)di[p] - d0 - (int64_t)p);   // a NUL per earlier read
  if (nreads == 0 || nbytes < nreads) return;
  const int64_t ncodes = (int64_t)(nbytes - nreads);
  const uint8_t *first = reinterpret_cast<const uint8_t *>(seq) + d0;
  const int64_t mis = (int64_t)(reinterpret_cast<uintptr_t>(first) & 15u);
  const uint8_t *base = first - mis;           // byte x of base is byte p = x - mis
  for (uint64_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
    const int64_t x0 = (int64_t)(tile * TILE);
    const int64_t pf = max(x0 - mis, (int64_t)0);
    const int64_t pl = min(x0 + (int64_t)TILE - mis, (int64_t)nbytes) - 1;
    if (pf > pl) break;                        // past the last byte
    const uint32_t wave = threadIdx.x >> 6;
    if (wave < 2u) {
      const uint32_t r = wave_owner(di, nreads, d0 + (wave ? pl : pf));
      if ((threadIdx.x & 63u) == 0u) bounds[wave] = r;
    }
    __syncthreads();
    const uint32_t r0 = bounds[0], r1 = bounds[1];
    // where read r0 + i ends, its NUL included
    const uint32_t nin = r1 >= r0 ? r1 - r0 + 1u : 1u;
    const bool staged = nin <= kEnds;
    if (staged)
      for (uint32_t i = threadIdx.x; i < nin; i += 256u) ends[i] = (int64_t)di[r0 + i + 1u] - d0;
    __syncthreads();
    const int64_t o0 = pf - (int64_t)r0;       // the tile's first code
    uint8_t *dst = codes + base_off + o0;
    const uint32_t m = (uint32_t)(reinterpret_cast<uintptr_t>(dst) & 15u);
    auto end_of = [&](uint32_t i) -> int64_t {
      return staged ? ends[i] : (int64_t)di[r0 + i + 1u] - d0;
    };
    for (uint32_t c = threadIdx.x; c < TILE / 16u; c += 256u) {
      const int64_t pc = x0 + 16 * (int64_t)c - mis;
      if (pc > pl || pc + 15 < pf) continue;
      const uint4 v = *reinterpret_cast<const uint4 *>(base + x0 + 16 * (int64_t)c);
      const uint32_t e[4] = {encode4(v.x), encode4(v.y), encode4(v.z), encode4(v.w)};
      const int64_t pa = max(pc, pf);
      uint32_t lo = 0, cnt = nin - 1u;         // ends at or before pa: reads already over
      while (cnt > 0u) {
        const uint32_t h = cnt / 2u;
        if (end_of(lo + h) <= pa) { lo += h + 1u; cnt -= h + 1u; }
        else cnt = h;
      }
      int64_t end = end_of(lo);
#pragma unroll
      for (uint32_t j = 0; j < 16u; ++j) {
        const int64_t p = pc + (int64_t)j;
        if (p < pf || p > pl) continue;
        if (p == end - 1) {                    // the read's NUL
          if (lo + 1u < nin) end = end_of(++lo);
          continue;
        }
        const int64_t o = p - (int64_t)lo - pf;
        if (o >= 0 && o < (int64_t)TILE)
          out[m + (uint32_t)o] = (uint8_t)(e[j >> 2] >> (8u * (j & 3u)));
      }
    }
    __syncthreads();
    // codes o0 .. of the tile: its bytes less the NULs among them
    int64_t n = pl + 1 - (int64_t)r1 - (end_of(nin - 1u) - 1 == pl ? 1 : 0) - o0;
    n = o0 < 0 ? 0 : min(min(n, (int64_t)TILE), ncodes - o0);
    for (uint32_t c = threadIdx.x; 16 * (int64_t)c < (int64_t)m + n; c += 256u) {
      const uint32_t a = 16u * c;
      if (a >= m && (int64_t)a + 16 <= (int64_t)m + n) {
        *reinterpret_cast<uint4 *>(dst - m + a) = *reinterpret_cast<const uint4 *>(out + a);
      } else {
        for (uint32_t j = a < m ? m : a; j < a + 16u && (int64_t)j < (int64_t)m + n; ++j)
          dst[(int64_t)j - (int64_t)m] = out[j];
      }
    }
    __syncthreads();
  }
}

// The same, a thread per byte with a search of its own: for a small batch, whose
// tiles are a few workgroups with a chain of loads each.
__global__ __launch_bounds__(256) void fastq_encode_small_kernel(const char *seq, const int32_t *di,
                                                                 uint32_t nreads, uint64_t nbytes,
                                                                 uint64_t base_off,
                                                                 uint64_t read_off, uint8_t *codes,
                                                                 uint64_t *offsets) {
  const uint64_t p = (uint64_t)blockIdx.x * 256u + threadIdx.x;
  const int64_t d0 = di[0];
  if (p <= nreads) offsets[read_off + p] = (uint64_t)((int64_t)di[p] - d0 - (int64_t)p);
  if (p >= nbytes || nreads == 0) return;
  const int64_t at = d0 + (int64_t)p;
  const uint32_t c = (uint8_t)seq[at];               // before the search it does not depend on
  uint32_t lo = 0, hi = nreads;                      // the last read that starts at or before it
  while (hi - lo > 1u) {
    const uint32_t mid = lo + (hi - lo) / 2u;
    if ((int64_t)di[mid] <= at) lo = mid;
    else hi = mid;
  }
  if (at == (int64_t)di[lo + 1] - 1) return;         // its NUL
  const int64_t o = (int64_t)p - (int64_t)lo;
  if (o >= 0 && nbytes >= nreads && (uint64_t)o < nbytes - nreads)
    codes[base_off + (uint64_t)o] = (uint8_t)encode4(c);
}

// 2-bit packing of nbases codes: thread t packs bases 16t .. 16t + 15 into
// packed[t] (base i at bits 2(i % 16)) and their N flags into nmask's bits
// (base i at bit i % 16 of the 16-bit word t); an N packs as 0.
__global__ __launch_bounds__(256) void pack_codes_kernel(const uint8_t *codes, uint64_t nbases,
                                                         uint32_t *packed, uint16_t *nmask) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  const uint64_t words = (nbases + 15) / 16;
  for (uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; t < words; t += stride) {
    uint32_t w = 0;
    uint32_t m = 0;
    for (uint32_t j = 0; j < 16; ++j) {
      const uint64_t i = 16 * t + j;
      if (i >= nbases) break;
      const uint32_t c = codes[i];
      if (c > 3u) m |= 1u << j;
      else w |= c << (2 * j);
    }
    packed[t] = w;
    if (nmask) nmask[t] = (uint16_t)m;
  }
}

}  // namespace

hipError_t launch_fastq_encode(const char *seq, const int32_t *data_indices, uint32_t nreads,
                               uint64_t nbytes, uint64_t base_off, uint64_t read_off,
                               uint8_t *codes, uint64_t *offsets, hipStream_t s) {
  // A thread per byte up to 512 KiB: 6.2 us for 100 reads of 100 bases, 7.1 for
  // 3000, where tiles take 8.1 and 8.7, but 11.8 and 9.1 for 10,000.
  if (nbytes <= (512u << 10) && nreads <= (512u << 10)) {
    const uint64_t work = std::max<uint64_t>(nbytes, (uint64_t)nreads + 1u);
    hipLaunchKernelGGL(fastq_encode_small_kernel, dim3((uint32_t)((work + 255u) / 256u)), dim3(256),
                       0, s, seq, data_indices, nreads, nbytes, base_off, read_off, codes, offsets);
    return hipGetLastError();
  }
  // Tiles of 4096 bytes where those of 8192 would be too few to fill the device:
  // 9.1 us for 1 MB where they take 12.4, 18.5 and 18.9 for 10 MB, but 61.0 and
  // 59.2 for 50 MB.  A tile more than the bytes fill: they may start 15 bytes into
  // the first.  With no bytes the one workgroup writes the offsets alone.
  const uint32_t tile = nbytes <= (16u << 20) ? 4096u : 8192u;
  const uint64_t ntiles = nbytes ? (nbytes + 15u + tile - 1u) / tile : 0u;
  const uint64_t want = std::max<uint64_t>(ntiles, ((uint64_t)nreads + 2048u) / 2048u);
  const dim3 grid((uint32_t)std::min<uint64_t>(std::max<uint64_t>(want, 1u), 65536u));
  if (tile == 4096u)
    hipLaunchKernelGGL(fastq_encode_kernel<4096u>, grid, dim3(256), 0, s, seq, data_indices, nreads,
                       nbytes, ntiles, base_off, read_off, codes, offsets);
  else
    hipLaunchKernelGGL(fastq_encode_kernel<8192u>, grid, dim3(256), 0, s, seq, data_indices, nreads,
                       nbytes, ntiles, base_off, read_off, codes, offsets);
  return hipGetLastError();
}

hipError_t launch_pack_codes(const uint8_t *codes, uint64_t nbases, uint32_t *packed,
                             uint16_t *nmask, hipStream_t s) {
  const uint64_t words = (nbases + 15) / 16;
  if (words == 0) return hipSuccess;
  uint64_t grid = (words + 255) / 256;
  if (grid > 65536) grid = 65536;
  hipLaunchKernelGGL(pack_codes_kernel, dim3((uint32_t)grid), dim3(256), 0, s, codes, nbases,
                     packed, nmask);
  return hipGetLastError();
}

}  // namespace fmi
