// host_check.cpp -- drives the host-side code of libhpgfm.so (the CPU index
// builder, the index file reader and writer, the reference-directory
// importer, the text formatter) under AddressSanitizer and
// UndefinedBehaviorSanitizer, built from the same sources with g++ (see
// Makefile target `check`).  No GPU code is involved.
//
//   host_check selftest SEED   build, save and load indexes of several
//                              texts; load every truncation of a file and
//                              files with flipped bytes (checksum kept and
//                              recomputed); format records of random fields
//   host_check load PATH       load one index file, print its status
//   host_check import DIR      import one reference directory, print status
//   host_check spread N        the memory that decides the 1-error search's load
//                              mode: its own arrays, whatever else is kept
//   host_check items 32|64     share out a wavefront's items at and around the
//                              most that each item type is taken for: every 64
//                              of them are one wavefront's, once
//
// Exit status 0 unless a check fails (a sanitizer report aborts first).
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>
#include <string>
#include <vector>

#include "../../../include/fmi.h"
#include "../fmi_index.h"
#include "../fmi_items.h"

namespace {

uint64_t fnv1a(const std::vector<uint8_t> &b, size_t n) {
  uint64_t h = 1469598103934665603ull;
  for (size_t i = 0; i < n; ++i) {
    h ^= b[i];
    h *= 1099511628211ull;
  }
  return h;
}

std::vector<uint8_t> slurp(const std::string &p) {
  std::vector<uint8_t> v;
  FILE *f = fopen(p.c_str(), "rb");
  if (!f) return v;
  int c;
  while ((c = fgetc(f)) != EOF) v.push_back((uint8_t)c);
  fclose(f);
  return v;
}

bool spit(const std::string &p, const std::vector<uint8_t> &v, size_t n) {
  FILE *f = fopen(p.c_str(), "wb");
  if (!f) return false;
  const bool ok = fwrite(v.data(), 1, n, f) == n;
  return (fclose(f) == 0) && ok;
}

int load_status(const std::string &p) {
  fmi_index ix;
  std::string err;
  return fmi::load_index(p.c_str(), &ix, &err);
}

int fail(const char *what) {
  fprintf(stderr, "host_check: %s\n", what);
  return 1;
}

int selftest(uint32_t seed, const std::string &tmp) {
  std::mt19937_64 rng(seed);
  const uint64_t sizes[] = {1, 2, 97, 191, 192, 193, 5000, 40000};
  for (uint64_t n : sizes) {
    std::vector<uint8_t> text(n);
    for (auto &c : text) c = (uint8_t)(rng() & 3u);
    if (n > 1000) std::fill(text.begin() + 100, text.begin() + 700, (uint8_t)2);   // a run
    fmi_index ix;
    std::string err;
    if (fmi::build_index(text.data(), n, 1 + (uint32_t)(rng() % 32), &ix, &err) != FMI_OK)
      return fail("build_index");
    const std::string p = tmp + "/x.fmi";
    if (fmi::save_index(&ix, p.c_str(), &err) != FMI_OK) return fail("save_index");
    if (load_status(p) != FMI_OK) return fail("load of a good file");
    const std::vector<uint8_t> good = slurp(p);
    const std::string q = tmp + "/bad.fmi";
    // every truncation (a stride through large files)
    const size_t step = good.size() > 4096 ? good.size() / 1500 : 1;
    for (size_t cut = 0; cut < good.size(); cut += step) {
      if (!spit(q, good, cut)) return fail("write");
      if (load_status(q) == FMI_OK) return fail("a truncated file loaded");
    }
    // flipped bytes, with the checksum left and with it recomputed
    for (int t = 0; t < 300; ++t) {
      std::vector<uint8_t> b = good;
      const size_t at = (size_t)(rng() % (b.size() - 8));
      b[at] ^= (uint8_t)(1u << (rng() % 8));
      if (!spit(q, b, b.size())) return fail("write");
      if (load_status(q) == FMI_OK) return fail("a flipped byte loaded");
      const uint64_t h = fnv1a(b, b.size() - 8);
      std::memcpy(&b[b.size() - 8], &h, 8);
      if (!spit(q, b, b.size())) return fail("write");
      (void)load_status(q);   // may load (a valid file): must not misbehave
    }
    // text lines of random records
    std::vector<fmi_hit> hits(8);
    std::vector<int32_t> chrom(8 * 4);
    std::vector<uint64_t> coord(8 * 4);
    for (auto &h : hits) {
      std::memset(&h, 0, sizeof h);
      h.k = (int64_t)(rng() % (n + 1));
      h.l = h.k + (int64_t)(rng() % 3) - 1;
      h.start = (int16_t)(rng() % 50);
      h.end = (int16_t)(rng() % 120);
      h.err_pos = (int16_t)(rng() % 2000) - 1000;
      h.num_mismatches = (uint8_t)(rng() % 2);
      h.err_kind = (uint8_t)(rng() % 4);
      h.err_base = (uint8_t)(rng() % 5);
      h.dir = (uint8_t)(rng() % 2);
    }
    for (auto &c : chrom) c = (int32_t)(rng() % 3) - 1;
    for (auto &c : coord) c = rng();
    std::string out;
    uint64_t missing = 0;
    const char *read = "ACGTNACGTTGCA";
    for (uint32_t nw : {0u, 5u, 13u, 20u})
      if (fmi::format_results(&ix, rng(), (int)(rng() % 2), read, nw, hits.data(), 8,
                              chrom.data(), coord.data(), 4, &out, &missing) != FMI_OK)
        return fail("format_results");
  }
  return 0;
}

// The steps of every 509th wavefront of a launch over `lanes` lanes of at most
// `per_lane` items, 64 of which bring `total`.
template <class T>
int shares(uint64_t lanes, uint64_t per_lane, uint64_t total) {
  const uint32_t parts = fmi::item_parts(lanes, per_lane);
  for (uint32_t i = 0; i <= parts / 509u; ++i) {
    const uint32_t part = i < parts / 509u ? 509u * i : parts - 1u;
    uint64_t want = 64ull * part;
    T base = (T)want;
    if (want != (uint64_t)base) return fail("a wavefront starts at another place");
    while (want < total) {
      if ((uint64_t)base != want) return fail("a wavefront steps to another place");
      want += 64ull * parts;
      if (fmi::items_next<T>(base, (T)total, parts) != (want < total))
        return fail(want < total ? "a wavefront ends early" : "a wavefront does not end");
    }
  }
  return 0;
}

int items(uint32_t bits) {
  std::vector<uint64_t> per{1, 63, 64, 65, 1000, 1ull << 20, fmi::kItems32 - 1, fmi::kItems32};
  if (bits == 64) per.insert(per.end(), {fmi::kItems32 + 1, 1ull << 26, 1ull << 30});
  for (uint64_t lanes : {1ull, 64ull, 65ull, 1000ull, 1ull << 20})
    for (uint64_t p : per)
      for (uint64_t total : {(uint64_t)1, p, 63 * p + 1, 64 * p - 1, 64 * p}) {
        const int rc = bits == 32 ? shares<uint32_t>(lanes, p, total)
                                  : shares<uint64_t>(lanes, p, total);
        if (rc) return rc;
      }
  return 0;
}

int spread(uint64_t n) {
  std::vector<uint8_t> text(n, 1);
  fmi_index ix;
  std::string err;
  if (fmi::build_index(text.data(), n, 16, &ix, &err) != FMI_OK) return fail("build_index");
  const uint64_t compact = fmi::search1_spread_bytes(&ix);
  if (compact < n / 3 || compact > 64 * n + 4096) return fail("the compact index's bytes");
  ix.full_bytes = 16 * n;
  ix.kmer_bytes = 1 << 20;
  ix.ctx_bytes = 8 * n;                          // read by other searches only
  return fmi::search1_spread_bytes(&ix) == compact + 16 * n + (1 << 20)
             ? 0 : fail("the row contexts move the load mode");
}

}  // namespace

int main(int argc, char **argv) {
  if (argc < 3) return fail("usage: host_check selftest SEED [TMPDIR] | load PATH | import DIR | items BITS | spread N");
  const std::string cmd = argv[1];
  if (cmd == "selftest") return selftest((uint32_t)strtoul(argv[2], nullptr, 10), argc > 3 ? argv[3] : "/tmp");
  if (cmd == "spread") return spread(strtoull(argv[2], nullptr, 10));
  if (cmd == "items") return items((uint32_t)strtoul(argv[2], nullptr, 10));
  if (cmd == "load") {
    printf("%d\n", load_status(argv[2]));
    return 0;
  }
  if (cmd == "import") {
    fmi_index ix;
    std::string err;
    printf("%d\n", fmi::import_reference_dir(argv[2], &ix, &err));
    return 0;
  }
  return fail("unknown command");
}
