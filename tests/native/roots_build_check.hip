// roots_build_check -- the two-level interval index placed by the library's
// kernels (launch_roots_count, launch_roots_place) against the host build of
// the same table (build_root_index in foundry_amd/csrc/reloc_index.h).
//
//   roots_build_check TABLE
//
// TABLE: u64 n, u64 policy, then n lo, n hi, n new_lo (little endian).  One
// JSON line on stdout: the host's root entries and lines, the device's line
// count, and how many of either differ.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "../../foundry_amd/csrc/kernels.h"
#include "../../foundry_amd/csrc/reloc_index.h"

using namespace fdy;

static void check(hipError_t e, const char* what) {
  if (e == hipSuccess) return;
  std::fprintf(stderr, "%s: %s\n", what, hipGetErrorString(e));
  std::exit(3);
}

static uint8_t* device(size_t bytes) {
  void* p = nullptr;
  check(hipMalloc(&p, bytes), "hipMalloc");
  return static_cast<uint8_t*>(p);
}

int main(int argc, char** argv) {
  FILE* f = argc == 2 ? std::fopen(argv[1], "rb") : nullptr;
  if (!f) {
    std::fprintf(stderr, "usage: %s TABLE\n", argv[0]);
    return 2;
  }
  std::vector<uint64_t> t;
  for (uint64_t x; std::fread(&x, 8, 1, f) == 1;) t.push_back(x);
  std::fclose(f);
  if (t.size() < 5 || t.size() != 2 + 3 * t[0]) {
    std::fprintf(stderr, "bad table file\n");
    return 2;
  }
  const uint64_t n = t[0], *lo = t.data() + 2, *hi = lo + n, *nlo = hi + n;
  HostRootIndex x;
  std::string why;
  if (build_root_index(lo, hi, nlo, n, (uint32_t)t[1], &x, &why)) {
    std::fprintf(stderr, "%s\n", why.c_str());
    return 2;
  }
  uint64_t bits = 0;
  for (uint64_t i = 0; i < n; ++i) bits |= lo[i] - lo[0];
  const RootShape sh = root_shape(lo, hi, n, bits);
  const uint64_t blocks = (sh.nb + kRootBlock - 1) / kRootBlock;
  IndexArgs a{};
  uint8_t* table = device(24 * n);
  check(hipMemcpy(table, lo, 24 * n, hipMemcpyHostToDevice), "table");
  a.lo = reinterpret_cast<uint64_t*>(table);
  a.hi = a.lo + n;
  a.nlo = a.hi + n;
  a.n = n;
  a.nb = sh.nb;
  a.shift = sh.shift;
  a.fence_shift = sh.fence_shift;
  a.exact = sh.exact;
  a.block_sum = reinterpret_cast<uint64_t*>(device(8 * (blocks + 1)));
  a.total = a.block_sum + blocks;
  a.ends = reinterpret_cast<uint32_t*>(device(4 * sh.nb));
  check(launch_roots_count(a, nullptr), "count");
  uint64_t total = 0;
  check(hipMemcpy(&total, a.total, 8, hipMemcpyDeviceToHost), "total");
  uint64_t bad_roots = 0, bad_lines = 0;
  if (total == x.line.size() && x.root.size() == sh.nb) {
    a.root = reinterpret_cast<RelocRoot*>(device(sizeof(RelocRoot) * sh.nb));
    a.line = reinterpret_cast<RelocLine*>(device(sizeof(RelocLine) * total));
    check(launch_roots_place(a, nullptr), "place");
    std::vector<RelocRoot> root(sh.nb);
    std::vector<RelocLine> line(total);
    check(hipMemcpy(root.data(), a.root, sizeof(RelocRoot) * sh.nb, hipMemcpyDeviceToHost), "roots");
    check(hipMemcpy(line.data(), a.line, sizeof(RelocLine) * total, hipMemcpyDeviceToHost), "lines");
    for (uint64_t b = 0; b < sh.nb; ++b) bad_roots += std::memcmp(&root[b], &x.root[b], sizeof(RelocRoot)) != 0;
    for (uint64_t l = 0; l < total; ++l) bad_lines += std::memcmp(&line[l], &x.line[l], sizeof(RelocLine)) != 0;
  }
  std::printf("{\"roots\": %zu, \"lines\": %zu, \"device_lines\": %llu, \"bad_roots\": %llu, \"bad_lines\": %llu}\n",
              x.root.size(), x.line.size(), (unsigned long long)total, (unsigned long long)bad_roots,
              (unsigned long long)bad_lines);
  return 0;
}
