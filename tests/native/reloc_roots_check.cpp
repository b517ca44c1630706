// reloc_roots_check -- the two-level interval index (foundry_amd/csrc/
// reloc_index.h) and its search by one lane (reloc_word in restore_dev.h)
// executed on the CPU.
//
//   reloc_roots_check TABLE WORDS OUT
//
// TABLE: u64 n, u64 policy, then n lo, n hi, n new_lo (little endian).
// WORDS: u64 words.  OUT: the relocated words; then one JSON line on stdout
// with the index's shape: root entries, whether their fences are exact,
// lines, and the entries by what is below them ("direct": nothing, "flat":
// leaves alone, "deep": a tree), and the words of pairs that reloc_pair moves
// otherwise than reloc_word.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "../../foundry_amd/csrc/reloc_index.h"

using namespace fdy;

static std::vector<uint64_t> read_all(const char* path) {
  std::vector<uint64_t> v;
  FILE* f = std::fopen(path, "rb");
  if (!f) {
    std::perror(path);
    std::exit(2);
  }
  uint64_t x;
  while (std::fread(&x, 8, 1, f) == 1) v.push_back(x);
  std::fclose(f);
  return v;
}

int main(int argc, char** argv) {
  if (argc != 4) {
    std::fprintf(stderr, "usage: %s TABLE WORDS OUT\n", argv[0]);
    return 2;
  }
  const std::vector<uint64_t> t = read_all(argv[1]), w = read_all(argv[2]);
  if (t.size() < 2 || t.size() != 2 + 3 * t[0]) {
    std::fprintf(stderr, "bad table file\n");
    return 2;
  }
  const uint64_t n = t[0], *lo = t.data() + 2, *hi = lo + n, *nlo = hi + n;
  HostRootIndex x;
  std::string why;
  const int rc = build_root_index(lo, hi, nlo, n, (uint32_t)t[1], &x, &why);
  if (rc) {
    std::printf("{\"error\": %d}\n", rc);
    return 0;
  }
  RelocDev d = x.dev;
  d.root = x.root.data();
  d.line = x.line.data();
  uint64_t deep = 0, direct = 0;
  for (size_t b = 0; b < x.root.size(); ++b) {
    deep += (x.root[b].line & kRootTree) != 0;
    direct += (x.root[b].line & kRootDirect) != 0;
  }
  std::vector<uint64_t> out(w.size());
  for (size_t i = 0; i < w.size(); ++i) out[i] = reloc_word(d, w[i]);
  // Two words at once, either or both of them: each as by itself.
  uint64_t bad_pairs = 0;
  for (size_t i = 0; i < w.size(); ++i)
    for (uint32_t mask = 0; mask < 4; ++mask) {
      const size_t j = (i * 7 + 3) % w.size();
      uint64_t p[2] = {w[i], w[j]};
      reloc_pair(d, p, mask);
      bad_pairs += p[0] != (mask & 1 ? out[i] : w[i]) || p[1] != (mask & 2 ? out[j] : w[j]);
    }
  FILE* f = std::fopen(argv[3], "wb");
  if (!f || std::fwrite(out.data(), 8, out.size(), f) != out.size()) {
    std::perror(argv[3]);
    return 2;
  }
  std::fclose(f);
  std::printf("{\"roots\": %zu, \"exact\": %d, \"lines\": %zu, \"direct\": %llu, \"flat\": %llu, \"deep\": %llu, \"bad_pairs\": %llu}\n", x.root.size(),
              (int)(n == 0 || root_shape(lo, hi, n, [&] {
                      uint64_t bits = 0;
                      for (uint64_t i = 0; i < n; ++i) bits |= lo[i] - lo[0];
                      return bits;
                    }()).exact),
              x.line.size(), (unsigned long long)direct, (unsigned long long)(x.root.size() - direct - deep),
              (unsigned long long)deep, (unsigned long long)bad_pairs);
  return 0;
}
