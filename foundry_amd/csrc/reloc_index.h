// reloc_index.h -- the interval indexes of the relocation search and their
// builders, whose steps are host and device code alike.  The two-level index
// (root entries over leaf lines) serves archives and relocation plans and is
// built by kernels (kernels.hip), a thread per root entry and per line; the
// index of root lines serves the no-allocation entry point (built on the
// host) and is what a plan is inspected by (built by kernels).  The CPU
// checks (tests/native) build both on the host, so both sides produce the
// same lines.
#pragma once

#include <stdint.h>

#include <algorithm>
#include <cstring>
#include <string>
#include <vector>

#include "../../include/foundry_restore.h"
#include "restore_dev.h"

namespace fdy {

// The interval index of a table, built on the host: its lines and the
// search parameters (dev.line is set when the lines are placed on the
// device).
struct HostIndex {
  std::vector<RelocLine> line;
  RelocDev dev{};
};

// Root lines per interval, about (between k/2 and k per interval, a power
// of two in all): a root line whose range holds more than four intervals
// takes a second read, its child.  More root lines mean fewer second reads
// and a larger index (64 B per line): 2 per interval for the no-allocation
// entry point's index, 16 for the lines a relocation plan is inspected by.
constexpr uint64_t kRootLinesPerInterval = 2;
constexpr uint64_t kPlanRootLinesPerInterval = 16;
constexpr uint32_t kLeafIntervals = kLineSlots;  // the interval at or before B, and three starting inside
constexpr uint64_t kMaxIndexLines = 0xFFFFFFF0ull;

// The root lines: 2^shift bytes each from lo_min, nb of them.
struct IndexShape {
  uint32_t shift;
  uint64_t nb;
};

// What check_table asks of interval i (prev_hi: the hi before it, or lo).
__host__ __device__ inline bool interval_ok(uint64_t lo, uint64_t hi, uint64_t prev_hi) {
  return lo < hi && hi != UINT64_MAX && prev_hi <= lo;
}

// A table's arguments before its intervals are looked at.
inline int check_table_args(const uint64_t* lo, const uint64_t* hi, const uint64_t* nlo, uint64_t n, uint32_t policy,
                            std::string* why) {
  if (policy > FDY_RELOC_INCLUSIVE) *why = "unknown relocation policy";
  else if (n && (!lo || !hi || !nlo)) *why = "null interval array";
  else return FDY_OK;
  return FDY_E_INVALID;
}

// Checks a table: sorted, non-overlapping, non-empty intervals below 2^64-1
// spanning less than 2^54 bytes, fewer than 2^32 of them.  *off_bits gets
// the OR of every lo - lo[0] (the starts' common alignment).
inline int check_table(const uint64_t* lo, const uint64_t* hi, const uint64_t* nlo, uint64_t n, uint32_t policy,
                       uint64_t* off_bits, std::string* why) {
  auto err = [why](int code, const std::string& msg) {
    *why = msg;
    return code;
  };
  *off_bits = 0;
  if (const int rc = check_table_args(lo, hi, nlo, n, policy, why)) return rc;
  if (n == 0) return FDY_OK;
  // One pass without branches; a table that fails is walked again for the
  // first interval at fault.
  uint64_t bits = 0, bad = (uint64_t)!interval_ok(lo[0], hi[0], lo[0]);
  for (uint64_t i = 1; i < n; ++i) {
    bad |= (uint64_t)!interval_ok(lo[i], hi[i], hi[i - 1]);
    bits |= lo[i] - lo[0];
  }
  for (uint64_t i = 0; bad && i < n; ++i) {
    if (lo[i] >= hi[i]) return err(FDY_E_INVALID, "interval " + std::to_string(i) + " is empty (lo >= hi)");
    if (hi[i] == UINT64_MAX) return err(FDY_E_INVALID, "interval " + std::to_string(i) + " ends at 2^64-1");
    if (i && hi[i - 1] > lo[i])
      return err(FDY_E_INVALID, "intervals " + std::to_string(i - 1) + " and " + std::to_string(i) +
                                    " overlap or are not sorted by lo");
  }
  if (n > 0xFFFFFFF0ull) return err(FDY_E_INVALID, "more than 2^32 intervals");
  if ((hi[n - 1] - lo[0]) >> 54) return err(FDY_E_INVALID, "intervals span more than 2^54 bytes");
  *off_bits = bits;
  return FDY_OK;
}

// The line width for at most `target` root lines over [lo_min, hi_max]: the
// smallest power of two, and at most 2^31 so offsets inside a line fit in 31
// bits (a span of 2^47, a process's whole address space, then takes at most
// 2^16 root lines).
inline IndexShape shape_for(uint64_t span, uint64_t target) {
  IndexShape s{0, 0};
  while ((span >> s.shift) + 1 > target) ++s.shift;
  if (s.shift > kMaxLineShift) s.shift = kMaxLineShift;
  s.nb = (span >> s.shift) + 1;  // w - lo_min <= span, so (w - lo_min) >> shift < nb
  return s;
}

// The root lines of a checked table of n intervals over `span` bytes, at most
// `root_lines_per_interval` per interval rounded up to a power of two in all.
inline IndexShape line_shape(uint64_t span, uint64_t n, uint64_t root_lines_per_interval) {
  uint64_t target = 1;
  while (target < root_lines_per_interval * n) target <<= 1;
  return shape_for(span, target);
}

// First address of root line b.
__host__ __device__ inline uint64_t root_start(uint64_t lo0, uint32_t shift, uint64_t b) {
  const uint64_t off = b << shift;  // b <= nb, so no overflow below 2^55
  return off > UINT64_MAX - lo0 ? UINT64_MAX : lo0 + off;
}

// The intervals root line b's range [s0, s1) holds: i, the last with
// lo <= s0 (lo[0] <= s0 always), and i + 1 .. j, those starting inside it.
__host__ __device__ inline void root_range(const uint64_t* lo, uint64_t n, uint64_t s0, uint64_t s1, uint64_t* i,
                                           uint64_t* j) {
  uint64_t a = 0, b = n;  // first lo > s0
  while (a < b) {
    const uint64_t mid = (a + b) >> 1;
    if (lo[mid] <= s0) a = mid + 1;
    else b = mid;
  }
  *i = a ? a - 1 : 0;
  uint64_t c = *i, d = n;  // first lo >= s1
  while (c < d) {
    const uint64_t mid = (c + d) >> 1;
    if (lo[mid] < s1) c = mid + 1;
    else d = mid;
  }
  *j = c ? c - 1 : 0;
  if (*j < *i) *j = *i;
}

// A fence line's children for m intervals (m > kLeafIntervals): up to 15
// leaves; past 60 intervals, the fewest children one level deeper (capacity
// `big`) beside children of capacity `small`, so that most intervals stay
// as shallow as the count allows.  Child c holds size(c) intervals.
struct FenceKids {
  uint32_t kids;
  uint64_t m, small, t, q, r;  // past 60: 15 - t children of `small`, then t of q + 1 (the first r) or q
  __host__ __device__ explicit FenceKids(uint64_t m_) : m(m_), small(0), t(0), q(0), r(0) {
    constexpr uint64_t kKids = kLineFences + 1;
    if (m <= kKids * kLeafIntervals) {
      kids = (uint32_t)((m + kLeafIntervals - 1) / kLeafIntervals);
      return;
    }
    kids = (uint32_t)kKids;
    uint64_t big = kKids * kLeafIntervals;
    small = kLeafIntervals;
    while (kKids * big < m) {
      small = big;
      big *= kKids;
    }
    t = (m - kKids * small + (big - small) - 1) / (big - small);  // 1 .. 15 deeper children
    const uint64_t rest = m - (kKids - t) * small;
    q = rest / t;
    r = rest % t;
  }
  __host__ __device__ uint64_t size(uint32_t c) const {
    if (!small) return c + 1 < kids ? kLeafIntervals : m - (uint64_t)c * kLeafIntervals;
    const uint64_t n_small = kLineFences + 1 - t;
    if (c < n_small) return small;
    return q + (c - n_small < r ? 1 : 0);
  }
};

// Lines below a root line whose range holds m intervals.  A fence line's
// children take at most three sizes, so the count walks a short list of
// {size, multiplicity} pairs (each level adds at most three, and 2^32
// intervals take eight levels): `size` and `mult` hold kSubtreeStack each
// (in LDS on the device, where an array in registers would be private
// memory that the runtime sizes for every lane of the GPU).
constexpr uint32_t kSubtreeStack = 24;
__host__ __device__ inline uint64_t subtree_lines(uint64_t m, uint64_t* size, uint64_t* mult) {
  uint32_t top = 0;
  uint64_t total = 0;
  if (m > kLeafIntervals) {
    size[0] = m;
    mult[0] = 1;
    top = 1;
  }
  while (top) {
    --top;
    const uint64_t k = mult[top];
    const FenceKids f(size[top]);
    total += k * f.kids;
    if (!f.small) continue;  // leaves only
    const uint64_t run_size[3] = {f.small, f.q + 1, f.q};
    const uint64_t run_mult[3] = {kLineFences + 1 - f.t, f.r, f.t - f.r};
    for (uint32_t e = 0; e < 3; ++e)
      if (run_mult[e] && run_size[e] > kLeafIntervals && top < kSubtreeStack) {
        size[top] = run_size[e];
        mult[top] = k * run_mult[e];
        ++top;
      }
  }
  return total;
}

// The end field of interval k in a line from s0.
__host__ __device__ inline uint32_t slot_end(uint64_t s0, uint64_t hi) {
  if (hi < s0) return 0;
  const uint64_t e = hi - s0 + 1;
  return e > 0xFFFFFFFFull ? 0xFFFFFFFFu : (uint32_t)e;
}

// A leaf line whose range from s0 holds intervals i
// (lo[i] <= s0, the last such) .. j.
__host__ __device__ inline RelocLine leaf_line(uint64_t s0, uint64_t i, uint64_t j, const uint64_t* lo,
                                               const uint64_t* hi, const uint64_t* nlo) {
  RelocLine L;
  L.s[0] = RelocSlot{0, slot_end(s0, hi[i]), nlo[i] - lo[i]};
  for (uint32_t k = 1; k < kLineSlots; ++k) {
    if (i + k <= j) L.s[k] = RelocSlot{(uint32_t)(lo[i + k] - s0), slot_end(s0, hi[i + k]), nlo[i + k] - lo[i + k]};
    else L.s[k] = RelocSlot{kLineNone, 0, 0};
  }
  return L;
}

// The line at `at` whose range from s0 holds intervals i (lo[i] <= s0, the
// last such) .. j: a leaf for up to four, else a fence line whose children
// take the next free lines (*next on), each holding until it is placed the
// {s0, i, j} it is to be placed with.
__host__ __device__ inline void place_line(RelocLine* line, uint64_t at, uint64_t s0, uint64_t i, uint64_t j,
                                           const uint64_t* lo, const uint64_t* hi, const uint64_t* nlo,
                                           uint64_t* next) {
  const uint64_t m = j - i + 1;
  if (m <= kLeafIntervals) {
    line[at] = leaf_line(s0, i, j, lo, hi, nlo);
    return;
  }
  // A fence line, written field by field in place (a fence array indexed
  // at run time would be private memory on the device).
  const FenceKids f(m);
  const uint64_t base = *next;
  *next += f.kids;
  line[at].s[0].lo = kLineFence;
  line[at].s[0].end = (uint32_t)base;
  uint32_t* fence = line_fences(line[at]);
  uint64_t ci = i;
  for (uint32_t c = 0; c < f.kids; ++c) {
    if (c) fence[c - 1] = (uint32_t)(lo[ci] - s0);  // a start inside the line: 0 < lo - s0 < 2^31
    RelocLine P;  // pending: {s0, i, j} of the child
    P.s[0] = RelocSlot{0, 0, c ? lo[ci] : s0};
    P.s[1] = RelocSlot{0, 0, ci};
    P.s[2] = RelocSlot{0, 0, ci + f.size(c) - 1};
    P.s[3] = RelocSlot{0, 0, 0};
    line[base + c] = P;
    ci += f.size(c);
  }
  for (uint32_t e = f.kids - 1; e < kLineFences; ++e) fence[e] = kLineNone;
}

// Root line b and every line below it, its descendants taking lines base ..
// base + subtree_lines(j - i + 1) - 1 breadth first (children of one line
// together), each placed after its parent.
__host__ __device__ inline void place_root(RelocLine* line, uint64_t b, uint64_t s0, uint64_t i, uint64_t j,
                                           const uint64_t* lo, const uint64_t* hi, const uint64_t* nlo,
                                           uint64_t base) {
  uint64_t next = base;
  place_line(line, b, s0, i, j, lo, hi, nlo, &next);
  for (uint64_t at = base; at < next; ++at) {
    const RelocLine P = line[at];  // this thread's own pending line
    place_line(line, at, P.s[0].delta, P.s[1].delta, P.s[2].delta, lo, hi, nlo, &next);
  }
}

// The whole index of root lines on the host.
inline int build_reloc_index(const uint64_t* lo, const uint64_t* hi, const uint64_t* nlo, uint64_t n,
                             uint32_t policy, HostIndex* out, std::string* why,
                             uint64_t root_lines_per_interval = kRootLinesPerInterval) {
  std::memset(&out->dev, 0, sizeof(out->dev));
  uint64_t off_bits;
  const int rc = check_table(lo, hi, nlo, n, policy, &off_bits, why);
  if (rc || n == 0) return rc;
  const IndexShape sh = line_shape(hi[n - 1] - lo[0], n, root_lines_per_interval);
  std::vector<uint64_t> ri(sh.nb), rj(sh.nb), base(sh.nb);
  uint64_t total = sh.nb;
  for (uint64_t b = 0; b < sh.nb; ++b) {
    root_range(lo, n, root_start(lo[0], sh.shift, b), root_start(lo[0], sh.shift, b + 1), &ri[b], &rj[b]);
    base[b] = total;
    uint64_t st_size[kSubtreeStack], st_mult[kSubtreeStack];
    total += subtree_lines(rj[b] - ri[b] + 1, st_size, st_mult);
    if (total > kMaxIndexLines) {
      *why = "interval index too large";
      return FDY_E_INVALID;
    }
  }
  out->line.assign(total, RelocLine{});
  for (uint64_t b = 0; b < sh.nb; ++b)
    place_root(out->line.data(), b, root_start(lo[0], sh.shift, b), ri[b], rj[b], lo, hi, nlo, base[b]);
  out->dev.n = n;
  out->dev.lo_min = lo[0];
  out->dev.hi_max = hi[n - 1];
  out->dev.span = hi[n - 1] - lo[0] + (policy ? 1 : 0);
  out->dev.delta = nlo[0] - lo[0];
  out->dev.shift = sh.shift;
  out->dev.policy = policy;
  return FDY_OK;
}

// ---- the two-level index ---------------------------------------------------
//
// Root entries over equal address ranges.  An entry inside whose range no
// interval starts answers by itself; the others name the lines that hold
// their range's intervals four at a time (RelocRoot).  With 28 intervals or
// fewer a search is one entry and one leaf line; past that (or past four
// where the starts are not on the fences' unit) the entry names the top line
// of a tree of full lines: leaves of four intervals, fence lines of 15
// children, every level's lines together, the top level first.

constexpr uint64_t kLineKids = kLineFences + 1;
constexpr uint64_t kRootIntervals = (kRootFences + 1) * kLeafIntervals;

struct RootShape {
  uint32_t shift, fence_shift;
  uint64_t nb;
  bool exact;  // every start lies on a multiple of 2^fence_shift from its entry's first address
};

// Root entries of a checked table: one to two per interval up to 2^16 (1 MB:
// with their lines they stay in the L2s), then one per four to eight.  On the
// relocation workloads' mix of sizes no lookup then meets a tree at 40,000
// intervals (2% of a 64 GiB archive region's do with a quarter of the entries),
// 2% at 200,000 and more.  Where the starts' alignment is coarser than 1/2^15
// of an entry's range, narrower entries (up to four per interval, and up to
// 32768: 512 KB) make the fences exact.
inline RootShape root_shape(const uint64_t* lo, const uint64_t* hi, uint64_t n, uint64_t off_bits) {
  RootShape r{0, 0, 0, true};
  if (n == 0) return r;
  const uint64_t span = hi[n - 1] - lo[0];
  uint64_t t = 1;
  while (t < 2 * n && (t < (1ull << 16) || 4 * t < n)) t <<= 1;
  IndexShape s = shape_for(span, t);
  uint32_t align = 0;  // starts are multiples of 2^align apart
  while (align < kMaxLineShift && !((off_bits >> align) & 1)) ++align;
  if (s.shift > kRootFenceBits + align) {
    const uint64_t nb = (span >> (kRootFenceBits + align)) + 1;
    if (nb <= std::max<uint64_t>(4 * n, 32768)) s = IndexShape{kRootFenceBits + align, nb};
  }
  r.shift = s.shift;
  r.nb = s.nb;
  r.fence_shift = s.shift > kRootFenceBits ? s.shift - kRootFenceBits : 0;
  r.exact = r.fence_shift <= align;
  return r;
}

// The first interval of a root entry's range: the last with lo <= s0, its
// first address, when e intervals start before s0.
__host__ __device__ inline uint64_t root_first(const uint64_t* lo, uint64_t n, uint64_t s0, uint64_t e) {
  return e < n && lo[e] == s0 ? e : e - 1;
}

// Whether m intervals are leaves right below their root entry.
__host__ __device__ inline bool root_flat(uint64_t m, bool exact) {
  return m <= kLeafIntervals || (exact && m <= kRootIntervals);
}

// Lines below a root entry whose range holds m intervals (the last one
// starting at or before its first address among them).
__host__ __device__ inline uint64_t root_lines(uint64_t m, bool exact) {
  if (m == 1) return 0;  // a direct entry
  uint64_t w = kLeafIntervals, total = (m + w - 1) / w;
  if (root_flat(m, exact)) return total;
  while (w < m) {
    w *= kLineKids;
    total += (m + w - 1) / w;
  }
  return total;
}

// The root entry from s0 whose range holds intervals i .. j, its lines from
// line `first` on.
__host__ __device__ inline RelocRoot root_entry(uint64_t s0, uint64_t i, uint64_t j, const uint64_t* lo,
                                                const uint64_t* hi, const uint64_t* nlo, uint32_t fence_shift,
                                                bool exact, uint64_t first) {
  RelocRoot r;
  if (i == j) {
    const uint64_t delta = nlo[i] - lo[i];
    r.line = kRootDirect;
    r.word[0] = slot_end(s0, hi[i]);
    r.word[1] = (uint32_t)delta;
    r.word[2] = (uint32_t)(delta >> 32);
    return r;
  }
  const bool flat = root_flat(j - i + 1, exact);
  uint32_t levels = 0;  // of fence lines: at most 8 below 2^32 intervals
  if (!flat)
    for (uint64_t w = kLeafIntervals; w < j - i + 1; w *= kLineKids) ++levels;
  r.line = (uint32_t)first | (flat ? 0u : kRootTree);
  for (uint32_t e = 0; e < kRootFences / 2; ++e) {
    uint32_t f[2];
    for (uint32_t h = 0; h < 2; ++h) {
      const uint64_t k = i + (uint64_t)(2 * e + h + 1) * kLeafIntervals;
      f[h] = flat && k <= j ? (uint32_t)((lo[k] - s0) >> fence_shift) : 0xFFFFu;
    }
    r.word[e] = f[0] | (f[1] << 16);
  }
  if (!flat) r.word[kRootFences / 2 - 1] = 0xFFFFu | (0xFFFFu - kRootLevels + levels) << 16;
  return r;
}

// Line 0, a leaf that moves nothing.
__host__ __device__ inline RelocLine null_line() {
  RelocLine L;
  L.s[0] = RelocSlot{0, 0, 0};
  for (uint32_t k = 1; k < kLineSlots; ++k) L.s[k] = RelocSlot{kLineNone, 0, 0};
  return L;
}

// Line k of the root_lines() lines (the first at `first`) below an entry
// whose range from s0 holds intervals i .. j.
__host__ __device__ inline void place_below(RelocLine* line, uint64_t first, uint64_t k, uint64_t s0, uint64_t i,
                                            uint64_t j, const uint64_t* lo, const uint64_t* hi, const uint64_t* nlo,
                                            bool exact) {
  const uint64_t m = j - i + 1;
  // The level holding line k: intervals per line, its first line, its lines.
  uint64_t w = kLeafIntervals, at = 0, size = 0;
  if (!root_flat(m, exact)) {
    while (w < m) w *= kLineKids;
    for (;; w /= kLineKids) {
      size = (m + w - 1) / w;
      if (k < at + size) break;
      at += size;
    }
  }
  const uint64_t a = i + (k - at) * w;          // the line's first interval
  const uint64_t B = k == at ? s0 : lo[a];      // and first address
  const uint64_t z = j - a < w ? j : a + w - 1; // its last interval
  if (w == kLeafIntervals) {
    line[first + k] = leaf_line(B, a, z, lo, hi, nlo);
    return;
  }
  const uint64_t cw = w / kLineKids;  // intervals per child
  uint32_t* L = reinterpret_cast<uint32_t*>(line + first + k);
  L[0] = kLineFence;
  L[1] = (uint32_t)(first + at + size + (k - at) * kLineKids);
  for (uint32_t e = 0; e < kLineFences; ++e) {
    const uint64_t c = a + (e + 1) * cw;
    L[2 + e] = c <= z ? (uint32_t)(lo[c] - B) : kLineNone;
  }
}

// The whole two-level index on the host (what the device build is held to).
struct HostRootIndex {
  std::vector<RelocRoot> root;
  std::vector<RelocLine> line;
  RelocDev dev{};
};
inline int build_root_index(const uint64_t* lo, const uint64_t* hi, const uint64_t* nlo, uint64_t n, uint32_t policy,
                            HostRootIndex* out, std::string* why) {
  std::memset(&out->dev, 0, sizeof(out->dev));
  uint64_t off_bits;
  const int rc = check_table(lo, hi, nlo, n, policy, &off_bits, why);
  if (rc || n == 0) return rc;
  const RootShape sh = root_shape(lo, hi, n, off_bits);
  out->root.resize(sh.nb);
  out->line.assign(1, null_line());
  uint64_t e = 0;
  for (uint64_t b = 0; b < sh.nb; ++b) {
    const uint64_t s0 = root_start(lo[0], sh.shift, b), s1 = root_start(lo[0], sh.shift, b + 1);
    const uint64_t i = root_first(lo, n, s0, e);
    while (e < n && lo[e] < s1) ++e;
    const uint64_t first = out->line.size(), below = root_lines(e - i, sh.exact);
    out->root[b] = root_entry(s0, i, e - 1, lo, hi, nlo, sh.fence_shift, sh.exact, first);
    out->line.resize(first + below);
    for (uint64_t k = 0; k < below; ++k)
      place_below(out->line.data(), first, k, s0, i, e - 1, lo, hi, nlo, sh.exact);
  }
  out->dev.n = n;
  out->dev.lo_min = lo[0];
  out->dev.hi_max = hi[n - 1];
  out->dev.span = hi[n - 1] - lo[0] + (policy ? 1 : 0);
  out->dev.delta = nlo[0] - lo[0];
  out->dev.shift = sh.shift;
  out->dev.fence_shift = sh.fence_shift;
  out->dev.policy = policy;
  return FDY_OK;
}

}  // namespace fdy
