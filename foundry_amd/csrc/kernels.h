// kernels.h -- launch wrappers for the restore kernels (kernels.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/foundry_restore.h"
#include "restore_dev.h"

namespace fdy {

// Default RestoreArgs::hash_wait_spins: about 1 ms of s_sleep.
constexpr uint32_t kHashWaitSpins = 1u << 14;

// Everything the restore kernels read or write for one archive.
struct RestoreArgs {
  const uint8_t* img;         // .cugraph images, each 256-B aligned
  const DevGraph* graphs;
  const CrcConsts* cc;
  uint32_t num_graphs;
  uint32_t num_slots;
  uint32_t num_chunks;        // node chunks over all graphs
  uint2* chunk_gt;            // per node chunk: {graph, template} (the grouping pass writes both)
  uint32_t num_units;         // digest units (4 KB slices of keys and dependency tables) over all graphs
  const DigestUnit* units;
  NodeChunk* chunks;          // per node chunk
  uint64_t* digests;          // 4 per graph
  const uint32_t* explicit_template;  // or null
  uint64_t* key_hash;                 // per graph: the grouping pass's published key hash (epoch-tagged)
  uint32_t epoch;                     // this restore's tag for published key hashes (1..65535)
  uint32_t hash_wait_spins;           // s_sleep rounds the grouping scan waits for an unpublished hash
                                      // before hashing that key itself (0: at once)
  uint32_t* template_of;
  uint32_t* status;
  uint32_t* gwords;
  uint64_t* pbytes;           // param bytes per graph
  uint8_t* node_flags;
  NodeDesc* node_desc;
  uint64_t* node_ptrs;        // 2 per node
  uint32_t* tile_node;        // per slot
  SlotDesc* tslot_desc;       // descriptors of the template graphs' slots holding words (capacity: num_slots)
  uint32_t* tslot_count;      // entries of tslot_desc
  SlotDesc* slot_desc;        // per slot
  uint64_t* aux;              // ragged-word sources (per word), or null until a restore finds a ragged node
  uint64_t* image;            // relocated param images R
  uint32_t* live_src;         // per node
  uint32_t* live_cur;         // per graph
  fdy_override* ovr;          // override records: graph g's in canonical order from index word_base(g) >> rec_shift,
                              // at most ((word_base + word_cap) >> rec_shift) - (word_base >> rec_shift) of them
  uint32_t rec_shift;         // 0: a record per capacity word; kCompactShift: one per 2^kCompactShift
  uint32_t cand_cap;          // candidates in a sub-range's own region (kSubWords, or fewer with spill space)
  uint32_t spill_cap;         // candidates a slot's sub-ranges can spill past their own regions (0: none)
  Candidate* cand;            // per slot: kSubsPerSlot regions of cand_cap candidates, then spill_cap more
  uint32_t* slot_spill;       // per slot: spill entries taken by this restore
  uint32_t* sub_off;          // per (slot, sub-range): first entry of its candidate list in the slot's area
  uint32_t* sub_count;        // per (slot, sub-range): candidates | compared candidates << 16
  uint32_t* slot_rec;         // records per slot
  uint32_t* restore_flags;    // kFlag* raised by this restore
  uint64_t* node_pbytes;      // param bytes per node (nodes the first node pass handles itself)
  RelocDev reloc;
};

hipError_t launch_group(const RestoreArgs& a, hipStream_t s);
hipError_t launch_node(const RestoreArgs& a, hipStream_t s);
hipError_t launch_diff_templates(const RestoreArgs& a, hipStream_t s);
hipError_t launch_diff_members(const RestoreArgs& a, hipStream_t s);
hipError_t launch_diff_search(const RestoreArgs& a, hipStream_t s);

// Closing the gaps in override arrays (k_repack).
struct RepackArgs {
  const DevGraph* graphs;
  const uint32_t* sub_count;
  const uint32_t* slot_rec;
  fdy_override* ovr;
  uint32_t num_graphs;
  uint32_t rec_shift;
};
hipError_t launch_repack(const RepackArgs& a, hipStream_t s);

struct SwitchArgs {
  const fdy_override* ovr_cur;  // current graph's overrides
  uint64_t n_cur;
  const fdy_override* ovr_new;  // target graph's overrides
  uint64_t n_new;
  const uint64_t* tmpl_image;   // R of the template
  uint64_t* live;               // live image of the template
  const uint8_t* flags_cur;     // node flags of the current graph
  const uint8_t* flags_new;     // node flags of the target
  uint32_t* live_src;           // node sources of the template's group
  uint8_t* dirty;               // or null: per node, set to 1 when the node must be re-set
  uint32_t num_nodes;           // template's node count
  uint32_t target;
  uint32_t tmpl;
};
hipError_t launch_switch(const SwitchArgs& a, hipStream_t s);

// Up to kSwitchBatch switches of different groups in one launch.
constexpr uint32_t kSwitchBatch = 16;
struct SwitchBatch {
  SwitchArgs sw[kSwitchBatch];
  uint32_t end[kSwitchBatch];  // running block counts
  uint32_t n;
};
static_assert(sizeof(SwitchBatch) <= 2048, "a switch batch travels as kernel arguments");
// Blocks of one switch's scatter (the same split as launch_switch's).
uint32_t switch_blocks(const SwitchArgs& a);
hipError_t launch_switch_many(const SwitchBatch& b, hipStream_t s);

// A sequence of switches in one launch, cut by groups and by tiles of
// kSeqWords template words: a workgroup makes all of its group's switches
// within its tile (and its share of the group's nodes), so that no workgroup
// waits for another.
constexpr uint32_t kSeqWords = 1024;
struct SeqGraph {
  uint64_t rec;       // first override record
  uint64_t num_rec;
  uint64_t off;       // first entry of `offs`: per tile, the graph's records before it (and in all)
  uint64_t live;      // (template) first word of the live image
  uint64_t image;     // (template) first word of R
  uint64_t node_base;
  uint32_t num_nodes;
  uint32_t words;     // words of the graph's template
};
// Tiles of a template of `words` words, at least one.
__host__ __device__ inline uint32_t seq_tiles(uint32_t words) {
  return words ? (uint32_t)(((uint64_t)words + kSeqWords - 1) / kSeqWords) : 1u;
}
// The tables of graphs first .. first + num_graphs - 1, whose entries travel
// as kernel arguments (nothing is staged, so nothing waits): graphs[first + i]
// = g[i], and offs[g.off + k] = the records of g whose word lies before tile
// k, k = 0 .. seq_tiles.
constexpr uint32_t kSeqIndexGraphs = 64;
struct SeqIndexArgs {
  SeqGraph* graphs;
  const fdy_override* ovr;
  uint32_t* offs;
  uint32_t first;
  uint32_t num_graphs;
  SeqGraph g[kSeqIndexGraphs];
};
static_assert(sizeof(SeqIndexArgs) <= 4096, "graph entries travel as kernel arguments");
hipError_t launch_seq_index(const SeqIndexArgs& a, hipStream_t s);

constexpr uint32_t kSeqGroups = 32;    // groups per launch
constexpr uint32_t kSeqTargets = 704;  // list entries per launch: every group's current graph, then its targets
struct SwitchSeq {
  const SeqGraph* graphs;
  const uint32_t* offs;
  const fdy_override* ovr;
  const uint64_t* image;
  uint64_t* live;
  const uint8_t* flags;    // node flags of all graphs
  uint32_t* live_src;
  uint32_t num_groups;
  uint32_t pad_;
  uint32_t tmpl[kSeqGroups];
  uint32_t end[kSeqGroups];        // running workgroup counts (a group's tiles)
  uint32_t first[kSeqGroups + 1];  // the group's entries of `target`
  uint32_t target[kSeqTargets];
};
static_assert(sizeof(SwitchSeq) <= 4096, "a sequence travels as kernel arguments");
hipError_t launch_switch_seq(const SwitchSeq& q, hipStream_t s);

// Copy of the dirty nodes' live words (or of every node's) into the host
// mirror of a group graph, with the dirty marks; clears the device marks.
struct MirrorArgs {
  const uint64_t* live;   // the group's live image
  const NodeDesc* desc;   // the template's node descriptors (gword, nwords)
  uint8_t* dirty;         // per node (device memory)
  uint64_t* h_live;       // device-visible host memory, same indexing as live
  uint8_t* h_dirty;       // device-visible host memory, per node
  uint32_t num_nodes;
  uint32_t all;           // 1: copy every node and mark it dirty
};
constexpr uint32_t kMirrorNodes = 64;  // nodes per block
hipError_t launch_mirror(const MirrorArgs& a, hipStream_t s);

// Relocates packed words through the table's two-level index, or (r.root
// null and more than one interval) through its root lines.
hipError_t launch_reloc_words(const RelocDev& r, const uint64_t* in, uint64_t* out, uint64_t n, hipStream_t s);

// A table's index built on the device (the builders of reloc_index.h).  The
// count launches write each workgroup's first line into block_sum and the
// line count into *total; the place launches then write the entries and
// lines (line holds *total of them).  launch_roots_*: the two-level index,
// kRootBlock root entries per workgroup.  launch_index_*: the index of root
// lines, one thread per root line, kIndexThreads per workgroup.
constexpr uint32_t kIndexThreads = 64;  // one wave: 24 KB of LDS for the subtree counts
constexpr uint32_t kRootBlock = 256;
struct IndexArgs {
  const uint64_t* lo;   // the table, on the device
  const uint64_t* hi;
  const uint64_t* nlo;
  uint64_t n;           // intervals (> 0)
  uint64_t nb;          // root lines, or root entries
  uint32_t shift;       // their width: 2^shift bytes
  uint32_t fence_shift; // two-level index: the fences' unit
  uint32_t exact;       // two-level index: every start is on that unit
  uint32_t pad_;
  uint32_t* ends;       // two-level index: per root entry, the intervals starting before its range's end
  uint64_t* block_sum;  // one per workgroup of the count launch
  uint64_t* total;
  RelocRoot* root;      // two-level index
  RelocLine* line;
};
// The table's check (check_table's, of the intervals): workgroup b writes
// {whether an interval is at fault, the OR of its starts' offsets} to
// part[2 * b]; returns the workgroups in *blocks, at most kTableBlocks.
constexpr uint32_t kTableBlocks = 256;
hipError_t launch_table_check(const IndexArgs& a, uint64_t* part, uint32_t* blocks, hipStream_t s);
hipError_t launch_index_count(const IndexArgs& a, hipStream_t s);
hipError_t launch_index_place(const IndexArgs& a, hipStream_t s);
hipError_t launch_roots_count(const IndexArgs& a, hipStream_t s);
hipError_t launch_roots_place(const IndexArgs& a, hipStream_t s);

// A memset node of a restored graph, run as a kernel node: `height` rows of
// `row_bytes` bytes, `pitch` bytes apart, each byte k of a row taking byte
// k % 4 of `pattern` (the value replicated to 32 bits).
struct FillArgs {
  uint8_t* dst;
  uint64_t pitch;
  uint64_t row_bytes;
  uint64_t height;
  uint32_t pattern;
  uint32_t pad_;
};
constexpr uint32_t kFillThreads = 256;
// Host handle of the fill kernel, for hipKernelNodeParams::func.
void* fill_kernel();
dim3 fill_grid(const FillArgs& f);

}  // namespace fdy
