// merge.hpp -- the merge of equal subtrees and the words, for every level of a build (build.hip) or
// of a forest (forest.hip).  See merge.hip.
#pragma once

#include "build_parts.hpp"

namespace cpvs {

// One octree level with nodes.
struct MLevel {
    const u32* mask;
    const u32* cstart;  // first child of each node (null at the leafmask level)
    u32* id;            // identities (ChildIds)
    u64* tab;           // table merge: the level's table; sort merge: one entry per node.  k_offsets
                        // leaves rank << 32 | word offset in each first occurrence's entry
    uint8_t* flag;      // words of the node if it is its key's first occurrence, else 0
    u32* uniq;          // rank -> first occurrence
    u32* off;           // rank -> word offset in the level
    u32 n, slots;
    int L;
    u32 leaf;           // 1: leafmask nodes (two words per partial child)
    u32 lone;           // 1: not merged (a single build's root), so without identities
    u32 late;           // 1: its insert leaves the key compares to merge_write (kLateMax)
};

// The levels, deepest first; tile0[k] is level k's first tile of kTileNodes nodes.
struct MArgs {
    int nlev;
    u32 tile0[kMaxLevels + 1];
    MLevel lv[kMaxLevels];
    const u64* leafm;
    const u32* heads;  // leaf level: each node's run head
    bool sorted;       // identities of the sort merge
    // The level that k's children lie in, or -1.
    __host__ __device__ int child(int k) const { return (k > 0 && lv[k - 1].L + 1 == lv[k].L) ? k - 1 : -1; }
};

constexpr u32 kTileThreads = 256;
constexpr u32 kTilePer = 8;  // nodes per thread; k_offsets loads their flags as 8 bytes
constexpr u32 kTileNodes = kTileThreads * kTilePer;

constexpr u32 kLateMax = 1u << 18;  // nodes of a level whose compares a single build leaves to merge_write

inline size_t tile_pre_count(size_t tiles) { return tiles + kMaxLevels + 1; }
inline size_t flag_words(size_t n) { return (n + 7) / 8; }  // 64-bit words of MLevel::flag

// Launches.  insert_level: identities of level k of `a` by its table (a.lv[k].tab, cleared before);
// hash: the leaf level's key hashes from the leaf kernel, or null.
void merge_insert(const MArgs& a, int k, const u64* hash, u32* meta, u32 hbits, hipStream_t s);
// The sort merge of level k; scratch arrays of n entries each, seg and sort_scratch as in build.hip.
struct SortScratch {
    u32 *skey, *sval, *ktmp, *vtmp, *seg, *sort_scratch, *scan_scratch;
};
void merge_sort_level(const MArgs& a, int k, const SortScratch& t, u32* meta, hipStream_t s);
// After every level has its identities: first occurrences, their ranks and word offsets, level totals in meta.  tile_sums: one entry per tile;
// tile_pre: tile_pre_count(tiles).  R >= 0: a single build, whose level bases and root mask go to meta too.  host_meta
// (pinned, may be null) receives meta.
void merge_finish(const MArgs& a, u32* tile_sums, ulonglong2* tile_pre, u32* meta, int R, u32* host_meta, hipStream_t s);
// A single build's words, level bases from meta, into out; nothing when they exceed cap words.  Counts
// the late levels' key collisions in meta (kMetaColl).
void merge_write(const MArgs& a, u32* meta, u32* out, u64 cap, hipStream_t s);

// Empties `slots` table slots (where no leaf kernel does).
void table_clear(u64* tab, u64 slots, hipStream_t s);

}  // namespace cpvs
