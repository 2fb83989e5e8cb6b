// build.hip -- CompressedShadow::create on the device (src/CompressedShadow.cpp:49-392).
//
// The reference builds an uncompressed 9/17-word octree on the host, merges equal subtrees
// level by level with a linear search, drops the holes and relayouts the array.  Here every
// octree level is a set of compact per-node arrays, processed as:
//
//   1. BFS classification, root -> level 3 (or 0): one thread per node reads its 2x2 pyramid
//      texels and writes the 16-bit child mask; an exclusive scan of the partial-child counts
//      gives each node's first child, and the scan's output stage writes the children's
//      coordinates in (parent, child index) order -- the reference's breadth-first order.
//   2. Leaves (level 2): smooth 8x8 texel columns (level-3 texels) one per lane, walls one per wave.
//      The leaf nodes of a column are its partial level-3 cells, contiguous in z; a node equal to its
//      z-neighbour (the common case along walls) is copied, not recomputed.  The level-3 scan records
//      where each (column, z) leaf sits in breadth-first order.
//   3. Merge, bottom-up from the leaves to the root's children (merge.hip).  Key = (mask, partial
//      leafmasks) or (mask, identities of the partial children).  Default (a): the key's 64-bit hash
//      goes into an open-addressing table whose 64-bit slots hold a hash tag and the smallest node
//      index with it; the slot is the node's identity, and full keys are compared within a slot: a
//      collision re-runs the build with (b).  (b): a stable LSD radix sort of (32-bit hash, node
//      index), segment starts by a max-scan and a full-key compare against the segment head (a
//      mismatch falls back to a scan of the segment).
//   4. Compress: first occurrences, their ranks and word offsets in index order, as mergeLevel's linear
//      search yields (src/CompressedShadowUtil.h:154-182), level bases root first, then one pass writes
//      [mask, absolute child offsets] or [mask, lo, hi, ...] (src/CompressedShadow.cpp:326-392).
#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstring>

#include "merge.hpp"

namespace cpvs {

__global__ __launch_bounds__(256) void k_classify(const u64* __restrict__ coord, u32 count, const float2* __restrict__ lv,
                                                  const float* __restrict__ depth, u32 N, int L, u32 T,
                                                  u32* __restrict__ mask_out) {
    const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count) return;
    mask_out[i] = classify_node(coord[i], lv, depth, N, L, T);
}

// ---------------------------------------------------------------------------------------
// 2. Leaves: createChildmask1x1x8 + createLeafmask (src/CompressedShadowUtil.cpp:59-99).
//
// Slice s of leaf node z3 (depth z = 8*z3 + s) is lit at texel t iff float(z) + 0.5 <= d_t*H
// (absoluteVisible, H = N*T), i.e. iff u_t >= s with f_t = floor(d_t*H - 0.5) and
// u_t = f_t - 8*z3.  With one texel per lane, slice s's leafmask is B_s = ballot(u >= s): eight
// compares give the whole node.  The B_s are nested (B_0 >= B_1 >= ...), so the slices with
// B_s all ones (fully lit) come first, then the partial ones, then those with B_s = 0 (shadow).
// Everything past the compares is wave-uniform scalar work: the childmask, the key hash over
// (mask, partial leafmasks), and the lane placement of the leafmasks for the store.
// Node z3 equals node z3-1 of the same column unless some u_t lies in [-8, 6].
// ---------------------------------------------------------------------------------------

// ---------------------------------------------------------------------------------------
// The leaf kernels.  k_leaf_lanes walks one column per lane (leaf_lane), for launches with enough
// columns to fill the chip that way, and leaves walls and steep columns to k_leaf_waves, one column
// per wave and one texel per lane (leaf_column).  In the latter:
// * Which nodes differ from their predecessor follows from the texels alone.  With
//   h_t = f_t + 8 - 8*zs, node q changes iff some h_t - 8q lies in [0, 14]: q = floor(h_t/8), or
//   q = floor(h_t/8) - 1 when h_t mod 8 != 7.  Each texel flags at most two nodes in LDS and a
//   ballot over the flags read back gives a chunk's changed nodes at once; only those (the run
//   heads) get compares.
// * Only a run's first node stores its mask and leafmasks: the merge and the final write read
//   those of first occurrences only, and a key's first occurrence is always the first node of a
//   run (breadth-first order grows with z inside a column).  Every node stores the breadth-first
//   index of its run's first node.
// * A run head's leafmasks go to the row at its own breadth-first index (8 slots per node), so the
//   leaf insert, the key compares and the write find them at the node's index, with no slot map.
// Measured at 8192^2 (1 M columns, 6.7 M nodes): 8 columns per wave for all, bound by instruction issue
// (vector units 73% busy, scalar 57%), 210 us; lanes 103 us and waves 34 us (49 before list_share) for the rest, whose
// columns hold most of the nodes (2, 4 and 8 of them in turn per wave took 51, 63 and 77 us: a wave
// waits for each column's chunks).  Small maps are all latency: 256^2 13 -> 4 us and 1024^2
// 17 -> 9 us with one column per wave instead of 8.
// Workgroups are dealt to the XCDs in turn (block b to XCD b mod kXcds), each XCD with its own L2.
// XCD x takes the contiguous units [x*chunk, (x+1)*chunk): neighbouring columns, whose 8-texel depth
// rows share 128-byte lines, are then read through one L2.  Of a list each XCD takes a contiguous
// eighth (list_share) where a wave takes one column; k_leaf_lanes' list (of a z-tile) fills only its
// first workgroups, 256 columns each, so there consecutive ones go to different XCDs.
// ---------------------------------------------------------------------------------------
__device__ inline LeafCol map_column(const LeafColumns& lc, const float* depth, u32 N, float HT, u32 col) {
    const uint4 ci = lc.info[col];
    const u32 x = even_bits(col), y = even_bits(col >> 1);
    return LeafCol{col, depth + ((size_t)(8 * y) * N + 8 * x), N, HT, ci.x, ci.y, (int)ci.z, 0u};
}

// kList: the columns col_list[0 .. *n_list), at most ncol (the z-tile's columns with leaf nodes, or
// those that k_leaf_lanes left), over which the waves stride; otherwise all ncol of them.
template <bool kList>
__global__ __launch_bounds__(64) void k_leaf_waves(LeafColumns lc, u32 ncol, const float* __restrict__ depth, u32 N, u32 T,
                                                   const float2* __restrict__ lv3, LeafOut o, u32 chunk,
                                                   u64* __restrict__ tab, u64 tab_slots,
                                                   const u32* __restrict__ col_list, const u32* __restrict__ n_list) {
    __shared__ uint8_t s_chg[128];
    const u32 b = blockIdx.x;
    const ListShare share = kList ? list_share(min(*n_list, ncol), b, gridDim.x)
                                  : ListShare{(b % kXcds) * chunk + b / kXcds, ncol, ncol};
    for (u32 u = share.u0; u < share.end; u += share.step) {
        const LeafCol c = map_column(lc, depth, N, (float)(N * T), kList ? col_list[u] : u);
        if (c.cnt) leaf_wave(c, lv3 + (size_t)even_bits(c.col >> 1) * lc.w3 + even_bits(c.col), o, s_chg, threadIdx.x);
    }
    clear_table(tab, tab_slots);  // after all the work: stores issued earlier would be waited for with the loads
}

template <bool kList>
__global__ __launch_bounds__(kLaneThreads) void k_leaf_lanes(LeafColumns lc, u32 ncol, const float* __restrict__ depth, u32 N,
                                                             u32 T, LeafOut o, u32 chunk, u64* __restrict__ tab,
                                                             u64 tab_slots, const u32* __restrict__ col_list,
                                                             const u32* __restrict__ n_list) {
    const u32 unit = kList ? blockIdx.x : (blockIdx.x % kXcds) * chunk + blockIdx.x / kXcds;
    const u32 n = kList ? min(*n_list, ncol) : ncol, u = unit * kLaneThreads + threadIdx.x;
    if (unit * kLaneThreads < n) {
        LeafCol c{};
        if (u < n) c = map_column(lc, depth, N, (float)(N * T), kList ? col_list[u] : u);
        leaf_lanes(c, o);
    }
    clear_table(tab, tab_slots);
}

// First launch after the scratch is laid out when no level is small: the root's coordinate, and
// the meta words zeroed (k_small_topdown does both otherwise).
__global__ void k_start(u64* root_coord, u64 root, u32* meta, u32 meta_words) {
    *root_coord = root;
    for (u32 i = 0; i < meta_words; ++i) meta[i] = 0u;
}

// ---------------------------------------------------------------------------------------
// Host orchestration.
// ---------------------------------------------------------------------------------------
namespace {

struct Level {
    u32 count = 0;
    u64* coord = nullptr;
    u32* mask = nullptr;
    u32* cstart = nullptr;
    u32* id = nullptr;
    u32* uniq = nullptr;
    u32* off = nullptr;
    uint8_t* flag = nullptr;
    u64* tab = nullptr;
    u32 slots = 0;
};

// ---------------------------------------------------------------------------------------
// Small levels in one workgroup.  The upper octree levels hold few nodes (at 8192^2 the levels
// above 6 hold a few thousand together), yet each costs about ten launches of the per-level
// path at several microseconds apiece.  A level of at most kSmallMax nodes is handled by one
// 1024-thread workgroup instead, all such levels in one launch per phase: top-down classification
// and child emission, and bottom-up inserts (hash tables in LDS).  Results are those of the
// per-level path.
// ---------------------------------------------------------------------------------------
// Measured at 8192^2: a limit of 4096 nodes beats 2048 (1.29 against 1.31 ms per build) and 8192
// (1.34 ms: one workgroup then spends more on the 7.9 K-node level than its per-level launches do).
constexpr u32 kSmallMax = 4096;
constexpr int kSmallThreads = 1024;
constexpr u32 kSmallPer = kSmallMax / kSmallThreads;  // nodes per thread
constexpr u32 kSmallSlots = 2 * kSmallMax;             // LDS table of 8-byte slots: 64 KB
inline u32 small_slots(u32 c) {
    u32 S = 64;
    while (S < 2 * c) S <<= 1;
    return S;
}

struct SmallArgs {
    int R, Ls, deepest;  // the small levels are [Ls, R]; deepest = lowest level with nodes
    u32 count[kMaxLevels];
    u64* coord[kMaxLevels];
    u32* mask[kMaxLevels];
    u32* cstart[kMaxLevels];
    u32* id[kMaxLevels];
    u64* tab[kMaxLevels];
    u32 slots[kMaxLevels];
    u32 n_below;       // nodes of the level below Ls
    const u32* heads;  // run heads when that level is the leaf level, else null
    const float2* lv[kMaxLevels];
    u32* meta;
};

// The levels' counts and arrays in LDS, and a uniform value read from there.  Looked up in the
// kernel's arguments level by level, each was a scalar load of its own from memory, on the one
// workgroup's critical path.
struct SmallLevels {
    u32 count[kMaxLevels], slots[kMaxLevels];
    u64* coord[kMaxLevels];
    u32 *mask[kMaxLevels], *cstart[kMaxLevels], *id[kMaxLevels];
    u64* tab[kMaxLevels];
    const float2* lv[kMaxLevels];
};
__device__ inline void load_levels(const SmallArgs& a, SmallLevels& s) {  // (a barrier before its use)
    const u32 t = threadIdx.x;
    if (t >= kMaxLevels) return;
    s.count[t] = a.count[t];
    s.slots[t] = a.slots[t];
    s.coord[t] = a.coord[t];
    s.mask[t] = a.mask[t];
    s.cstart[t] = a.cstart[t];
    s.id[t] = a.id[t];
    s.tab[t] = a.tab[t];
    s.lv[t] = a.lv[t];
}
__device__ inline u32 uniform(u32 v) { return __builtin_amdgcn_readfirstlane(v); }
template <class P>
__device__ inline P* uniform(P* p) {
    const u64 v = reinterpret_cast<u64>(p);
    return reinterpret_cast<P*>(((u64)uniform((u32)(v >> 32)) << 32) | uniform((u32)v));
}

// The small levels' cells and masks stay in LDS (cells in two buffers: a level and its children); only
// the children of the last small level, which the multi-workgroup path classifies, go to memory.  The
// pyramid levels up to kPyrWidth wide, which lie one behind the other, are copied to LDS at the start:
// a level then waits for LDS, not for memory.  Nodes are striped over the threads (consecutive lanes,
// consecutive children: contiguous nodes per thread put all lanes' stores in the same banks), and the
// rounds are a loop, not unrolled.  1024^2 25.3 -> 21.7 us, 8192^2 18.1 -> 16.2; what is left is one
// workgroup's chain of LDS reads, scans and stores, about 1 us a level, and its start.
constexpr u32 kPyrWidth = 64;
constexpr u32 kPyrTexels = (kPyrWidth * kPyrWidth - 1) / 3 * 4;  // down to 2 x 2
constexpr u32 kSmallWaves = kSmallThreads / kWave;
static_assert(kSmallWaves * kSmallPer == kWave, "one lane for each wave's sum of a round");
__global__ __launch_bounds__(kSmallThreads) void k_small_topdown(SmallArgs a, const float* __restrict__ depth, u32 N, u32 T,
                                                                 u64 root, LeafColumns cols, int pyr_level) {
    __shared__ u32 s_wave[2][kWave];  // (alternating: a slower wave may still read the last level's)
    __shared__ u64 s_coord[2][kSmallMax];
    __shared__ unsigned short s_mask[kSmallMax];
    __shared__ float4 s_pyr[kPyrTexels / 2];
    __shared__ SmallLevels lv;
    load_levels(a, lv);
    const u32 lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
    const u32 wp = N >> pyr_level;  // at most kPyrWidth
    {
        const float4* src = reinterpret_cast<const float4*>(a.lv[pyr_level]);
        const u32 m = (wp * wp - 1) / 3 * 2;
        for (u32 i = threadIdx.x; i < m; i += kSmallThreads) s_pyr[i] = src[i];
    }
    if (threadIdx.x == 0) s_coord[a.R & 1][0] = root;  // create(): root offset (0, 0, 2*zTileIndex)
    for (u32 i = threadIdx.x; i < kMetaWords; i += kSmallThreads) a.meta[i] = 0u;  // the first launch to use them
    __syncthreads();
    for (int L = a.R; L >= a.Ls; --L) {
        const u32 c = uniform(lv.count[L]);  // at most kSmallMax
        const u32 rounds = (c + kSmallThreads - 1) / kSmallThreads;
        const u64* cell = s_coord[L & 1];
        u32* sums = s_wave[L & 1];
        const u32 w = N >> L;
        const float h = (float)(w * T);
        const float4* pyr = s_pyr + (wp * wp - w * w) / 3 * 2;
        u32* const mask = uniform(lv.mask[L]);
#pragma unroll 1
        for (u32 e = 0; e < rounds; ++e) {
            const u32 i = e * kSmallThreads + threadIdx.x;
            u32 k = 0;
            if (i < c) {
                const u64 cc = cell[i];
                u32 m;
                if (L >= pyr_level) {
                    const u32 x = min(unpack_x(cc), w - 2) >> 1, y = min(unpack_y(cc), w - 2);
                    m = classify_texels(unpack_z(cc), h, pyr[y * (w / 2) + x], pyr[(y + 1) * (w / 2) + x]);
                } else {
                    m = classify_node(cc, uniform(lv.lv[L]), depth, N, L, T);
                }
                mask[i] = m;
                s_mask[i] = (unsigned short)m;
                k = num_children(m);
            }
            const u32 inc = wave_inclusive_scan(k, OpSum{});
            if (lane == kWave - 1) sums[e * kSmallWaves + wid] = inc;
        }
        if (threadIdx.x >= rounds * kSmallWaves && threadIdx.x < kWave) sums[threadIdx.x] = 0u;
        __syncthreads();
        const u32 sum = sums[lane], upto = wave_inclusive_scan(sum, OpSum{});
        // Children on a small level (count at most kSmallMax) go to the other LDS buffer.
        u64* child = (L - 1 >= a.Ls) ? s_coord[(L - 1) & 1] : uniform(lv.coord[L - 1]);
        EmitChildrenOut emit{mask, nullptr, uniform(lv.cstart[L]), child, uniform(lv.count[L - 1]), (L == 3) ? cols : LeafColumns{}};
#pragma unroll 1
        for (u32 e = 0; e < rounds; ++e) {
            const u32 i = e * kSmallThreads + threadIdx.x;
            const u32 m = (i < c) ? s_mask[i] : 0u, k = num_children(m);
            const u32 first = wave_inclusive_scan(k, OpSum{}) - k + __shfl(upto - sum, (int)(e * kSmallWaves + wid), kWave);
            if (i < c) emit(i, first, k, EmitChildrenOut::Pre{m, cell[i]});
        }
        if (threadIdx.x == kWave - 1) a.meta[kMetaC + L] = upto;
        __syncthreads();  // the child level's coordinates are read next
    }
}

// The LDS table of the small levels: one 64-bit word per slot, as in the global table.
__device__ inline u32 lds_insert(u64* tab, u32 S, u64 h, u32 i) {
    const u32 tag = (u32)(h >> 32);
    const u64 mine = ((u64)tag << 32) | i;
    u32 slot = (u32)(h ^ (h >> 31)) & (S - 1);
    for (;;) {
        // Read first: lanes with equal keys take an atomic on one address in turn.
        u64 cur = *const_cast<volatile u64*>(tab + slot);
        if (cur == kEmptySlot) {
            cur = atomicCAS(reinterpret_cast<unsigned long long*>(tab + slot), (unsigned long long)kEmptySlot,
                            (unsigned long long)mine);
            if (cur == kEmptySlot) return slot;
        }
        if ((u32)(cur >> 32) == tag) {
            if ((u32)cur > i) atomicMin(reinterpret_cast<unsigned long long*>(tab + slot), (unsigned long long)mine);
            return slot;
        }
        slot = (slot + 1) & (S - 1);
    }
}

// Inserts of the small levels Ls .. R-1 (the root is never merged), each into a table in LDS that is
// then copied to the level's own.  The identities are also kept in LDS (two buffers: a level and its
// children), where the next level's keys read them, and a level's masks and child starts are loaded
// while the level below is inserted.
__global__ __launch_bounds__(kSmallThreads) void k_small_insert(SmallArgs a, u32 hbits) {
    __shared__ u64 tab[kSmallSlots];
    __shared__ u32 s_id[2][kSmallMax];
    __shared__ SmallLevels lv;
    load_levels(a, lv);
    __syncthreads();
    u32 pm[kSmallPer], pc[kSmallPer];  // masks and child starts of the level's nodes
    auto load = [&](int L) {
        const u32 c = uniform(lv.count[L]);
        const u32 *mask = uniform(lv.mask[L]), *cstart = uniform(lv.cstart[L]);
#pragma unroll
        for (u32 e = 0; e < kSmallPer; ++e) {
            const u32 i = e * kSmallThreads + threadIdx.x;
            pm[e] = (i < c) ? mask[i] : 0u;
            pc[e] = (i < c) ? cstart[i] : 0u;
        }
    };
    if (a.Ls < a.R) load(a.Ls);
    for (int L = a.Ls; L < a.R; ++L) {
        const u32 c = uniform(lv.count[L]), S = uniform(lv.slots[L]);
        u32* const id = uniform(lv.id[L]);
        u64* const out = uniform(lv.tab[L]);
        for (u32 j = threadIdx.x; j < S; j += kSmallThreads) tab[j] = kEmptySlot;
        u64 h[kSmallPer];
#pragma unroll
        for (u32 e = 0; e < kSmallPer; ++e) {
            const u32 i = e * kSmallThreads + threadIdx.x;
            h[e] = 0;
            if (i >= c) continue;
            const u32 k = (L > a.deepest) ? num_children(pm[e]) : 0u;
            u32 r[8] = {};
            if (k) {
                // The first small level's children are in memory.
                if (L == a.Ls) {
                    load_child_ids(ChildIds{uniform(lv.id[L - 1]), a.heads, a.n_below}, pc[e], k, r);
                } else {
#pragma unroll
                    for (u32 j = 0; j < 8; ++j) r[j] = (j < k) ? s_id[(L - 1) & 1][min(pc[e] + j, kSmallMax - 1)] : 0u;
                }
            }
            h[e] = weaken_hash(inner_key_hash(pm[e], r), hbits);
        }
        if (L + 1 < a.R) load(L + 1);
        __syncthreads();  // the table is clear
#pragma unroll
        for (u32 e = 0; e < kSmallPer; ++e) {
            const u32 i = e * kSmallThreads + threadIdx.x;
            if (i >= c) continue;
            const u32 slot = lds_insert(tab, S, h[e], i);
            s_id[L & 1][i] = slot;
            id[i] = slot;
        }
        __syncthreads();  // every insert is in; the next level reads these identities
        for (u32 j = threadIdx.x; j < S; j += kSmallThreads) out[j] = tab[j];
        // (each thread clears for the next level the slots that it has just copied)
    }
}

// The DAG's word buffer: from the admission's allocator when it has one (a server keeps its budget
// there), else from the context's buffer cache.
void* alloc_words(cpvs_ctx* ctx, const Admit* admit, u64 words) {
    const size_t bytes = sizeof(u32) * words;
    return (admit && admit->alloc) ? admit->alloc(admit->user, bytes) : ctx->buffers.take(bytes);
}

inline dim3 grid1d(u32 n, u32 block = 256) { return dim3(ceil_div<u32>(n ? n : 1, block)); }

// The small levels [Ls, R] of a build with these node counts (R + 1: none).
int small_levels(const u64* cnt, int deepest, int R, bool use_table, bool leaf) {
    int Ls = R + 1;
    if (use_table && leaf)
        for (int L = R; L >= std::max(deepest, 3) && cnt[L] <= kSmallMax; --L) Ls = L;
    return Ls;
}
int deepest_level(const u64* cnt, int bottom, int R) {
    int d = R;  // lowest level with nodes (the counts are exact)
    while (d > bottom && cnt[d - 1] > 0) --d;
    return d;
}
// Slots of level L's table (0: the root and absent levels have none).  With the sort merge one entry
// per node.
u32 level_slots(const u64* cnt, int L, int R, int Ls, bool use_table, bool leaf, bool small_tables) {
    if (L >= R || !cnt[L]) return 0;
    if (!use_table) return (u32)std::min<u64>(cnt[L], 0xFFFFFFFFull);
    if (L >= Ls) return small_slots((u32)cnt[L]);
    return (leaf && L == 2) ? leaf_table_slots(cnt[L], small_tables) : inner_table_slots(cnt[L], small_tables);
}
u64 bound_words_of(const u64* cnt, int bottom, int R, bool leaf) {
    u64 w = 0;
    for (int L = bottom; L <= R; ++L) w += cnt[L] + ((L > bottom) ? cnt[L - 1] : 0) + ((leaf && L == 2) ? 16 * cnt[L] : 0);
    return w;
}

// The nodes' cells are read for the last time by the level scans, a sort's arrays by its last level, and
// the tables are emptied or written after that: one region holds all three.  Each with its own place, a
// sort without leafmasks needed 20% more than the fixed scratch of cpvs_build_noalloc was sized by.
size_t sort_bytes(size_t cmax) { return 5 * arena_bytes(cmax, 4) + arena_bytes(sort_scratch_words(cmax), 4); }
size_t shared_bytes(size_t cell_bytes, size_t tab_slots, size_t cmax, bool use_table) {
    return std::max({cell_bytes, arena_bytes(tab_slots, 8), use_table ? 0 : sort_bytes(cmax)});
}

constexpr int kRetryWithSort = -1000;
constexpr int kRetryFullTable = -1001;
constexpr int kRetryExactCounts = -1002;  // the counts exceed the emitted nodes (a map with NaN depths)


// *dst = v, plus 1 when *src (may be null) is not 0.
__global__ void k_store_word(u32* dst, u32 v, const u32* src) { *dst = v + ((src && *src) ? 1u : 0u); }

constexpr u32 kHostReady = kMetaWords, kHostDone = kMetaWords + 1;  // flags behind the meta readback
static_assert(sizeof(u32) * (kMetaWords + 2) <= sizeof(u64) * kPinnedWords, "the readback fits the pinned staging");

// Waits until none of n words of pinned memory, which queued kernels of stream s store to, reads
// `unset` any more.  Reading them is about 6 us quicker than a stream synchronisation (6 against 12 us
// for an empty kernel), which takes over after kPollUs: longer waits should not keep a core busy, and
// a kernel that fails never stores.
constexpr double kPollUs = 500.0;
int wait_words(const volatile u32* w, size_t n, u32 unset, hipStream_t s) {
    size_t k = 0;
    const auto t0 = std::chrono::steady_clock::now();
    for (u32 spins = 1;; ++spins) {
        while (k < n && w[k] != unset) ++k;
        if (k == n) {
            std::atomic_thread_fence(std::memory_order_acquire);
            return CPVS_OK;
        }
        __builtin_ia32_pause();
        if ((spins & 63u) == 0 &&
            std::chrono::duration<double, std::micro>(std::chrono::steady_clock::now() - t0).count() > kPollUs)
            break;
    }
    CPVS_HIP_CHECK(hipStreamSynchronize(s));
    for (; k < n; ++k)
        if (w[k] == unset) {
            set_error("build: a readback word was not stored");
            return CPVS_EINTERNAL;
        }
    return CPVS_OK;
}

}  // namespace

// As wait_stream; *set (may be null) = whether the device word *src was not 0 then.
static int wait_stream_word(u64* pinned, const u32* src, bool* set, hipStream_t s) {
    u32* done = reinterpret_cast<u32*>(pinned) + kHostDone;
    *static_cast<volatile u32*>(done) = 0;
    CPVS_LAUNCH("done", k_store_word, dim3(1), dim3(1), 0, s, done, 1u, src);
    CPVS_HIP_CHECK(hipGetLastError());
    const int rc = wait_words(done, 1, 0u, s);
    if (set) *set = *static_cast<volatile u32*>(done) > 1;
    return rc;
}
int wait_stream(u64* pinned, hipStream_t s) { return wait_stream_word(pinned, nullptr, nullptr, s); }

namespace {

int store_and_wait(u32* dst, u32 v, u64* pinned, hipStream_t s) {
    CPVS_LAUNCH("store_word", k_store_word, dim3(1), dim3(1), 0, s, dst, v, nullptr);
    return wait_stream(pinned, s);
}

int build_once(cpvs_ctx* ctx, Arena& A, u64* pinned, const cpvs_pyramid* p, u32 t, u32 T, hipStream_t s, int merge_mode,
               cpvs_dag** out, const Admit* admit, bool small_tables, bool exact, DagOut* into) {
    const int n = p->n;
    const int R = n - 2;
    const bool leaf = n >= 5 && ctx->leafmasks != 0;  // useLeafmasks (src/CompressedShadow.cpp:20-27)
    const int bottom = leaf ? 2 : 0;
    const u32 N = p->N;
    const bool use_table = merge_mode == CPVS_MERGE_TABLE;

    // --- exact node counts (one readback) ---------------------------------------------
    const u32 w3 = leaf ? (N >> 3) : 0;
    const u32 ncol = w3 * w3;
    const size_t meta_bytes = arena_bytes(kMetaWords, sizeof(u32));
    const size_t col_bytes = leaf ? arena_bytes(ncol, sizeof(uint4)) : 0;
    int rc = A.reserve(meta_bytes + col_bytes, s);
    if (rc) return rc;
    uint4* colinfo = leaf ? A.take<uint4>(ncol) : nullptr;
    CountLayout lay;
    rc = pyramid_node_counts(p, t, T, leaf, pinned_partials(pinned), colinfo, s, &lay, exact);
    if (rc) return rc;
    rc = wait_words(pinned_partials(pinned), lay.block_start[lay.nlev] + 1, kUnsetCount, s);
    if (rc) return rc;
    u64 cnt[kMaxLevels] = {};
    sum_node_counts(lay, pinned_partials(pinned), cnt);
    cnt[R] = 1;
    if (cnt[R - 1] == 0) {
        // No partial child of the root (a z-tile above or below every surface, a flat map): the
        // DAG is the root's childmask alone, written without any further kernel.
        const u32 word = pinned_partials(pinned)[lay.block_start[lay.nlev]];
        if (into && into->cap < 1) {
            set_error("build: the DAG has 1 word, the output holds %llu", (unsigned long long)into->cap);
            return CPVS_EINVAL;
        }
        if (admit) {
            rc = admit->fn(admit->user, A, 0, sizeof(u32));
            if (rc) return rc;
        }
        u32* d_words = into ? into->words : static_cast<u32*>(alloc_words(ctx, admit, 1));
        if (!d_words) {
            set_error("build: hipMalloc of one DAG word failed");
            return CPVS_ENOMEM;
        }
        rc = store_and_wait(d_words, word, pinned, s);
        if (rc) {
            if (!into) ctx->buffers.give(d_words);
            return rc;
        }
        if (into) {
            into->nwords = 1;
            into->root_mask = word;
            return CPVS_OK;
        }
        cpvs_dag* d = new cpvs_dag();
        d->ctx = ctx;
        d->n = n;
        d->words = 1;
        d->d_words = d_words;
        d->root_mask = word;
        d->N = N;
        d->zTileIndex = t;
        d->zTileNum = T;
        d->merge_mode = merge_mode;
        d->leafmasks = leaf;
        d->nodes[R] = 1;
        d->uniques[R] = 1;
        *out = d;
        return CPVS_OK;
    }
    for (int L = bottom; L <= R; ++L) {
        if (cnt[L] > 0xFFFFFFF0ull) {
            set_error("build: level %d has %llu nodes (limit 2^32)", L, (unsigned long long)cnt[L]);
            return CPVS_EINVAL;
        }
    }

    // --- scratch sizing ----------------------------------------------------------------------
    u32 cmax = 1;
    for (int L = bottom; L < R; ++L) cmax = cnt[L] > cmax ? (u32)cnt[L] : cmax;
    const u32 scan_n = (leaf && ncol > cmax) ? ncol : cmax;
    const size_t c2 = leaf ? (cnt[2] ? cnt[2] : 1) : 1;
    const bool col_list = leaf && T > 1;  // compact the z-tile's columns with leaf nodes
    const int deepest = deepest_level(cnt, bottom, R);
    const int Ls = small_levels(cnt, deepest, R, use_table, leaf);
    const size_t need = build_scratch_bytes(cnt, R, leaf, ncol, col_list, use_table, small_tables);
    if (admit) {
        rc = admit->fn(admit->user, A, need, 4 * bound_words_of(cnt, bottom, R, leaf));
        if (rc) return rc;
    }
    bool moved = false;
    rc = A.reserve(need, s, &moved);  // keeps the contents when large enough
    if (rc) return rc;
    colinfo = leaf ? A.take<uint4>(ncol) : nullptr;
    u32* meta = A.take<u32>(kMetaWords);
    if (leaf && moved) {  // the arena was reallocated: count the columns again
        rc = pyramid_node_counts(p, t, T, leaf, nullptr, colinfo, s, nullptr, exact);
        if (rc) return rc;
    }
    // meta is zeroed by the first kernel below (k_small_topdown or k_start).

    Level lv[kMaxLevels];
    u32 ntiles = 0;
    size_t tab_slots = 0, clear_slots = 0;  // of all levels; of those whose tables a launch must clear
    size_t cell_bytes = 0;
    for (int L = bottom; L <= R; ++L) {
        lv[L].slots = level_slots(cnt, L, R, Ls, use_table, leaf, small_tables);
        tab_slots += lv[L].slots;
        if (L < Ls) clear_slots += lv[L].slots;
        if (!(leaf && L == 2)) cell_bytes += arena_bytes(cnt[L] ? cnt[L] : 1, sizeof(u64));
    }
    const size_t shared_cap = shared_bytes(cell_bytes, tab_slots, cmax, use_table);
    char* const shared = A.take<char>(shared_cap);
    Arena cells, sorting;
    cells.base = sorting.base = shared;
    cells.cap = sorting.cap = shared_cap;
    u64* const tab = reinterpret_cast<u64*>(shared);
    for (int L = bottom; L <= R; ++L) {
        const size_t c = cnt[L] ? cnt[L] : 1;
        const bool is_leaf = leaf && L == 2;
        lv[L].count = (u32)cnt[L];
        lv[L].coord = is_leaf ? nullptr : cells.take<u64>(c);
        lv[L].mask = A.take<u32>(c);
        lv[L].cstart = is_leaf ? nullptr : A.take<u32>(c);
        lv[L].id = A.take<u32>(c);
        lv[L].uniq = A.take<u32>(c);
        lv[L].off = A.take<u32>(c);
        lv[L].flag = reinterpret_cast<uint8_t*>(A.take<u64>(flag_words(c)));
        ntiles += ceil_div<u32>((u32)cnt[L], kTileNodes);
    }
    {
        u64* t0 = tab;  // deepest level first: the tables to clear are one run
        for (int L = bottom; L <= R; ++L) {
            lv[L].tab = t0;
            t0 += lv[L].slots;
        }
    }
    u32* tile_sums = A.take<u32>(ntiles);
    ulonglong2* tile_pre = A.take<ulonglong2>(tile_pre_count(ntiles));
    u64* leafm = leaf ? A.take<u64>(c2 * 8) : nullptr;
    // The run heads' key hashes, from the leaf kernel to the leaf insert, in the place of the leaf
    // level's unique list and offsets (two arrays side by side), which k_offsets writes later.
    const bool lane_leaf = leaf && (col_list ? std::min<u64>(ncol, cnt[2]) : ncol) >= kLaneLeafMin;
    u64* leaf_hash = lane_leaf ? reinterpret_cast<u64*>(lv[2].uniq) : nullptr;
    u32* runhead = leaf ? A.take<u32>(c2) : nullptr;
    u32* colbfs = leaf ? A.take<u32>(c2) : nullptr;
    u32* clist = col_list ? A.take<u32>(ncol) : nullptr;
    u32* nclist = col_list ? A.take<u32>(1) : nullptr;
    SortScratch srt{};
    if (!use_table) {
        srt.skey = sorting.take<u32>(cmax);
        srt.sval = sorting.take<u32>(cmax);
        srt.ktmp = sorting.take<u32>(cmax);
        srt.vtmp = sorting.take<u32>(cmax);
        srt.seg = sorting.take<u32>(cmax);
        srt.sort_scratch = sorting.take<u32>(sort_scratch_words(cmax));
    }
    u32* scan_scratch = A.take<u32>(scan_scratch_words(scan_n));
    srt.scan_scratch = scan_scratch;
    if (A.used > A.cap || cells.used > shared_cap || sorting.used > shared_cap) {
        set_error("build: scratch layout exceeds its reservation (%zu > %zu)", A.used, A.cap);
        return CPVS_EINTERNAL;
    }

    LeafColumns lc{};
    if (leaf) {
        lc.info = colinfo;
        lc.bfs = colbfs;
        lc.w3 = w3;
        if (col_list)
            device_scan(ColPairIn{colinfo}, ColListOut{colinfo, clist, nclist, ncol}, ncol, OpSum64{}, nullptr, scan_scratch, s);
        else
            device_scan(ColCountIn{colinfo}, ColStartOut{colinfo}, ncol, OpSum{}, nullptr, scan_scratch, s);
    }

    // --- 1/2. BFS classification -------------------------------------------------------------
    const u64 root = pack_xyz(0, 0, 2 * t);  // create(): root offset (0,0,2*zTileIndex)
    // Small levels [Ls, R] go through the one-workgroup kernels (with the hash-table merge).
    SmallArgs sa{};
    sa.R = R;
    sa.Ls = Ls;
    sa.deepest = deepest;
    sa.meta = meta;
    sa.n_below = (Ls - 1 >= bottom && Ls - 1 < R) ? std::max<u32>(lv[Ls - 1].count, 1u) : 1u;
    sa.heads = (leaf && Ls == 3) ? runhead : nullptr;
    for (int L = bottom; L <= R; ++L) {
        sa.count[L] = lv[L].count;
        sa.coord[L] = lv[L].coord;
        sa.mask[L] = lv[L].mask;
        sa.cstart[L] = lv[L].cstart;
        sa.id[L] = lv[L].id;
        sa.tab[L] = lv[L].tab;
        sa.slots[L] = lv[L].slots;
        sa.lv[L] = p->lv[L];
    }
    const int top_big = std::min(R, Ls - 1);  // highest level of the per-level path
    if (Ls <= R)
    {
        int pyr_level = 3;  // the first level that the kernel keeps in LDS (levels lie in one run from 3 on)
        while ((N >> pyr_level) > kPyrWidth) ++pyr_level;
        CPVS_LAUNCH("small_topdown", k_small_topdown, dim3(1), dim3(kSmallThreads), 0, s, sa, p->depth, N, T, root, lc,
                    pyr_level);
    }
    else
        CPVS_LAUNCH("start", k_start, dim3(1), dim3(1), 0, s, lv[R].coord, root, meta, (u32)kMetaWords);
    for (int L = top_big; L >= deepest; --L) {
        const u32 c = lv[L].count;
        if (leaf && L == 2) {
            // With a column list, at most min(columns, leaf nodes) columns have nodes.
            const u32 bound = col_list ? std::min(ncol, c) : ncol;
            const u64 slots = use_table ? clear_slots : 0u;  // the merge's tables are cleared here
            // (the list of slow columns lies where the identities are written later)
            const LeafOut lo{colbfs, lv[2].mask, leafm, runhead, leaf_hash, lv[2].id, meta + kMetaSlow, c};
            if (lane_leaf) {
                const u32 units = ceil_div<u32>(bound, kLaneThreads), chunk = ceil_div<u32>(units, kXcds);
                if (col_list)
                    CPVS_LAUNCH("leaf_lanes", k_leaf_lanes<true>, dim3(units), dim3(kLaneThreads), 0, s, lc, bound, p->depth,
                                N, T, lo, chunk, tab, slots, clist, nclist);
                else
                    CPVS_LAUNCH("leaf_lanes", k_leaf_lanes<false>, dim3(chunk * kXcds), dim3(kLaneThreads), 0, s, lc, bound,
                                p->depth, N, T, lo, chunk, tab, slots, nullptr, nullptr);
                const u32 most = std::min(bound, c);
                CPVS_LAUNCH("leaf_waves", k_leaf_waves<true>, dim3(list_waves(most)), dim3(64), 0, s, lc, most,
                            p->depth, N, T, p->lv[3], lo, 0u, tab, 0u, lv[2].id, meta + kMetaSlow);
            } else if (col_list) {
                CPVS_LAUNCH("leaf_waves", k_leaf_waves<true>, dim3(list_waves(bound)), dim3(64), 0, s, lc, bound,
                            p->depth, N, T, p->lv[3], lo, 0u, tab, slots, clist, nclist);
            } else {
                const u32 chunk = ceil_div<u32>(bound, kXcds);
                CPVS_LAUNCH("leaf_waves", k_leaf_waves<false>, dim3(chunk * kXcds), dim3(64), 0, s, lc, bound, p->depth, N, T,
                            p->lv[3], lo, chunk, tab, slots, nullptr, nullptr);
            }
            break;
        }
        // A level is classified inside its emit scan when that scan loads its outputs' prefetch
        // before the block scan.  Above 1 M nodes the output stage loads after the scan, where
        // classifying (two dependent loads) costs more than the classify launch it saves.
        if (L > bottom && scan_prefetches(c)) {
            const Classify cls{lv[L].coord, p->lv[L], p->depth, N, L, T};
            EmitChildrenOut emit{lv[L].mask, lv[L].coord, lv[L].cstart, lv[L - 1].coord, lv[L - 1].count, LeafColumns{},
                                 lv[L].mask, cls};
            if (leaf && L == 3) emit.cols = lc;
            device_scan(ClassifyCountIn{cls}, emit, c, OpSum{}, meta + kMetaC + L, scan_scratch, s);
        } else {
            CPVS_LAUNCH("classify", k_classify, grid1d(c), dim3(256), 0, s, lv[L].coord, c, p->lv[L], p->depth, N, L, T,
                        lv[L].mask);
            if (L > bottom) {
                EmitChildrenOut emit{lv[L].mask, lv[L].coord, lv[L].cstart, lv[L - 1].coord, lv[L - 1].count, LeafColumns{}};
                if (leaf && L == 3) emit.cols = lc;
                device_scan(ChildCountIn{lv[L].mask}, emit, c, OpSum{}, meta + kMetaC + L, scan_scratch, s);
            }
        }
    }
    CPVS_HIP_CHECK(hipGetLastError());

    // --- 3. merge, bottom-up (the root is never merged) --------------------------------------
    MArgs ma{};
    ma.leafm = leafm;
    ma.heads = runhead;
    ma.sorted = !use_table;
    u32 tile = 0;
    for (int L = deepest; L <= R; ++L) {
        const Level& v = lv[L];
        ma.tile0[ma.nlev] = tile;
        tile += ceil_div<u32>(v.count, kTileNodes);
        ma.lv[ma.nlev++] = MLevel{v.mask, v.cstart, v.id, v.tab, v.flag, v.uniq, v.off, v.count, v.slots, L,
                                  (leaf && L == 2) ? 1u : 0u, L == R ? 1u : 0u,
                                  (use_table && L < R && (L >= Ls || v.count <= kLateMax)) ? 1u : 0u};
    }
    ma.tile0[ma.nlev] = tile;
    // Without a leaf level its kernel did not clear the tables.
    if (use_table && clear_slots && !(leaf && deepest == 2)) table_clear(tab, clear_slots, s);
    for (int L = deepest; L < std::min(R, Ls); ++L) {
        if (use_table)
            merge_insert(ma, L - deepest, leaf_hash, meta,
                         (leaf && L == 2) ? ctx->leaf_hash_bits.load() : ctx->inner_hash_bits.load(), s);
        else
            merge_sort_level(ma, L - deepest, srt, meta, s);
    }
    if (Ls < R) CPVS_LAUNCH("small_insert", k_small_insert, dim3(1), dim3(kSmallThreads), 0, s, sa,
                             ctx->inner_hash_bits.load());
    // --- 4. first occurrences, offsets, bases, one readback, words -------------------------
    // The host reads the totals that k_totals stores in pinned memory while k_offsets runs, so the
    // words go straight to a buffer of their exact size and the GPU does not wait for the host.
    volatile u32* host_meta = reinterpret_cast<volatile u32*>(pinned);
    host_meta[kHostReady] = 0;
    merge_finish(ma, tile_sums, tile_pre, meta, R, reinterpret_cast<u32*>(pinned), s);
    CPVS_HIP_CHECK(hipGetLastError());
    rc = wait_words(host_meta + kHostReady, 1, 0u, s);
    if (rc) return rc;
    u32 hm[kMetaWords];
    std::memcpy(hm, pinned, sizeof(hm));

    // Counts first: a level whose count exceeds its emitted children merged unwritten nodes too.
    for (int L = deepest + 1; L <= R; ++L) {
        if (hm[kMetaC + L] != lv[L - 1].count) {
            if (!exact) return kRetryExactCounts;  // cells under a NaN texel were counted: count exactly
            set_error("build: level %d emitted %u children, expected %u", L, hm[kMetaC + L], lv[L - 1].count);
            return CPVS_EINTERNAL;
        }
    }
    if (use_table && hm[kMetaFull] != 0) return small_tables ? kRetryFullTable : kRetryWithSort;
    if (use_table && hm[kMetaColl] != 0) return kRetryWithSort;
    if (deepest > bottom && hm[kMetaC + deepest] != 0) {
        set_error("build: level %d emitted children below the deepest level", deepest);
        return CPVS_EINTERNAL;
    }
    u64 total = 0;
    for (int L = deepest; L <= R; ++L) total += hm[kMetaS + L];
    if (total >= 0xFFFFFFFEull) {
        set_error("build: DAG of %llu words exceeds 32-bit offsets", (unsigned long long)total);
        return CPVS_EINVAL;
    }

    if (into && total > into->cap) {
        set_error("build: the DAG has %llu words, the output holds %llu", (unsigned long long)total,
                  (unsigned long long)into->cap);
        return CPVS_EINVAL;
    }
    u32* d_words = into ? into->words : static_cast<u32*>(alloc_words(ctx, admit, total ? total : 1));
    if (!d_words) {
        set_error("build: hipMalloc of %llu DAG words failed", (unsigned long long)total);
        return CPVS_ENOMEM;
    }
    merge_write(ma, meta, d_words, total, s);
    bool collided = false;  // the late levels' compares run beside the write
    rc = wait_stream_word(pinned, use_table ? meta + kMetaColl : nullptr, &collided, s);
    if (rc == CPVS_OK && collided) rc = kRetryWithSort;
    if (rc) {
        if (!into) ctx->buffers.give(d_words);
        return rc;
    }
    if (into) {
        into->nwords = total;
        into->root_mask = hm[kMetaRoot];
        return CPVS_OK;
    }

    cpvs_dag* d = new cpvs_dag();
    d->ctx = ctx;
    d->n = n;
    d->words = total;
    d->d_words = d_words;
    d->root_mask = hm[kMetaRoot];
    d->N = N;
    d->zTileIndex = t;
    d->zTileNum = T;
    d->merge_mode = merge_mode;
    d->key_collisions = hm[kMetaSortColl];
    d->leafmasks = leaf;
    for (int L = 0; L < n && L < kMaxLevels; ++L) {
        d->nodes[L] = (L >= bottom && L <= R) ? cnt[L] : 0;
        d->uniques[L] = (L >= deepest && L <= R) ? hm[kMetaU + L] : 0;
    }
    *out = d;
    return CPVS_OK;
}

}  // namespace

// What build_once lays out: cnt the nodes per level (bottom .. R), ncol the leaf columns.
size_t build_scratch_bytes(const u64* cnt, int R, bool leaf, u32 ncol, bool col_list, bool use_table, bool small_tables) {
    const int bottom = leaf ? 2 : 0;
    const int Ls = small_levels(cnt, deepest_level(cnt, bottom, R), R, use_table, leaf);
    size_t need = arena_bytes(kMetaWords, sizeof(u32)) + (leaf ? arena_bytes(ncol, sizeof(uint4)) : 0);
    // (64 bits throughout: estimates are asked for maps that no build takes)
    size_t cmax = 1, ntiles = 0, slots = 0, cells = 0;
    for (int L = bottom; L <= R; ++L) {
        const size_t c = cnt[L] ? cnt[L] : 1;
        if (L < R) cmax = std::max<size_t>(cmax, cnt[L]);
        const bool is_leaf = leaf && L == 2;
        cells += is_leaf ? 0 : arena_bytes(c, 8);
        need += (is_leaf ? 0 : arena_bytes(c, 4)) + 4 * arena_bytes(c, 4) +
                arena_bytes(flag_words(c), 8);
        slots += level_slots(cnt, L, R, Ls, use_table, leaf, small_tables);
        ntiles += ceil_div<size_t>(cnt[L], kTileNodes);
    }
    need += shared_bytes(cells, slots, cmax, use_table) + arena_bytes(ntiles, 4) + arena_bytes(tile_pre_count(ntiles), 16);
    const size_t c2 = leaf ? (cnt[2] ? cnt[2] : 1) : 1;
    if (leaf) need += arena_bytes(c2 * 8, 8) + 2 * arena_bytes(c2, 4);  // leafmask rows, run heads, column map
    if (col_list) need += arena_bytes(ncol, 4) + arena_bytes(1, 4);
    need += arena_bytes(scan_scratch_words(leaf ? std::max<size_t>(ncol, cmax) : cmax), 4);
    return need + (1 << 20);
}

// A build that finds its merge table too small runs again with a full-size table, one with a key
// collision again with the sort merge, and one whose counts exceed the emitted nodes again with
// exact counts; each switch is made at most once.
int build_dag(cpvs_ctx* ctx, Arena& A, u64* pinned, int merge_mode, const cpvs_pyramid* p, u32 t, u32 T, hipStream_t s,
              cpvs_dag** out, const Admit* admit, DagOut* into) {
    bool small_tables = true, exact = false;
    int rc = CPVS_OK;
    for (int attempt = 0; attempt < 4; ++attempt) {
        rc = build_once(ctx, A, pinned, p, t, T, s, merge_mode, out, admit, small_tables, exact, into);
        if (rc == kRetryFullTable && small_tables) small_tables = false;
        else if (rc == kRetryWithSort && merge_mode != CPVS_MERGE_SORT) merge_mode = CPVS_MERGE_SORT, small_tables = false;
        else if (rc == kRetryExactCounts && !exact) exact = true;
        else break;
    }
    // The host acts on readbacks that kernels store before the last launches end, so a build that fails
    // here may still be writing its scratch and reading its map.  The scratch is the context's (or, for
    // cpvs_build_noalloc, the device's) and the next call may come on another stream.
    if (rc != CPVS_OK) (void)hipStreamSynchronize(s);
    if (rc == kRetryFullTable || rc == kRetryWithSort || rc == kRetryExactCounts) {
        set_error("build: no consistent build after every fallback (status %d)", rc);
        return CPVS_EINTERNAL;
    }
    return rc;
}

}  // namespace cpvs
