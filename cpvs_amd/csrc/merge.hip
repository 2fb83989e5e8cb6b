// merge.hip -- equal subtrees merged level by level, and the DAG's words.
//
// Bottom-up, each level takes one launch: the key of every node -- its mask and the partial
// leafmasks, or its mask and its children's identities -- goes into the level's hash table, and the
// slot it ends in is the node's own identity for its parents' keys.  Slots never move, so equal keys
// have equal identities before anything is known of their order.  A node's key is compared in the
// same launch, in full, with that of a node that the slot already held.  What needs finished tables is
// left to launches over all levels at once:
//   k_firsts    per node the smallest index in its slot; a byte for each node, its words if it is that
//               one; the first occurrences and words of each tile of nodes;
//   k_totals    a scan of the tiles, the levels' totals and bases (k_offsets does it for few tiles);
//   k_offsets   rank and word offset of every first occurrence, in index order, which is the order
//               that mergeLevel's linear search gives (src/CompressedShadowUtil.h:154-182).
// Before, a launch over all nodes looked up each node's slot and compared its key with the first
// occurrence's: 77 us and 209 MB of scattered reads of 690 us at 8192^2, 16 of 144 us at 1024^2.  Keys
// are compared here while they are in registers: 8 z-tiles 2118 -> 1992 us, 32 maps 2182 -> 2086.
//
// Keys that a table cannot tell apart are found by the compares, and the build is done again with
// the sort merge, whose identities are first occurrences' indices.
#include "merge.hpp"

namespace cpvs {

// --- the table merge -------------------------------------------------------------------------

// One 64-bit word per slot: the key hash's high 32 bits (its tag) above the smallest node index
// with that hash, so a probe touches one cache line and a new key costs one atomic.  ~0 marks an
// empty slot (node indices stay below 2^32 - 1).  Two keys whose tags are equal and whose probe
// chains meet share a slot; the full-key compare of a later one then sends the build down the
// sorting path, as for equal 64-bit hashes.

__global__ __launch_bounds__(256) void k_table_clear(u64* __restrict__ tab, u64 slots) { clear_table(tab, slots); }

// The run heads of a window of kT nodes are listed in LDS; equal hashes meet in an LDS table,
// the distinct ones are spread over the threads for the global inserts, and every head's key is then
// compared with its window's first of that hash, that one's with the global slot's earlier node.  The
// compares take four lanes to a pair of leafmask rows (16 bytes a lane): one lane to a row would touch
// 64 lines with each load.  The rows are what the compares cost (at 8192^2, with four nodes a thread: 57 -> 98 us).
// What bounds it besides: the tables' atomics and coherent reads, performed at memory, about 7 G atomics/s.
// One node a thread: where heads lie dense, a thread with several walks their reads and atomics one
// after another (4 a thread 99 us, 16 a thread 148 us at 8192^2, one 77; 30, 18 at 2048^2).  Windows of
// 512 and 1024 meet fewer equal hashes than they lose to workgroups waiting: 32 maps 227, 248, 287 us.
__global__ __launch_bounds__(kLeafInsertThreads) void k_insert_leaf(const u32* __restrict__ mask, const u64* __restrict__ leafm,
                                                                    const u32* __restrict__ runhead,
                                                                    const u64* __restrict__ hash, u32 n,
                                                                    u64* __restrict__ tab, u32 S, u32* __restrict__ tslot,
                                                                    u32* __restrict__ meta, u32 hbits, u32 late) {
    constexpr u32 kT = kLeafInsertThreads, kSlots = 2 * kT;  // at most half full: every probe ends
    __shared__ u64 gh[kSlots];  // a hash, then its global slot << 32 | the node that the slot held before
    __shared__ u32 gi[kSlots];  // smallest node index of the slot's hash
    __shared__ unsigned short glist[kT];  // LDS slots in use
    __shared__ unsigned short heads[kT], hslot[kT];  // the window's run heads and their LDS slots
    __shared__ u32 gcount, nheads;
    const u32 t = threadIdx.x, lane = t & (kWave - 1), i0 = blockIdx.x * kT;
    if (t == 0) gcount = nheads = 0;
    const bool head = i0 + t < n && runhead[i0 + t] == i0 + t;
    for (u32 j = t; j < kSlots; j += kT) {
        gh[j] = 0ull;  // 0 marks an empty LDS slot
        gi[j] = kNoRep;
    }
    __syncthreads();
    {
        const u64 bits = __ballot(head);
        u32 at = 0;
        if (lane == 0 && bits) at = atomicAdd(&nheads, (u32)__popcll(bits));
        at = __builtin_amdgcn_readfirstlane(at);
        if (head) heads[at + (u32)__popcll(bits & ((1ull << lane) - 1ull))] = (unsigned short)t;
    }
    __syncthreads();
    const u32 nh = nheads;
    if (t < nh) {
        // The key hash of a run's first node (the run's smallest index): from the leaf kernel where a
        // lane walked its column, else from its mask and leafmasks (its row at its own index).
        const u32 i = i0 + heads[t];
        u64 h = hash ? hash[i] : 0ull;
        if (h == 0ull) h = leaf_key_hash(mask[i], leafm + (size_t)i * 8);
        h = weaken_hash(h, hbits);
        if (h == 0ull) h = 1ull;
        u32 sl = (u32)(h ^ (h >> 29)) & (kSlots - 1);
        for (;;) {
            const u64 cur = atomicCAS(reinterpret_cast<unsigned long long*>(gh + sl), 0ull, (unsigned long long)h);
            if (cur == 0ull) {
                glist[atomicAdd(&gcount, 1u)] = (unsigned short)sl;
                break;
            }
            if (cur == h) break;
            sl = (sl + 1) & (kSlots - 1);
        }
        atomicMin(gi + sl, i);
        hslot[t] = (unsigned short)sl;
    }
    __syncthreads();
    if (t < gcount) {
        const u32 sl = glist[t];
        u32 occ;
        const u32 slot = table_insert(tab, S, gh[sl], gi[sl], meta + kMetaFull, occ);
        gh[sl] = ((u64)slot << 32) | occ;
    }
    __syncthreads();
    bool eq = true;
    if (t < nh) tslot[i0 + heads[t]] = (u32)(gh[hslot[t]] >> 32);
    for (u32 j = t / 4; j < nh && !late; j += kT / 4) {
        const u32 i = i0 + heads[j], sl = hslot[j], rep = gi[sl];
        const u32 with = (rep != i) ? rep : (u32)gh[sl];
        if (with >= n) continue;
        const u32 q = t & 3, ma = mask[i], mb = mask[with];
        const u32 k = num_children(ma);
        eq = eq && ma == mb;
        if (2 * q < k) {
            const ulonglong2 x = *reinterpret_cast<const ulonglong2*>(leafm + (size_t)i * 8 + 2 * q);
            const ulonglong2 y = *reinterpret_cast<const ulonglong2*>(leafm + (size_t)with * 8 + 2 * q);
            eq = eq && x.x == y.x && (2 * q + 1 >= k || x.y == y.y);
        }
    }
    if (!eq) atomicAdd(meta + kMetaColl, 1u);  // two keys share a slot: the build is redone by sorting
}

// A table slot hit by many threads at once serialises their atomics, and equal keys are common
// (flat regions repeat the same subtrees all over a level; a level of a few hundred thousand nodes
// runs almost all at once, before any first occurrence has landed).  So each workgroup first merges
// its own equal hashes in an LDS table, with the keys beside it for the compares: only the smallest
// index of each distinct hash in the group touches the global table, and the others take its slot.
// The window: levels up to kInnerSmallMax nodes are one chain of reads and atomics for each workgroup,
// shorter in small ones (256 threads against 512: 7.6-10 us against 8.4-10.5); above, larger windows meet
// more equal keys (32 maps, 6.4 M nodes: 256 nodes 169 us, 512 165, two a thread 155).
template <u32 kPer, u32 kT>
__global__ __launch_bounds__(kT) void k_insert_inner(const u32* __restrict__ mask, const u32* __restrict__ cstart, ChildIds ch,
                                                     u32 n, u64* __restrict__ tab, u32 S, u32* __restrict__ id,
                                                     u32* __restrict__ meta, u32 hbits, u32 late) {
    constexpr u32 kSlots = 2 * kPer * kT;
    __shared__ u64 gh[kSlots];
    __shared__ u32 gi[kSlots];  // smallest node index of the slot's hash, then its global slot
    const u32 t = threadIdx.x, i0 = blockIdx.x * (kPer * kT) + t;
    u32 m[kPer], c[kPer], k[kPer], r[kPer][8], ls[kPer], rep[kPer], slot[kPer];
    u64 h[kPer];
#pragma unroll
    for (u32 e = 0; e < kPer; ++e) {
        const u32 i = i0 + e * kT;
        m[e] = (i < n) ? mask[i] : 0u;
        c[e] = (i < n) ? cstart[i] : 0u;
    }
    for (u32 j = t; j < kSlots; j += kT) {
        gh[j] = 0ull;
        gi[j] = kNoRep;
    }
#pragma unroll
    for (u32 e = 0; e < kPer; ++e) {
        k[e] = ch.id ? num_children(m[e]) : 0u;
#pragma unroll
        for (u32 j = 0; j < 8; ++j) r[e][j] = 0u;
        if (k[e]) load_child_ids(ch, c[e], k[e], r[e]);
    }
#pragma unroll
    for (u32 e = 0; e < kPer; ++e) {
        h[e] = weaken_hash(inner_key_hash(m[e], r[e]), hbits);
        if (h[e] == 0ull) h[e] = 1ull;  // 0 marks an empty LDS slot
    }
    __syncthreads();
#pragma unroll
    for (u32 e = 0; e < kPer; ++e) {
        ls[e] = 0;
        if (i0 + e * kT >= n) continue;
        u32 sl = (u32)(h[e] ^ (h[e] >> 29)) & (kSlots - 1);
        for (;;) {
            const u64 cur = atomicCAS(reinterpret_cast<unsigned long long*>(gh + sl), 0ull, (unsigned long long)h[e]);
            if (cur == 0ull || cur == h[e]) break;
            sl = (sl + 1) & (kSlots - 1);
        }
        atomicMin(gi + sl, i0 + e * kT);
        ls[e] = sl;
    }
    __syncthreads();
    // A node's key is compared with the group's smallest index of its hash, that one's with the table's.
    u32 with[kPer];
#pragma unroll
    for (u32 e = 0; e < kPer; ++e) {
        const u32 i = i0 + e * kT;
        rep[e] = (i < n) ? gi[ls[e]] : kNoRep;
        with[e] = (i < n) ? rep[e] : kNoRep;
        slot[e] = kNoRep;
        if (i < n && rep[e] == i) slot[e] = table_insert(tab, S, h[e], i, meta + kMetaFull, with[e]);
        if (late) with[e] = kNoRep;
    }
    __syncthreads();
#pragma unroll
    for (u32 e = 0; e < kPer; ++e)
        if (slot[e] != kNoRep) gi[ls[e]] = slot[e];
    u32 mo[kPer], co[kPer];
#pragma unroll
    for (u32 e = 0; e < kPer; ++e) {
        mo[e] = (with[e] < n) ? mask[with[e]] : m[e];
        co[e] = (with[e] < n) ? cstart[with[e]] : 0u;
    }
    bool eq = true;
#pragma unroll
    for (u32 e = 0; e < kPer; ++e) {
        eq = eq && mo[e] == m[e];
        if (with[e] < n && mo[e] == m[e] && k[e]) {
            u32 ro[8];
            load_child_ids(ch, co[e], k[e], ro);
#pragma unroll
            for (u32 j = 0; j < 8; ++j) eq = eq && ro[j] == r[e][j];
        }
    }
    if (!eq) atomicAdd(meta + kMetaColl, 1u);  // two keys share a slot: the build is redone by sorting
    __syncthreads();
#pragma unroll
    for (u32 e = 0; e < kPer; ++e)
        if (i0 + e * kT < n) id[i0 + e * kT] = gi[ls[e]];
}

// --- the sort merge --------------------------------------------------------------------------

__global__ __launch_bounds__(256) void k_sortkeys_leaf(const u32* __restrict__ mask, const u64* __restrict__ leafm,
                                                       const u32* __restrict__ runhead,
                                                       u32 n, u32* __restrict__ skey, u32* __restrict__ sval) {
    const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    u32 h = runhead[i];  // the key is the run's first node's
    h = (h < n) ? h : i;
    skey[i] = fold32(leaf_key_hash(mask[h], leafm + (size_t)h * 8));
    sval[i] = i;
}

__global__ __launch_bounds__(256) void k_sortkeys_inner(const u32* __restrict__ mask, const u32* __restrict__ cstart,
                                                        ChildIds ch, u32 n, u32* __restrict__ skey, u32* __restrict__ sval) {
    const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const u32 m = mask[i], s = cstart[i];
    const u32 k = ch.id ? num_children(m) : 0u;
    u32 r[8] = {};
    if (k) load_child_ids(ch, s, k, r);
    skey[i] = fold32(inner_key_hash(m, r));
    sval[i] = i;
}

// --- first occurrences -----------------------------------------------------------------------

__device__ inline int level_of_tile(const MArgs& a, u32 tile) {
    int k = 0;
    while (k + 1 < a.nlev && tile >= a.tile0[k + 1]) ++k;
    return k;
}

__device__ inline u32 node_words(u32 m, u32 leaf) { return 1u + (num_children(m) << leaf); }

__device__ inline u32 saturate32(u64 v) { return v > 0xFFFFFFFFull ? 0xFFFFFFFFu : (u32)v; }

// One workgroup: a scan over all tiles of all levels, four to a thread at a time.  tile_pre gets
// (first occurrences, words) before each tile, then, after the tiles, before each level and at the
// end; k_offsets subtracts its level's.  A level's total at or above 2^32 words is stored
// saturated, so that the host rejects the DAG.  Then the levels' bases (R >= 0): B[R] = 0, B[L-1] =
// B[L] + S[L], and the readback.  Levels' first tiles and the metadata are kept in LDS: looked up in
// the kernel's arguments by a varying index, and read back from memory, they took longer than the
// scan.
constexpr u32 kTotalsThreads = 1024;
constexpr u32 kInlineTiles = 1024;  // up to this many tiles k_offsets' workgroups scan them themselves
template <u32 kThreads>
__device__ inline void merge_totals(const MArgs& a, const u32* __restrict__ tile_sums, ulonglong2* __restrict__ tile_pre,
                                    u32* __restrict__ meta, int R, u32* __restrict__ host_meta) {
    constexpr u32 kWaves = kThreads / kWave, kPer = 4;
    __shared__ u32 s_c[2][kWaves], s_w[2][kWaves], s_tile0[kMaxLevels + 1], s_meta[kMetaWords];
    __shared__ u32 lev_c[kMaxLevels + 1];
    __shared__ u64 lev_w[kMaxLevels + 1];
    const u32 nt = a.tile0[a.nlev], nlev = (u32)a.nlev;
    const u32 lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
    if (threadIdx.x <= nlev) s_tile0[threadIdx.x] = a.tile0[threadIdx.x];
    for (u32 i = threadIdx.x; i < kMetaWords; i += kThreads)
        s_meta[i] = meta[i];
    u32 run_c = 0;  // of the chunks before
    u64 run_w = 0;
    u32 v[kPer];
    auto load = [&](u32 t0) {
#pragma unroll
        for (u32 j = 0; j < kPer; ++j)
            v[j] = (t0 + j < nt) ? tile_sums[t0 + j] : 0u;
    };
    load(threadIdx.x * kPer);
    u32 buf = 0;
    for (u32 base = 0; base < nt; base += kThreads * kPer, buf ^= 1u) {
        const u32 t0 = base + threadIdx.x * kPer;
        u32 x[kPer], c = 0, w = 0;  // (a chunk of 4096 tiles of at most 34816 words fits 32 bits)
#pragma unroll
        for (u32 j = 0; j < kPer; ++j) {
            x[j] = v[j];
            c += v[j] >> 16;
            w += v[j] & 0xFFFFu;
        }
        load(t0 + kThreads * kPer);  // the next chunk's, while this one is scanned
        const u32 ci = wave_inclusive_scan(c, OpSum{}), wi = wave_inclusive_scan(w, OpSum{});
        if (lane == kWave - 1) {
            s_c[buf][wid] = ci;
            s_w[buf][wid] = wi;
        }
        __syncthreads();  // (also: the levels' first tiles are in; the other buffer's readers are done)
        u32 pc = 0, pw = 0, tc = 0, tw = 0;
#pragma unroll
        for (u32 u = 0; u < kWaves; ++u) {
            if (u == wid) {
                pc = tc;
                pw = tw;
            }
            tc += s_c[buf][u];
            tw += s_w[buf][u];
        }
        u32 cc = run_c + pc + ci - c;
        u64 ww = run_w + pw + wi - w;
        run_c += tc;
        run_w += tw;
        u32 k = 0;
        while (k < nlev && s_tile0[k] < t0) ++k;
#pragma unroll
        for (u32 j = 0; j < kPer; ++j) {
            if (t0 + j >= nt) break;
            if (k < nlev && s_tile0[k] == t0 + j) {  // a level's first tile (every level has one)
                lev_c[k] = cc;
                lev_w[k] = ww;
                ++k;
            }
            if (tile_pre) tile_pre[t0 + j] = make_ulonglong2(cc, ww);
            cc += x[j] >> 16;
            ww += x[j] & 0xFFFFu;
        }
    }
    if (threadIdx.x == 0) {
        lev_c[nlev] = run_c;
        lev_w[nlev] = run_w;
    }
    __syncthreads();
    if (tile_pre && threadIdx.x <= nlev) tile_pre[nt + threadIdx.x] = make_ulonglong2(lev_c[threadIdx.x], lev_w[threadIdx.x]);
    if (threadIdx.x < nlev) {
        const u32 k = threadIdx.x;
        s_meta[kMetaU + a.lv[k].L] = lev_c[k + 1] - lev_c[k];
        s_meta[kMetaS + a.lv[k].L] = saturate32(lev_w[k + 1] - lev_w[k]);
    }
    __syncthreads();
    if (threadIdx.x == 0 && R >= 0) {
        s_meta[kMetaRoot] = a.lv[a.nlev - 1].mask[0];
        u64 acc = 0;
        for (int L = R; L >= 0; --L) {  // (levels absent have no words)
            s_meta[kMetaB + L] = saturate32(acc);
            acc += s_meta[kMetaS + L];
        }
        s_meta[kMetaW] = saturate32(acc);
    }
    __syncthreads();
    for (u32 i = threadIdx.x; i < kMetaWords; i += kThreads) {
        if (host_meta) reinterpret_cast<volatile u32*>(host_meta)[i] = s_meta[i];
        meta[i] = s_meta[i];
    }
    if (host_meta) {
        wait_stores();
        __syncthreads();
        if (threadIdx.x == 0) reinterpret_cast<volatile u32*>(host_meta)[kMetaWords] = 1u;  // ready: the host polls for it
    }
}

__global__ __launch_bounds__(kTotalsThreads) void k_totals(MArgs a, const u32* __restrict__ tile_sums,
                                                           ulonglong2* __restrict__ tile_pre, u32* __restrict__ meta, int R,
                                                           u32* __restrict__ host_meta) {
    merge_totals<kTotalsThreads>(a, tile_sums, tile_pre, meta, R, host_meta);
}

// First occurrences as bytes: flag[node] = the node's words if it is its key's first, else 0; and each
// tile's first occurrences << 16 | their words (at most 2048 and 34816).  The loads of the tile's
// rounds are issued together, stage by stage.
template <bool kSorted>
__global__ __launch_bounds__(kTileThreads) void k_firsts(MArgs a, u32* __restrict__ tile_sums) {
    __shared__ u32 s_wave[kTileThreads / kWave];
    const int k = level_of_tile(a, blockIdx.x);
    const MLevel& l = a.lv[k];
    const u32 n = l.n, base = (blockIdx.x - a.tile0[k]) * kTileNodes + threadIdx.x;
    u32 r[kTilePer], m[kTilePer];
    bool act[kTilePer];
#pragma unroll
    for (u32 j = 0; j < kTilePer; ++j) {
        const u32 i = base + j * kTileThreads;
        act[j] = i < n;
        if (l.leaf && act[j]) act[j] = a.heads[i] == i;  // a first occurrence heads its run
    }
#pragma unroll
    for (u32 j = 0; j < kTilePer; ++j) {
        const u32 i = base + j * kTileThreads;
        r[j] = (act[j] && !l.lone) ? l.id[i] : i;
        m[j] = act[j] ? l.mask[i] : 0u;
    }
    if (!kSorted && !l.lone) {
#pragma unroll
        for (u32 j = 0; j < kTilePer; ++j) r[j] = act[j] ? (u32)l.tab[min(r[j], l.slots - 1)] : 0u;
    }
    u32 acc = 0;
#pragma unroll
    for (u32 j = 0; j < kTilePer; ++j) {
        const u32 i = base + j * kTileThreads;
        const u32 w = (act[j] && r[j] == i) ? node_words(m[j], l.leaf) : 0u;
        if (i < n) l.flag[i] = (uint8_t)w;
        acc += w ? (1u << 16) | w : 0u;
    }
    acc = block_reduce(acc, s_wave, OpSum{});
    if (threadIdx.x == 0) tile_sums[blockIdx.x] = acc;
}

// The flags of a thread's kTilePer consecutive nodes of a tile.
__device__ inline u64 tile_flags(const MLevel& l, u32 tile, u32& i) {
    i = tile * kTileNodes + threadIdx.x * kTilePer;
    if (i >= l.n) return 0ull;
    const u64 v = *reinterpret_cast<const u64*>(l.flag + i);
    const u32 have = l.n - i;
    return have < kTilePer ? v & ((1ull << (8 * have)) - 1ull) : v;
}

// kInline: at most kInlineTiles tiles; each workgroup adds up those of its level before its own, and one
// more workgroup (the first, which the host waits for) does the totals meanwhile.
template <bool kInline>
__global__ __launch_bounds__(kTileThreads) void k_offsets(MArgs a, const u32* __restrict__ tile_sums,
                                                          const ulonglong2* __restrict__ tile_pre, u32* __restrict__ meta, int R,
                                                          u32* __restrict__ host_meta) {
    if (kInline && blockIdx.x == 0) {
        merge_totals<kTileThreads>(a, tile_sums, nullptr, meta, R, host_meta);
        return;
    }
    const u32 b = kInline ? blockIdx.x - 1 : blockIdx.x;
    const int k = level_of_tile(a, b);
    const MLevel& l = a.lv[k];
    u32 i0;
    const u64 v = tile_flags(l, b - a.tile0[k], i0);
    u32 rank;
    u64 off;
    if constexpr (kInline) {
        __shared__ u32 s_c[kTileThreads / kWave], s_w[kTileThreads / kWave];
        u32 c = 0, w = 0;  // (1024 tiles of at most 34816 words fit 32 bits)
        for (u32 t = a.tile0[k] + threadIdx.x; t < b; t += kTileThreads) {
            const u32 x = tile_sums[t];
            c += x >> 16;
            w += x & 0xFFFFu;
        }
        rank = block_reduce(c, s_c, OpSum{});
        off = block_reduce(w, s_w, OpSum{});
    } else {
        const ulonglong2 pre = tile_pre[b], lev = tile_pre[a.tile0[a.nlev] + k];
        rank = (u32)(pre.x - lev.x);
        off = pre.y - lev.y;
    }
    u32 sum[1] = {0}, ex[1];
#pragma unroll
    for (u32 q = 0; q < kTilePer; ++q) {
        const u32 w = (u32)(v >> (8 * q)) & 0xFFu;
        sum[0] += w ? (1u << 16) | w : 0u;
    }
    block_exclusive_scan_rounds<1>(sum, ex, OpSum{});
    if (!v) return;
    rank += ex[0] >> 16;
    off += ex[0] & 0xFFFFu;
    u32 id[kTilePer];
#pragma unroll
    for (u32 q = 0; q < kTilePer; ++q) id[q] = (((v >> (8 * q)) & 0xFFu) && !l.lone) ? l.id[i0 + q] : 0u;
#pragma unroll
    for (u32 q = 0; q < kTilePer; ++q) {
        const u32 w = (u32)(v >> (8 * q)) & 0xFFu;
        if (!w) continue;
        const u32 o = saturate32(off);
        l.uniq[rank] = i0 + q;
        l.off[rank] = o;
        if (!l.lone) l.tab[min(id[q], l.slots - 1)] = ((u64)rank << 32) | o;
        ++rank;
        off += w;
    }
}

// --- the words -------------------------------------------------------------------------------

// Every level's words in one launch, a grid-stride loop over the levels' blocks (their number is
// known on the device only, so no readback comes between): unique node r of an inner level as
// [mask, absolute offsets of its partial children], of the leaf level as [mask, (lo, hi) of each
// partial slice's leafmask] (src/CompressedShadow.cpp:326-392).
// The blocks from `writers` on make the compares that the late levels' inserts left out, one node a
// thread, each with its slot's first occurrence.  An insert of a small level is one chain of reads and
// atomics whatever its size, and the compare would make it longer; here it runs beside the write, and
// the host takes its collisions with the end of the write (256^2 100 -> 94.5 us, 1024^2 147 -> 141).
__device__ inline void compare_late(const MArgs& a, u32 block, u32* meta) {
    int k = 0;
    for (; k < a.nlev; ++k) {
        if (!a.lv[k].late) continue;
        const u32 nb = (a.lv[k].n + kNodeThreads - 1) / kNodeThreads;
        if (block < nb) break;
        block -= nb;
    }
    if (k == a.nlev) return;
    const MLevel& l = a.lv[k];
    const u32 i = block * kNodeThreads + threadIdx.x;
    if (i >= l.n || (l.leaf && a.heads[i] != i)) return;
    const u32 rank = (u32)(l.tab[min(l.id[i], l.slots - 1)] >> 32);  // (k_offsets' entry)
    const u32 r = (rank < l.n) ? l.uniq[rank] : i;
    if (r == i || r >= l.n) return;
    const u32 m = l.mask[i], mr = l.mask[r];
    bool same = m == mr;
    if (l.leaf) {
        const ulonglong2 *x = reinterpret_cast<const ulonglong2*>(a.leafm + (size_t)i * 8),
                         *y = reinterpret_cast<const ulonglong2*>(a.leafm + (size_t)r * 8);
        const u32 kk = same ? num_children(m) : 0u;
#pragma unroll
        for (u32 q = 0; q < 4; ++q)
            if (2 * q < kk) same = same && x[q].x == y[q].x && (2 * q + 1 >= kk || x[q].y == y[q].y);
    } else {
        const int kc = a.child(k);
        const ChildIds ch =
            kc >= 0 ? ChildIds{a.lv[kc].id, a.lv[kc].leaf ? a.heads : nullptr, a.lv[kc].n} : ChildIds{nullptr, nullptr, 1u};
        const u32 c = l.cstart[i], cr = l.cstart[r];
        const u32 kk = (same && ch.id) ? num_children(m) : 0u;
        if (kk) {
            u32 x[8], y[8];
            load_child_ids(ch, c, kk, x);
            load_child_ids(ch, cr, kk, y);
#pragma unroll
            for (u32 q = 0; q < 8; ++q) same = same && x[q] == y[q];
        }
    }
    if (!same) atomicAdd(meta + kMetaColl, 1u);
}

__global__ __launch_bounds__(kNodeThreads) void k_write_words(MArgs a, u32* meta, u32* __restrict__ out, u64 cap, u32 writers) {
    if (blockIdx.x >= writers) {
        compare_late(a, blockIdx.x - writers, meta);
        return;
    }
    __shared__ u32 s_first[kMaxLevels + 1], s_U[kMaxLevels], s_base[kMaxLevels], s_out[kStageWords];
    if (threadIdx.x < (u32)a.nlev) {
        s_U[threadIdx.x] = meta[kMetaU + a.lv[threadIdx.x].L];
        s_base[threadIdx.x] = meta[kMetaB + a.lv[threadIdx.x].L];
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        u32 acc = 0;
        for (int k = 0; k < a.nlev; ++k) {
            s_first[k] = acc;
            acc += (s_U[k] + kNodeThreads - 1) / kNodeThreads;
        }
        s_first[a.nlev] = acc;
    }
    __syncthreads();
    const u32 total = meta[kMetaW];
    if (total >= 0xFFFFFFFEu || total > cap) return;  // the host reports it
    const u32 nb = s_first[a.nlev];
    for (u32 vb = blockIdx.x; vb < nb; vb += writers) {
        int k = 0;
        while (k + 1 < a.nlev && vb >= s_first[k + 1]) ++k;
        const MLevel& l = a.lv[k];
        const u32 r0 = (vb - s_first[k]) * kNodeThreads, r = r0 + threadIdx.x;
        u32 o = 0, n = 0, w[17];
        if (r < s_U[k]) {
            const u32 i = l.uniq[r];
            o = l.off[r];
            w[0] = l.mask[i];
            const u32 kc = num_children(w[0]);
            n = node_words(w[0], l.leaf);
            if (l.leaf) {
                leaf_row(a.leafm + (size_t)i * 8, kc, w + 1);  // a first occurrence heads its run: its own row
            } else if (const int c = a.child(k); c >= 0 && kc) {
                const MLevel& lc = a.lv[c];
                const u32 s = l.cstart[i];
                u32 id[8];
#pragma unroll
                for (u32 j = 0; j < 8; ++j) id[j] = (j < kc) ? min(s + j, lc.n - 1) : 0u;
                if (lc.leaf && !a.sorted) {  // (children_of)
#pragma unroll
                    for (u32 j = 0; j < 8; ++j) id[j] = (j < kc) ? min(a.heads[id[j]], lc.n - 1) : 0u;
                }
#pragma unroll
                for (u32 j = 0; j < 8; ++j) id[j] = (j < kc) ? lc.id[id[j]] : 0u;
#pragma unroll
                for (u32 j = 0; j < 8; ++j) w[1 + j] = (j < kc) ? s_base[c] + (u32)lc.tab[min(id[j], lc.slots - 1)] : 0u;
            } else {
                n = 1;
            }
        }
        stage_words(s_out, l.off[r0], o, n, w, out + s_base[k], total - s_base[k]);
    }
}

// --- launches --------------------------------------------------------------------------------

static dim3 grid_of(u32 n, u32 block) { return dim3(ceil_div<u32>(n ? n : 1, block)); }

// The children's identities of level k.
static ChildIds children_of(const MArgs& a, int k, bool sorted) {
    const int c = a.child(k);
    if (c < 0) return ChildIds{nullptr, nullptr, 1u};
    return ChildIds{a.lv[c].id, (a.lv[c].leaf && !sorted) ? a.heads : nullptr, a.lv[c].n};
}

void table_clear(u64* tab, u64 slots, hipStream_t s) {
    const u64 blocks = (slots + 255) / 256;
    CPVS_LAUNCH("table_clear", k_table_clear, dim3((u32)(blocks < 65536 ? blocks : 65536)), dim3(256), 0, s, tab, slots);
}

void merge_insert(const MArgs& a, int k, const u64* hash, u32* meta, u32 hbits, hipStream_t s) {
    const MLevel& l = a.lv[k];
    if (l.leaf)
        CPVS_LAUNCH("insert_leaf", k_insert_leaf, grid_of(l.n, kLeafInsertThreads), dim3(kLeafInsertThreads), 0, s, l.mask,
                    a.leafm, a.heads, hash, l.n, l.tab, l.slots, l.id, meta, hbits, l.late);
    else if (l.n >= kInnerTwoMin)
        CPVS_LAUNCH("insert_inner", (k_insert_inner<2, 512>), grid_of(l.n, 1024), dim3(512), 0, s, l.mask, l.cstart,
                    children_of(a, k, false), l.n, l.tab, l.slots, l.id, meta, hbits, l.late);
    else if (l.n > kInnerSmallMax)
        CPVS_LAUNCH("insert_inner", (k_insert_inner<1, 512>), grid_of(l.n, 512), dim3(512), 0, s, l.mask, l.cstart,
                    children_of(a, k, false), l.n, l.tab, l.slots, l.id, meta, hbits, l.late);
    else
        CPVS_LAUNCH("insert_inner", (k_insert_inner<1, 256>), grid_of(l.n, 256), dim3(256), 0, s, l.mask, l.cstart,
                    children_of(a, k, false), l.n, l.tab, l.slots, l.id, meta, hbits, l.late);
}

void merge_sort_level(const MArgs& a, int k, const SortScratch& t, u32* meta, hipStream_t s) {
    const MLevel& l = a.lv[k];
    const ChildIds ch = children_of(a, k, true);
    if (l.leaf)
        CPVS_LAUNCH("sortkeys", k_sortkeys_leaf, grid_of(l.n, 256), dim3(256), 0, s, l.mask, a.leafm, a.heads, l.n, t.skey,
                    t.sval);
    else
        CPVS_LAUNCH("sortkeys", k_sortkeys_inner, grid_of(l.n, 256), dim3(256), 0, s, l.mask, l.cstart, ch, l.n, t.skey,
                    t.sval);
    radix_sort_pairs(t.skey, t.sval, t.ktmp, t.vtmp, l.n, 32, t.sort_scratch, s);
    device_scan(SegHeadIn{t.skey}, SegStartOut{t.seg}, l.n, OpMax{}, nullptr, t.scan_scratch, s);
    if (l.leaf)
        CPVS_LAUNCH("representative", k_representative<LeafEq>, grid_of(l.n, 256), dim3(256), 0, s, t.sval, t.seg, l.n,
                    LeafEq{l.mask, a.leafm, a.heads, l.n}, l.id, meta + kMetaSortColl);
    else
        CPVS_LAUNCH("representative", k_representative<InnerEq>, grid_of(l.n, 256), dim3(256), 0, s, t.sval, t.seg, l.n,
                    InnerEq{l.mask, l.cstart, ch.id, ch.n}, l.id, meta + kMetaSortColl);
}

void merge_finish(const MArgs& a, u32* tile_sums, ulonglong2* tile_pre, u32* meta, int R, u32* host_meta, hipStream_t s) {
    const u32 nt = a.tile0[a.nlev];
    if (a.sorted)
        CPVS_LAUNCH("firsts", k_firsts<true>, dim3(nt), dim3(kTileThreads), 0, s, a, tile_sums);
    else
        CPVS_LAUNCH("firsts", k_firsts<false>, dim3(nt), dim3(kTileThreads), 0, s, a, tile_sums);
    if (nt <= kInlineTiles) {
        CPVS_LAUNCH("offsets", k_offsets<true>, dim3(nt + 1), dim3(kTileThreads), 0, s, a, tile_sums, nullptr, meta, R,
                    host_meta);
        return;
    }
    CPVS_LAUNCH("totals", k_totals, dim3(1), dim3(kTotalsThreads), 0, s, a, tile_sums, tile_pre, meta, R, host_meta);
    CPVS_LAUNCH("offsets", k_offsets<false>, dim3(nt), dim3(kTileThreads), 0, s, a, tile_sums, tile_pre, nullptr, R, nullptr);
}

void merge_write(const MArgs& a, u32* meta, u32* out, u64 cap, hipStream_t s) {
    u32 most = 0, compares = 0;  // blocks of the largest possible write (every node unique), and of compare_late
    for (int k = 0; k < a.nlev; ++k) {
        most += ceil_div<u32>(a.lv[k].n, kNodeThreads);
        if (a.lv[k].late) compares += ceil_div<u32>(a.lv[k].n, kNodeThreads);
    }
    const u32 writers = most < 2048 ? most : 2048;
    CPVS_LAUNCH("write_words", k_write_words, dim3(writers + compares), dim3(kNodeThreads), 0, s, a, meta, out, cap, writers);
}

}  // namespace cpvs
