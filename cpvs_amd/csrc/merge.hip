// merge.hip -- equal subtrees merged level by level, and the DAG's words.
//
// Bottom-up, each level takes one launch: the key of every node -- its mask and the partial
// leafmasks, or its mask and its children's identities -- goes into the level's hash table, and the
// slot it ends in is the node's own identity for its parents' keys.  Slots never move, so equal keys
// have equal identities before anything is known of their order; what needs a finished table is
// left to three launches over all levels at once:
//   k_resolve   per node the smallest index in its slot, the full-key compare against it, and a bit
//               for each first occurrence; the first occurrences and words of each 1024-node tile;
//   k_totals    a scan of the tiles, the levels' totals and bases;
//   k_offsets   rank and word offset of every first occurrence, in index order, which is the order
//               that mergeLevel's linear search gives (src/CompressedShadowUtil.h:154-182).
// Ranks as identities took four launches a level (insert, resolve, scan, rank copies), and the copies
// alone read and wrote every node of the leaf level.
//
// Keys that a table cannot tell apart are found by the compares, and the build is done again with
// the sort merge, whose identities are first occurrences' indices.
#include "merge.hpp"

namespace cpvs {

// --- the table merge -------------------------------------------------------------------------

// One 64-bit word per slot: the key hash's high 32 bits (its tag) above the smallest node index
// with that hash, so a probe touches one cache line and a new key costs one atomic.  ~0 marks an
// empty slot (node indices stay below 2^32 - 1).  Two keys whose tags are equal and whose probe
// chains meet share a slot; the full-key compare in k_resolve then sends the build down the
// sorting path, as for equal 64-bit hashes.

__global__ __launch_bounds__(256) void k_table_clear(u64* __restrict__ tab, u32 S) {
    const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < S) tab[i] = kEmptySlot;
}

template <u32 kPer>
__global__ __launch_bounds__(kLeafInsertThreads) void k_insert_leaf(const u32* __restrict__ mask, const u64* __restrict__ leafm,
                                                                    const u32* __restrict__ runhead,
                                                                    const u64* __restrict__ hash, u32 n,
                                                                    u64* __restrict__ tab, u32 S, u32* __restrict__ tslot,
                                                                    u32* __restrict__ full, u32 hbits) {
    constexpr u32 kWindow = kPer * kLeafInsertThreads, kSlots = 2 * kWindow;  // at most half full: every probe ends
    __shared__ u64 gh[kSlots];
    __shared__ u32 gi[kSlots];  // smallest node index of the slot's hash, then its global slot
    __shared__ unsigned short glist[kWindow];  // LDS slots in use
    __shared__ u32 gcount;
    for (u32 j = threadIdx.x; j < kSlots; j += blockDim.x) {
        gh[j] = 0ull;  // 0 marks an empty LDS slot
        gi[j] = kNoRep;
    }
    if (threadIdx.x == 0) gcount = 0;
    const u32 i0 = blockIdx.x * kWindow + threadIdx.x;
    u32 rh[kPer];
#pragma unroll
    for (u32 k = 0; k < kPer; ++k) {
        const u32 i = i0 + k * kLeafInsertThreads;
        rh[k] = (i < n) ? runhead[i] : kNoRep;
    }
    // The key hash of each run's first node (the run's smallest index): from the leaf kernel where
    // a lane walked its column, else from its mask and leafmasks (its row at its own index).
    u64 h[kPer];
#pragma unroll
    for (u32 k = 0; k < kPer; ++k) {
        const u32 i = i0 + k * kLeafInsertThreads;
        h[k] = (hash && rh[k] == i) ? hash[i] : 0ull;
    }
    u32 hm[kPer];
#pragma unroll
    for (u32 k = 0; k < kPer; ++k) {
        const u32 i = i0 + k * kLeafInsertThreads;
        hm[k] = (rh[k] == i && h[k] == 0ull) ? mask[i] : 0u;
    }
#pragma unroll
    for (u32 k = 0; k < kPer; ++k) {
        const u32 i = i0 + k * kLeafInsertThreads;
        if (rh[k] != i) continue;
        if (h[k] == 0ull) h[k] = leaf_key_hash(hm[k], leafm + (size_t)i * 8);
        h[k] = weaken_hash(h[k], hbits);
        if (h[k] == 0ull) h[k] = 1ull;
    }
    __syncthreads();
    u32 ls[kPer];
#pragma unroll
    for (u32 k = 0; k < kPer; ++k) {
        const u32 i = i0 + k * kLeafInsertThreads;
        ls[k] = 0;
        if (rh[k] != i) continue;
        u32 sl = (u32)(h[k] ^ (h[k] >> 29)) & (kSlots - 1);
        for (;;) {
            const u64 cur = atomicCAS(reinterpret_cast<unsigned long long*>(gh + sl), 0ull, (unsigned long long)h[k]);
            if (cur == 0ull) {
                glist[atomicAdd(&gcount, 1u)] = (unsigned short)sl;
                break;
            }
            if (cur == h[k]) break;
            sl = (sl + 1) & (kSlots - 1);
        }
        atomicMin(gi + sl, i);
        ls[k] = sl;
    }
    __syncthreads();
    const u32 m = gcount;  // at most kWindow
    for (u32 j = threadIdx.x; j < m; j += blockDim.x) {
        const u32 sl = glist[j];
        gi[sl] = table_insert(tab, S, gh[sl], gi[sl], full);
    }
    __syncthreads();
#pragma unroll
    for (u32 k = 0; k < kPer; ++k) {
        const u32 i = i0 + k * kLeafInsertThreads;
        if (rh[k] == i) tslot[i] = gi[ls[k]];
    }
}

__global__ __launch_bounds__(kInsertBlock) void k_insert_inner(const u32* __restrict__ mask, const u32* __restrict__ cstart,
                                                               ChildIds ch, u32 n, u64* __restrict__ tab, u32 S,
                                                               u32* __restrict__ id, u32* __restrict__ full, u32 hbits) {
    const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
    const bool act = i < n;
    u64 h = 0;
    if (act) {
        const u32 m = mask[i], s = cstart[i];
        const u32 k = ch.id ? num_children(m) : 0u;
        u32 r[8] = {};
        if (k) load_child_ids(ch, s, k, r);
        h = weaken_hash(inner_key_hash(m, r), hbits);
    }
    const u32 slot = table_insert_group(tab, S, h, i, act, full);
    if (act) id[i] = slot;
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
// scan.  tile_sums and meta are read at agent scope: in k_resolve's last workgroup they were stored
// by other workgroups of the same launch.
constexpr u32 kTotalsThreads = 1024;
constexpr u32 kInlineTiles = 256;  // up to this many tiles k_resolve's last workgroup does this
template <u32 kThreads>
__device__ inline void merge_totals(const MArgs& a, const u32* tile_sums, ulonglong2* __restrict__ tile_pre,
                                    u32* __restrict__ meta, int R, u32* __restrict__ host_meta) {
    constexpr u32 kWaves = kThreads / kWave, kPer = 4;
    __shared__ u32 s_c[2][kWaves], s_w[2][kWaves], s_tile0[kMaxLevels + 1], s_meta[kMetaWords];
    __shared__ u32 lev_c[kMaxLevels + 1];
    __shared__ u64 lev_w[kMaxLevels + 1];
    const u32 nt = a.tile0[a.nlev], nlev = (u32)a.nlev;
    const u32 lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
    if (threadIdx.x <= nlev) s_tile0[threadIdx.x] = a.tile0[threadIdx.x];
    for (u32 i = threadIdx.x; i < kMetaWords; i += kThreads)
        s_meta[i] = __hip_atomic_load(meta + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    u32 run_c = 0;  // of the chunks before
    u64 run_w = 0;
    u32 v[kPer];
    auto load = [&](u32 t0) {
#pragma unroll
        for (u32 j = 0; j < kPer; ++j)
            v[j] = (t0 + j < nt) ? __hip_atomic_load(tile_sums + t0 + j, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0u;
    };
    load(threadIdx.x * kPer);
    u32 buf = 0;
    for (u32 base = 0; base < nt; base += kThreads * kPer, buf ^= 1u) {
        const u32 t0 = base + threadIdx.x * kPer;
        u32 x[kPer], c = 0, w = 0;  // (a chunk of 4096 tiles of at most 17408 words fits 32 bits)
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
            tile_pre[t0 + j] = make_ulonglong2(cc, ww);
            cc += x[j] >> 16;
            ww += x[j] & 0xFFFFu;
        }
    }
    if (threadIdx.x == 0) {
        lev_c[nlev] = run_c;
        lev_w[nlev] = run_w;
    }
    __syncthreads();
    if (threadIdx.x <= nlev) tile_pre[nt + threadIdx.x] = make_ulonglong2(lev_c[threadIdx.x], lev_w[threadIdx.x]);
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

template <bool kSorted>
__global__ __launch_bounds__(kTileThreads) void k_resolve(MArgs a, u32* tile_sums, ulonglong2* __restrict__ tile_pre,
                                                          u32* meta, int R, u32* __restrict__ host_meta) {
    u32* collisions = meta + kMetaColl;
    __shared__ u32 s_wave[kTileThreads / kWave];
    const int k = level_of_tile(a, blockIdx.x);
    const MLevel& l = a.lv[k];
    const u32 n = l.n, base = (blockIdx.x - a.tile0[k]) * kTileNodes + threadIdx.x;
    // The loads of the tile's rounds are issued together, stage by stage.
    u32 r[kTileRounds];
    bool act[kTileRounds];
#pragma unroll
    for (int j = 0; j < kTileRounds; ++j) {
        const u32 i = base + j * kTileThreads;
        act[j] = i < n;
        if (l.leaf && act[j]) act[j] = a.heads[i] == i;  // a first occurrence heads its run
    }
#pragma unroll
    for (int j = 0; j < kTileRounds; ++j) r[j] = (act[j] && !l.lone) ? l.id[base + j * kTileThreads] : 0u;
    if (!kSorted) {
#pragma unroll
        for (int j = 0; j < kTileRounds; ++j) r[j] = (act[j] && !l.lone) ? (u32)l.tab[min(r[j], l.slots - 1)] : 0u;
    }
    u32 acc = 0;  // first occurrences << 16 | their words (at most 1024 and 17408)
#pragma unroll
    for (int j = 0; j < kTileRounds; ++j) {
        const u32 i = base + j * kTileThreads;
        bool first = false;
        if (act[j]) {
            if (l.lone || r[j] >= n) r[j] = i;
            first = r[j] == i;
            const int kc = a.child(k);
            if (!kSorted && l.lone && kc >= 0 && a.lv[kc].leaf) {
                // A root over leaves (a 16 x 16 map) had no insert to store its children's identities.
                u32 unused[8];
                load_child_ids(ChildIds{a.lv[kc].id, a.heads, a.lv[kc].n}, l.cstart[i], num_children(l.mask[i]), unused);
            }
            if (!kSorted && !first) {
                const bool same = l.leaf ? LeafEq{l.mask, a.leafm, nullptr, n}(i, r[j])
                                         : InnerEq{l.mask, l.cstart, kc >= 0 ? a.lv[kc].id : nullptr, kc >= 0 ? a.lv[kc].n : 1u}(i, r[j]);
                if (!same) {
                    atomicAdd(collisions, 1u);  // two keys share a slot: the build is redone by sorting
                    __threadfence();  // counted before the workgroup's ticket
                    first = true;
                }
            }
            if (first) acc += (1u << 16) | node_words(l.mask[i], l.leaf);
        }
        const u64 bits = __ballot(first);
        if ((threadIdx.x & (kWave - 1)) == 0 && i < n) l.first[i / 64] = bits;
    }
    acc = block_reduce(acc, s_wave, OpSum{});
    if (gridDim.x > kInlineTiles) {  // k_totals follows
        if (threadIdx.x == 0) tile_sums[blockIdx.x] = acc;
        return;
    }
    // The last workgroup to finish does the totals: one launch less for small builds.
    __shared__ u32 s_last;
    if (threadIdx.x == 0) {
        __hip_atomic_store(tile_sums + blockIdx.x, acc, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        wait_stores();
        s_last = atomicAdd(meta + kMetaTicket, 1u) == gridDim.x - 1 ? 1u : 0u;
    }
    __syncthreads();
    if (!s_last) return;
    merge_totals<kTileThreads>(a, tile_sums, tile_pre, meta, R, host_meta);
}

__global__ __launch_bounds__(kTileThreads) void k_offsets(MArgs a, const ulonglong2* __restrict__ tile_pre) {
    const int k = level_of_tile(a, blockIdx.x);
    const MLevel& l = a.lv[k];
    const u32 base = (blockIdx.x - a.tile0[k]) * kTileNodes + threadIdx.x;
    const ulonglong2 pre = tile_pre[blockIdx.x], lev = tile_pre[a.tile0[a.nlev] + k];
    const u32 rank0 = (u32)(pre.x - lev.x);
    const u64 off0 = pre.y - lev.y;
    u32 v[kTileRounds], ex[kTileRounds], id[kTileRounds];
#pragma unroll
    for (int j = 0; j < kTileRounds; ++j) {
        const u32 i = base + j * kTileThreads;
        const bool first = i < l.n && ((l.first[i / 64] >> (i & 63)) & 1ull);
        v[j] = first ? 1u : 0u;
    }
#pragma unroll
    for (int j = 0; j < kTileRounds; ++j) {
        const u32 i = base + j * kTileThreads;
        id[j] = (v[j] && !l.lone) ? l.id[i] : 0u;
        if (v[j]) v[j] = (1u << 16) | node_words(l.mask[i], l.leaf);
    }
    block_exclusive_scan_rounds<kTileRounds>(v, ex, OpSum{});
#pragma unroll
    for (int j = 0; j < kTileRounds; ++j) {
        if (!v[j]) continue;
        const u32 rank = rank0 + (ex[j] >> 16);
        const u32 off = saturate32(off0 + (ex[j] & 0xFFFFu));
        l.uniq[rank] = base + j * kTileThreads;
        l.off[rank] = off;
        if (!l.lone) l.tab[min(id[j], l.slots - 1)] = ((u64)rank << 32) | off;
    }
}

// --- the words -------------------------------------------------------------------------------

// Every level's words in one launch, a grid-stride loop over the levels' blocks (their number is
// known on the device only, so no readback comes between): unique node r of an inner level as
// [mask, absolute offsets of its partial children], of the leaf level as [mask, (lo, hi) of each
// partial slice's leafmask] (src/CompressedShadow.cpp:326-392).
__global__ __launch_bounds__(kNodeThreads) void k_write_words(MArgs a, const u32* __restrict__ meta, u32* __restrict__ out,
                                                              u64 cap) {
    __shared__ u32 s_first[kMaxLevels + 1], s_U[kMaxLevels], s_base[kMaxLevels];
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
    for (u32 vb = blockIdx.x; vb < nb; vb += gridDim.x) {
        int k = 0;
        while (k + 1 < a.nlev && vb >= s_first[k + 1]) ++k;
        const MLevel& l = a.lv[k];
        const u32 r = (vb - s_first[k]) * blockDim.x + threadIdx.x;
        if (r >= s_U[k]) continue;
        const u32 i = l.uniq[r];
        const u32 o = s_base[k] + l.off[r];
        const u32 m = l.mask[i];
        out[o] = m;
        const u32 kc = num_children(m);
        if (!kc) continue;
        if (l.leaf) {
            const u64* p = a.leafm + (size_t)i * 8;  // a first occurrence heads its run: its own row
            u64 v[8];
#pragma unroll
            for (u32 j = 0; j < 8; ++j) v[j] = (j < kc) ? p[j] : 0ull;
#pragma unroll
            for (u32 j = 0; j < 8; ++j)
                if (j < kc) {
                    out[o + 1 + 2 * j] = (u32)v[j];
                    out[o + 2 + 2 * j] = (u32)(v[j] >> 32);
                }
            continue;
        }
        const int c = a.child(k);
        if (c < 0) continue;
        const MLevel& lc = a.lv[c];
        const u32 s = l.cstart[i];
        u32 id[8], co[8];
#pragma unroll
        for (u32 j = 0; j < 8; ++j) id[j] = (j < kc) ? lc.id[min(s + j, lc.n - 1)] : 0u;
#pragma unroll
        for (u32 j = 0; j < 8; ++j) co[j] = (j < kc) ? (u32)lc.tab[min(id[j], lc.slots - 1)] : 0u;
#pragma unroll
        for (u32 j = 0; j < 8; ++j)
            if (j < kc) out[o + 1 + j] = s_base[c] + co[j];
    }
}

// --- launches --------------------------------------------------------------------------------

static dim3 grid_of(u32 n, u32 block) { return dim3(ceil_div<u32>(n ? n : 1, block)); }

// The children's identities of level k: those of the leaf level reach its non-heads here.
static ChildIds children_of(const MArgs& a, int k, bool sorted) {
    const int c = a.child(k);
    if (c < 0) return ChildIds{nullptr, nullptr, 1u};
    return ChildIds{a.lv[c].id, (a.lv[c].leaf && !sorted) ? a.heads : nullptr, a.lv[c].n};
}

void merge_insert(const MArgs& a, int k, const u64* hash, u32* meta, u32 hbits, hipStream_t s) {
    const MLevel& l = a.lv[k];
    if (l.leaf && l.n <= kLeafOneMax)
        CPVS_LAUNCH("insert_leaf", k_insert_leaf<1>, grid_of(l.n, kLeafInsertThreads), dim3(kLeafInsertThreads), 0, s, l.mask,
                    a.leafm, a.heads, hash, l.n, l.tab, l.slots, l.id, meta + kMetaFull, hbits);
    else if (l.leaf)
        CPVS_LAUNCH("insert_leaf", k_insert_leaf<kLeafPer>, grid_of(l.n, kLeafPer * kLeafInsertThreads),
                    dim3(kLeafInsertThreads), 0, s, l.mask, a.leafm, a.heads, hash, l.n, l.tab, l.slots, l.id,
                    meta + kMetaFull, hbits);
    else
        CPVS_LAUNCH("insert_inner", k_insert_inner, grid_of(l.n, kInsertBlock), dim3(kInsertBlock), 0, s, l.mask, l.cstart,
                    children_of(a, k, false), l.n, l.tab, l.slots, l.id, meta + kMetaFull, hbits);
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

void merge_finish(const MArgs& a, bool sorted, u32* tile_sums, ulonglong2* tile_pre, u32* meta, int R, u32* host_meta,
                  hipStream_t s) {
    const u32 nt = a.tile0[a.nlev];
    if (sorted)
        CPVS_LAUNCH("resolve", k_resolve<true>, dim3(nt), dim3(kTileThreads), 0, s, a, tile_sums, tile_pre, meta, R,
                    host_meta);
    else
        CPVS_LAUNCH("resolve", k_resolve<false>, dim3(nt), dim3(kTileThreads), 0, s, a, tile_sums, tile_pre, meta, R,
                    host_meta);
    if (nt > kInlineTiles)
        CPVS_LAUNCH("totals", k_totals, dim3(1), dim3(kTotalsThreads), 0, s, a, tile_sums, tile_pre, meta, R, host_meta);
    CPVS_LAUNCH("offsets", k_offsets, dim3(nt), dim3(kTileThreads), 0, s, a, tile_pre);
}

void merge_write(const MArgs& a, const u32* meta, u32* out, u64 cap, hipStream_t s) {
    u32 most = 0;  // blocks of the largest possible write (every node unique)
    for (int k = 0; k < a.nlev; ++k) most += ceil_div<u32>(a.lv[k].n, kNodeThreads);
    CPVS_LAUNCH("write_words", k_write_words, dim3(most < 2048 ? most : 2048), dim3(kNodeThreads), 0, s, a, meta, out, cap);
}

}  // namespace cpvs
