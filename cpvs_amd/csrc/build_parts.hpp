// build_parts.hpp -- device code shared by the single-map build (build.hip) and the forest build
// of many maps (forest.hip): classification, the leaf columns, leaf hashing, the merge tables, the
// metadata layout and the staging of words.
//
// The subtree merge works on node indices, masks, child identities and leafmasks only, so a forest of
// many DAGs goes through the same merge kernels: its mask words carry the DAG's index in their
// upper 16 bits (hash and key compares then never merge across DAGs, and num_children() reads
// the low 16 bits only).
#pragma once

#include "internal.hpp"
#include "scan.hpp"

namespace cpvs {

constexpr u64 kHashSeed = 0x6A09E667F3BCC909ull;
constexpr u32 kNoRep = 0xFFFFFFFFu;

__device__ inline u32 fold32(u64 h) { return (u32)(h ^ (h >> 32)); }

__device__ inline u32 fmix32(u32 h) {
    h ^= h >> 16;
    h *= 0x85EBCA6Bu;
    h ^= h >> 13;
    h *= 0xC2B2AE35u;
    h ^= h >> 16;
    return h;
}

// ---------------------------------------------------------------------------------------
// 1. Inner classification: createChildmask (src/CompressedShadowUtil.cpp:20-54).
// ---------------------------------------------------------------------------------------
// The childmask of the node at level-L cell z from its 2 x 2 texels' rows a and b (L > 0).
__device__ inline u32 classify_texels(u32 z, float h, float4 a, float4 b) {
    const float mn[4] = {a.x, a.z, b.x, b.z}, mx[4] = {a.y, a.w, b.y, b.w};  // texel (x + (q&1), y + (q>>1))
    u32 mask = 0;
#pragma unroll
    for (u32 ch = 0; ch < 8; ++ch) {
        const u32 q = ch & 3;
        mask |= classify_cell(z + (ch >> 2), mn[q] * h, mx[q] * h) << (2 * ch);
    }
    return mask;
}
// The cell is clamped into the level: a node past a level's emitted children (counts that
// exceed them, which the host then reports) still reads inside the pyramid.
__device__ inline u32 classify_node(u64 c, const float2* __restrict__ lv, const float* __restrict__ depth, u32 N, int L,
                                    u32 T) {
    const u32 w = N >> L;
    const u32 x = min(unpack_x(c), w - 2) & ~1u, y = min(unpack_y(c), w - 2), z = unpack_z(c);
    const float h = (float)((N >> L) * T);
    if (L > 0)
        return classify_texels(z, h, *reinterpret_cast<const float4*>(lv + (size_t)y * w + x),
                               *reinterpret_cast<const float4*>(lv + (size_t)(y + 1) * w + x));
    const float2 a = *reinterpret_cast<const float2*>(depth + (size_t)y * N + x);
    const float2 b = *reinterpret_cast<const float2*>(depth + (size_t)(y + 1) * N + x);
    const float d[4] = {a.x, a.y, b.x, b.y};
    u32 mask = 0;
#pragma unroll
    for (u32 ch = 0; ch < 8; ++ch) mask |= classify_mid(z + (ch >> 2), d[ch & 3] * h) << (2 * ch);
    return mask;
}

// Leaf columns: per level-3 texel, in Morton order, one record {partial cells, first leaf's index in
// column order, first partial z cell, 0}, so a column's scalars come in one load and a node's four
// columns in one line.  The counts (x, z) come from
// the node-count pass, the starts (y) from a scan of the counts.
struct LeafColumns {
    uint4* info;
    u32* bfs;       // (column start + z - zs) -> breadth-first index of the leaf node
    u32 w3;         // N >> 3
};

struct ColCountIn {
    const uint4* info;
    __device__ u32 operator()(u32 i) const { return info[i].x; }
};
struct ColStartOut {
    uint4* info;
    __device__ void operator()(u32 i, u32 ex, u32) const { info[i].y = ex; }
};
// With several z-tiles most columns have no leaf node in a given tile.  One scan of
// (column has nodes ? 1 : 0) << 32 | nodes gives the column starts and the list of the columns
// with nodes, in column order (the halves cannot carry: node counts stay below 2^32).
struct ColPairIn {
    const uint4* info;
    __device__ u64 operator()(u32 i) const {
        const u32 c = info[i].x;
        return (c ? (1ull << 32) : 0ull) | c;
    }
};
struct ColListOut {
    uint4* info;
    u32* list;   // list[k] = the k-th column with nodes
    u32* nlist;  // device: the number of such columns
    u32 n;
    __device__ void operator()(u32 i, u64 ex, u64 v) const {
        info[i].y = (u32)ex;
        if ((u32)v) list[(u32)(ex >> 32)] = i;
        if (i == n - 1) *nlist = (u32)((ex + v) >> 32);
    }
};

// Scan functors: partial-child count in, (first child index, children coordinates) out.
struct ChildCountIn {
    const u32* mask;
    __device__ u32 operator()(u32 i) const { return num_children(mask[i]); }
};
// A level's classification inside its emit scan: the input classifies node i, and the output
// (which classifies it again from the same cached loads) stores the mask.  One launch per level
// fewer than a separate classify pass.
struct Classify {
    const u64* coord;
    const float2* lv;
    const float* depth;
    u32 N;
    int L;
    u32 T;
    __device__ u32 operator()(u32 i) const { return classify_node(coord[i], lv, depth, N, L, T); }
};
struct ClassifyCountIn {
    Classify cls;
    __device__ u32 operator()(u32 i) const { return num_children(cls(i)); }
};
struct EmitChildrenOut {
    const u32* mask;
    const u64* coord;
    u32* cstart;
    u64* child_coord;   // used when the child level is classified node by node
    u32 child_cap;      // nodes of the child level (exact count); writes beyond it are dropped
    LeafColumns cols;   // used when cols.bfs != null (the children are leaves)
    u32* mask_out = nullptr;  // when set, the node is classified here (cls) and its mask stored
    Classify cls = {};
    // The node's mask and cell, loaded by the scan before any output is written.
    struct Pre {
        u32 m;
        u64 c;
    };
    __device__ Pre load(u32 i) const { return Pre{mask_out ? cls(i) : mask[i], coord[i]}; }
    __device__ void operator()(u32 i, u32 first, u32 k, Pre pre) const {
        cstart[i] = first;
        if (mask_out) mask_out[i] = pre.m;
        if (!k) return;
        const u32 m = pre.m;
        const u64 c = pre.c;
        const u32 x = unpack_x(c), y = unpack_y(c), z = unpack_z(c);
        u32 j = first;
        // getChildCoordinates (src/CompressedShadowUtil.cpp:101-117): partial children in
        // ascending child index, child cell doubled.
        if (cols.bfs) {
            // (the column records read lie inside the level even for a node past its level's
            // emitted children)
            const u32 at = morton2(min(x, cols.w3 - 2) & ~1u, min(y, cols.w3 - 2) & ~1u);
            // Leaf children: children ch and ch + 4 lie in one column, so the node's (at most
            // four) column records are loaded first, all together, and the stores follow.
            uint4 ci[4];
#pragma unroll
            for (u32 q = 0; q < 4; ++q) {
                ci[q] = make_uint4(0u, 0u, 0u, 0u);
                if (m & ((2u << (2 * q)) | (2u << (2 * (q + 4))))) ci[q] = cols.info[at + q];
            }
#pragma unroll
            for (u32 ch = 0; ch < 8; ++ch) {
                if (!(m & (2u << (2 * ch)))) continue;
                const uint4 r = ci[ch & 3];
                const u32 slot = r.y + (z + (ch >> 2) - r.z);
                if (j < child_cap && slot < child_cap) cols.bfs[slot] = j;
                ++j;
            }
            return;
        }
#pragma unroll
        for (u32 ch = 0; ch < 8; ++ch) {
            if (!(m & (2u << (2 * ch)))) continue;
            // pack_xyz of the doubled child cell (no field of a node with children is near its width)
            if (j < child_cap) child_coord[j] = 2 * c + pack_xyz(2 * (ch & 1), 2 * ((ch >> 1) & 1), 2 * (ch >> 2));
            ++j;
        }
    }
};


// Empty slot of the merge hash tables (see table_insert).
constexpr u64 kEmptySlot = ~0ull;

// Grid-stride clear of the merge tables, folded into a kernel that runs before they are used.  A level's
// slots fit 32 bits; those of all levels, which lie in one run, need not.
__device__ inline void clear_table(u64* tab, u64 slots) {
    const u32 stride = gridDim.x * blockDim.x;
    for (u64 j = (u64)blockIdx.x * blockDim.x + threadIdx.x; j < slots; j += stride) tab[j] = kEmptySlot;
}

// Key hash of a leaf node (wave-uniform): two 32-bit multiply-xorshift streams over the low and
// high halves of the partial leafmasks, seeded by the childmask and coupled at every step, then
// a finaliser that is a bijection on the two streams (so it adds no collisions).
struct LeafHash {
    u32 a, b;
    __device__ explicit LeafHash(u32 mask) : a(mask * 0x9E3779B1u + 0x7F4A7C15u), b((mask ^ 0xA5A5u) * 0x85EBCA77u + 1u) {}
    __device__ void add(u64 m) {
        a = (a ^ (u32)m) * 0x9E3779B1u;
        a ^= a >> 15;
        b = (b ^ (u32)(m >> 32)) * 0x85EBCA77u;
        b ^= b >> 13;
        a += b;
    }
    __device__ u64 value() const {
        u32 x = (a ^ (b >> 16)) * 0x2C1B3C6Du;
        u32 y = (b ^ (x >> 15)) * 0x297A2D39u;
        x ^= y >> 13;
        return ((u64)y << 32) | x;
    }
};


// f = floor(D - 0.5) of a texel's scaled depth D = d * N * T: slice z of its column is lit iff
// z <= f (the midpoint test float(z) + 0.5 <= D, exact for |D| < 2^22).  NaN is never lit.  f is
// non-decreasing in d, so the f of a block's minimum (maximum) depth is the minimum (maximum) of
// its texels' f when the block holds no NaN.
__device__ inline int leaf_f(float D) {
    int f = -(1 << 30);
    if (D == D) f = (int)floorf(fminf(fmaxf(D, -2.0f), 4194304.0f) - 0.5f);
    return f;
}

// Key hash of a leaf node from its mask and its partial slices' leafmasks (slot8: the node's
// leafmask row, partial slices in ascending order).  All loads are issued before the hash.
__device__ inline u64 leaf_key_hash(u32 m, const u64* __restrict__ slot8) {
    const u32 k = num_children(m);
    u64 v[8];  // (16 bytes a load: a row takes half the line look-ups)
#pragma unroll
    for (u32 j = 0; j < 8; j += 2) {
        ulonglong2 x = make_ulonglong2(0ull, 0ull);
        if (j < k) x = *reinterpret_cast<const ulonglong2*>(slot8 + j);
        v[j] = x.x, v[j + 1] = x.y;
    }
    LeafHash hs(m);
#pragma unroll
    for (u32 j = 0; j < 8; ++j)
        if (j < k) hs.add(v[j]);
    return hs.value();
}

// Lane l of a vector value takes the wave-uniform v (v_writelane_b32, an ALU instruction this
// compiler has no builtin for); every other lane keeps `old`.  Works whatever the exec mask.  The
// lane select goes through M0 and the value through a plain SGPR (the instruction takes neither a
// second SGPR nor VCC beside M0).
// v and l must be wave-uniform; readfirstlane says so to the compiler (and costs nothing when
// they already sit in SGPRs).
__device__ inline u32 write_lane(u32 old, u32 v, u32 l) {
    u32 t;
    asm("s_mov_b32 %1, %2\n\ts_mov_b32 m0, %3\n\tv_writelane_b32 %0, %1, m0"
        : "+v"(old), "=&s"(t)
        : "s"(__builtin_amdgcn_readfirstlane(v)), "s"(__builtin_amdgcn_readfirstlane(l))
        : "m0");
    return old;
}

// One column's leaf nodes, the walk both leaf kernels (one map's and a forest's) run per column:
// nodes q = 0 .. cnt-1 of the column at level-2 z cells zs + q, lane = texel of the column's 8x8
// block with f = floor(depth * H - 0.5) (fmin, fmax: the column's extremes), first_bfs = the
// breadth-first index of node lane (the first 64 nodes), bfs_run[q] that of node q.  Writes each
// node's run head (the breadth-first index of its run's first node), and for every run head its
// mask (with gtag, a forest's DAG index, in the upper half) and the leafmasks of its partial slices
// in the row at its own index (8 slots per node); hash_out (may be null) gets 0 for each head.
// fl: the wave's 128 bytes of LDS flags.
//
// Node q differs from node q-1 iff some texel's h = f + 8 - 8*zs has h - 8q in [0, 14]: q =
// floor(h/8), or floor(h/8) - 1 when h mod 8 != 7.  Each lane flags its (at most two) nodes in LDS,
// then reads back the flag of node q0 + lane: one ballot gives a 64-node chunk's changed nodes.  LDS
// instructions of one wave run in program order, so the clear, the flags and the read need no wait
// between them; the fences keep the compiler from moving them across one another.
__device__ inline void leaf_column(int f, int fmin, int fmax, int zs, u32 cnt, u32 first_bfs, const u32* bfs_run,
                                   u32 gtag, u32 nleaf, uint8_t* fl, u32 lane, u32* __restrict__ mask_out,
                                   u64* __restrict__ leafm, u32* __restrict__ runhead, u64* __restrict__ hash_out) {
    const int h = f + 8 - 8 * zs;
    const int qa = h >> 3;  // floor(h / 8)
    const bool below = (h & 7) != 7;
    u32 head_bfs = 0;  // the run head carried into the next chunk
    // Nodes [q0, q0 + 64) of the column; bfs = breadth-first index of node q0 + lane.
    auto chunk = [&](u32 q0, u32 bfs) {
        const u32 qn = min(cnt - q0, 64u);
        const int ra = qa - (int)q0;
        // Node n's flag is byte n + 1 (n = -1 .. 63); every node outside the chunk lands on byte 65.
        // Bytes 0 .. 67 are cleared first (lanes past 16 repeat the last word).
        reinterpret_cast<u32*>(fl)[min(lane, 16u)] = 0u;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        fl[min((u32)(ra + 1), 65u)] = 1;           // node ra
        fl[below ? min((u32)ra, 65u) : 65u] = 1;   // node ra - 1
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        const bool hit = fl[lane + 1] != 0;           // read by every lane (no branch around it)
        u64 chg = __ballot(hit) & __ballot(lane < qn);  // wave-uniform
        if (q0 == 0) chg |= 1ull;            // a column's first node starts a run
        // The run heads of this chunk, one after the other (wave-uniform): mask and leafmasks (their
        // key hash is computed lane-parallel by the leaf insert, which reads them anyway).
        u32 my_mask = 0;
        // Node q0 + lane's run head: the last changed node at or before it, set head by head
        // (lanes before the chunk's first head continue the previous chunk's run).
        u32 my_head_bfs = head_bfs;
        // Node q0 + j lies at z8 = zb + 8j; its lit and partial slice counts come from the column
        // extremes relative to it.
        const int zb = 8 * (zs + (int)q0);
        const int fmin1 = fmin + 1 - zb, fmax1 = fmax + 1 - zb, fb = f - zb;
        for (u64 pend = chg; pend;) {
            const u32 j = (u32)__builtin_ctzll(pend);
            pend &= ~(1ull << j);
            const int j8 = 8 * (int)j;
            const int u = fb - j8;
            const u32 cmin = (u32)min(max(fmin1 - j8, 0), 8);
            const u32 cmax = (u32)min(max(fmax1 - j8, 0), 8);
            const u32 below_min = (1u << (2 * cmin)) - 1u, below_max = (1u << (2 * cmax)) - 1u;
            const u32 mask = (0x5555u & below_min) | (0xAAAAu & below_max & ~below_min) | gtag;
            u32 mine_lo = 0, mine_hi = 0;  // lane s gets the leafmask of partial slice cmin + s
            const u32 kp = cmax - cmin;
            for (u32 sl = 0; sl < kp; ++sl) {
                const u64 m = __ballot(u >= (int)(cmin + sl));
                mine_lo = write_lane(mine_lo, (u32)m, sl);
                mine_hi = write_lane(mine_hi, (u32)(m >> 32), sl);
            }
            // The head's leafmask row sits at its own breadth-first index.
            const u32 hrow = __builtin_amdgcn_readlane(bfs, j);
            if (lane < kp && hrow < nleaf)  // the two halves stored as they are (no 64-bit assembly)
                *reinterpret_cast<uint2*>(leafm + (size_t)hrow * 8 + lane) = make_uint2(mine_lo, mine_hi);
            my_mask = write_lane(my_mask, mask, j);
            my_head_bfs = (lane >= j) ? hrow : my_head_bfs;
        }
        head_bfs = __builtin_amdgcn_readlane(my_head_bfs, qn - 1);
        // nleaf bounds every index (only exceeded if the column map were inconsistent).
        if (lane < qn && bfs < nleaf) {
            runhead[bfs] = my_head_bfs;
            if ((chg >> lane) & 1ull) {
                mask_out[bfs] = my_mask;
                if (hash_out) hash_out[bfs] = 0ull;  // the leaf insert computes it from the row
            }
        }
    };
    // The first chunk's indices are staged; a longer column (box walls) loads the rest here.
    chunk(0u, first_bfs);
    for (u32 q0 = 64; q0 < cnt; q0 += 64) chunk(q0, bfs_run[min(q0 + lane, cnt - 1)]);
}

constexpr u32 kXcds = 8;

// ---------------------------------------------------------------------------------------
// Leaf columns, one column per lane.  A smooth surface crosses an 8x8 block in a few slices, all
// of them in one to three nodes; such a column's 64 texels stay in one lane's registers, and each
// partial slice's leafmask is 64 compares and carries (two instructions per texel for 64 columns
// at once, where the wave-per-column walk issues a ballot, its placement and the scalar work of a
// run head for one).  A column with more than kLaneSlices partial slices or kLaneNodes nodes (box
// walls, steep surfaces) or with a texel that is not finite goes to a list that the wave-per-column
// kernel walks in a launch of its own: shared out inside the workgroup, a box's edge kept four waves
// busy long after the other workgroups were done.
// ---------------------------------------------------------------------------------------
constexpr u32 kLaneThreads = 256;  // columns per workgroup
constexpr int kLaneSlices = 16;
constexpr u32 kLaneNodes = 4;

// One level-3 column: its index and 8x8 depth block, its leaf nodes' count, first column slot and
// first z, and its DAG's tag.
struct LeafCol {
    u32 col;
    const float* blk;
    u32 pitch;
    float HT;
    u32 cnt, start;
    int zs;
    u32 gtag;
};
struct LeafOut {
    const u32* bfs;  // column slot -> breadth-first index
    u32* mask;
    u64* leafm;
    u32* runhead;
    u64* hash;  // key hash of every run head whose column a lane walked, 0 for the others' (null: no lanes)
    u32* slow;  // the columns left to the wave-per-column kernel, *n_slow of them
    u32* n_slow;
    u32 nleaf;
};

// m with the bits of one texel's compare shifted in: 2 m + (zf <= d), two instructions.
__device__ inline u32 shift_in_le(u32 m, float zf, float d) {
    asm("v_cmp_le_f32 vcc, %1, %2\n\tv_addc_co_u32 %0, vcc, %0, %0, vcc" : "+v"(m) : "v"(zf), "v"(d) : "vcc");
    return m;
}

// Walks one column per lane; returns false when the column must be walked by a wave.
__device__ inline bool leaf_lane(const LeafCol& c, const LeafOut& o) {
    if (c.cnt == 0) return true;
    if (c.cnt > kLaneNodes) return false;
    float D[64];
#pragma unroll
    for (u32 r = 0; r < 8; ++r) {
        const float4* row = reinterpret_cast<const float4*>(c.blk + (size_t)r * c.pitch);
        const float4 a = row[0], b = row[1];
        D[8 * r + 0] = a.x, D[8 * r + 1] = a.y, D[8 * r + 2] = a.z, D[8 * r + 3] = a.w;
        D[8 * r + 4] = b.x, D[8 * r + 5] = b.y, D[8 * r + 6] = b.z, D[8 * r + 7] = b.w;
    }
    u32 b[kLaneNodes];
#pragma unroll
    for (u32 q = 0; q < kLaneNodes; ++q) b[q] = o.bfs[c.start + min(q, c.cnt - 1)];
    float lo = D[0], hi = D[0], sum = D[0];
#pragma unroll
    for (u32 t = 1; t < 64; ++t) {
        lo = fminf(lo, D[t]);
        hi = fmaxf(hi, D[t]);
        sum += D[t];
    }
    // Slices below zlo are lit at every texel, slices from zhi on at none (scaling by HT keeps the
    // order, and leaf_f is non-decreasing).
    const int zlo = leaf_f(lo * c.HT) + 1, zhi = leaf_f(hi * c.HT) + 1;
    const bool finite = sum - sum == 0.0f;  // no NaN or infinity (one that only the sum makes is set aside too)
    if (!finite || zhi - zlo > kLaneSlices) return false;
#pragma unroll
    for (u32 t = 0; t < 64; ++t) D[t] *= c.HT;
    const int z0 = 8 * c.zs, z1 = z0 + 8 * (int)c.cnt;  // the column's slices
    auto node_mask = [&](int zb) {
        const u32 cmin = (u32)min(max(zlo - zb, 0), 8), cmax = (u32)min(max(zhi - zb, 0), 8);
        const u32 below_min = (1u << (2 * cmin)) - 1u, below_max = (1u << (2 * cmax)) - 1u;
        return (0x5555u & below_min) | (0xAAAAu & below_max & ~below_min) | c.gtag;
    };
    // A node heads a run unless it is all lit or all shadow as the node below it.
    u32 head = 0, prev = 0;
#pragma unroll
    for (u32 q = 0; q < kLaneNodes; ++q) {
        if (q >= c.cnt) break;
        const u32 m = node_mask(z0 + 8 * (int)q);
        const bool part = (m & 0xAAAAu) != 0;
        const bool is_head = q == 0 || part || m != prev;
        prev = m;
        if (is_head) head = b[q];
        if (b[q] < o.nleaf) {  // (only exceeded if the column map were inconsistent)
            o.runhead[b[q]] = head;
            if (is_head) {
                o.mask[b[q]] = m;
                if (!part) {
                    const u64 h = LeafHash(m).value();
                    o.hash[b[q]] = h ? h : 1ull;
                }
            }
        }
    }
    // The partial slices, in order: leafmask, its place in its node's row, the node's key hash.
    const int ze = min(zhi, z1);
    u32 bq = 0, k = 0;
    LeafHash hs(0);
    for (int z = max(zlo, z0); z < ze; ++z) {
        const float zf = (float)z + 0.5f;
        u32 mlo = 0, mhi = 0;
#pragma unroll
        for (int t = 31; t >= 0; --t) mlo = shift_in_le(mlo, zf, D[t]);
#pragma unroll
        for (int t = 63; t >= 32; --t) mhi = shift_in_le(mhi, zf, D[t]);
        const u32 q = (u32)(z - z0) >> 3;
        if (k == 0) {
            bq = q == 0 ? b[0] : q == 1 ? b[1] : q == 2 ? b[2] : b[3];
            hs = LeafHash(node_mask(z0 + 8 * (int)q));
        }
        const u64 m = ((u64)mhi << 32) | mlo;
        if (bq < o.nleaf) o.leafm[(size_t)bq * 8 + k] = m;
        hs.add(m);
        ++k;
        if ((z & 7) == 7 || z + 1 == ze) {
            const u64 h = hs.value();
            if (bq < o.nleaf) o.hash[bq] = h ? h : 1ull;
            k = 0;
        }
    }
    return true;
}

// One column by a wave, lane = texel (all arguments but the lane's texel are wave-uniform); ext: its
// level-3 pyramid texel, the block's depth minimum and maximum (a block holding a NaN takes its
// extremes from its texels instead: the pyramid keeps a NaN only as a first operand).
__device__ inline void leaf_wave(const LeafCol& c, const float2* ext, const LeafOut& o, uint8_t* fl, u32 lane) {
    const float d = c.blk[(size_t)(lane >> 3) * c.pitch + (lane & 7)];
    const u32 b = o.bfs[c.start + min(lane, c.cnt - 1)];
    const float2 e = *ext;
    const float D = d * c.HT;
    const int f = leaf_f(D);
    int fmin = leaf_f(e.x * c.HT), fmax = leaf_f(e.y * c.HT);
    if (__ballot(!(D == D))) {
        fmin = __ockl_wfred_min_i32(f);
        fmax = __ockl_wfred_max_i32(f);
    }
    fmin = __builtin_amdgcn_readfirstlane(fmin);
    fmax = __builtin_amdgcn_readfirstlane(fmax);
    leaf_column(f, fmin, fmax, c.zs, c.cnt, b, o.bfs + c.start, c.gtag, o.nleaf, fl, lane, o.mask, o.leafm, o.runhead, o.hash);
}

// The entries of a list of n columns that workgroup b of g takes: u0, u0 + step, ... below end.  XCD x
// (workgroups x, x + kXcds, ...) takes a contiguous range: a 2 x 2 group's columns follow one another
// in the list, and their nodes one another in breadth-first order, so their run heads share lines,
// which one L2 then writes once (8192^2: 47 -> 35 us, 8 z-tiles 27 -> 19 us each; the walks wrote 110 MB).  g is a multiple of kXcds.
struct ListShare {
    u32 u0, end, step;
};
__device__ inline ListShare list_share(u32 n, u32 b, u32 g) {
    const u32 chunk = (n + kXcds - 1) / kXcds, x = b % kXcds;
    return ListShare{x * chunk + b / kXcds, min(n, (x + 1) * chunk), g / kXcds};
}

// The lanes' columns, those set aside appended to the list (one atomic per wave).
__device__ inline void leaf_lanes(const LeafCol& c, const LeafOut& o) {
    const bool slow = !leaf_lane(c, o);
    const u64 m = __ballot(slow);
    if (!m) return;
    const u32 lane = threadIdx.x & 63;
    u32 at = 0;
    if (lane == (u32)__builtin_ctzll(m)) at = atomicAdd(o.n_slow, (u32)__popcll(m));
    at = __builtin_amdgcn_readlane(at, __builtin_ctzll(m));
    // (a listed column has a node, so the list holds at most nleaf)
    const u32 k = at + (u32)__popcll(m & ((1ull << lane) - 1ull));
    if (slow && k < o.nleaf) o.slow[k] = c.col;
}

// The identity of each node of a level for its parents' keys: equal for equal subtrees, different
// otherwise (up to hash collisions, which the key compares find): the node's merge-table slot, or its
// first occurrence's index with the sort merge.  With heads set the level is the leaf level and only
// runs' first nodes (heads[c] == c) have one: a child's is its run's.
struct ChildIds {
    const u32* id;
    const u32* heads;
    u32 n;  // nodes of the level: bounds every index (first children past a level's emitted nodes)
};

// Identities of k children from node s on (entries j >= k are 0).  All loads of a stage are issued
// before any is used, so a node costs one memory round trip per stage, not one per child.
__device__ inline void load_child_ids(const ChildIds& c, u32 s, u32 k, u32 r[8]) {
    u32 at[8];
#pragma unroll
    for (u32 j = 0; j < 8; ++j) at[j] = min(s + j, c.n - 1);
    if (!c.heads) {
#pragma unroll
        for (u32 j = 0; j < 8; ++j) r[j] = (j < k) ? c.id[at[j]] : 0u;
        return;
    }
    u32 h[8];
#pragma unroll
    for (u32 j = 0; j < 8; ++j) h[j] = (j < k) ? c.heads[at[j]] : 0u;
#pragma unroll
    for (u32 j = 0; j < 8; ++j) r[j] = (j < k) ? c.id[min(h[j], c.n - 1)] : 0u;
}

// Key hash of an inner node with mask m, k children and their identities r: a sum of (mask,
// identities) times fixed odd 64-bit constants, whose collisions need an exact zero of the
// differences' sum mod 2^64, then a mixer that is a bijection.  Two 32-bit multiplies per child
// instead of a chain of two 64-bit ones: in the one-workgroup merge of the small levels, four waves
// per SIMD hash four nodes per thread and level, and a chain's multiplies alone were much of its time.
// The constants are published ones with well spread bits: splitmix64's increment (2^64 over the golden
// ratio), two of xxHash64's primes, the rrmxmx mixer's multiplier and wyhash's default secrets.
__device__ inline u64 inner_key_hash(u32 m, const u32 (&r)[8]) {
    constexpr u64 kMul[9] = {0x9E3779B97F4A7C15ull, 0xC2B2AE3D27D4EB4Full, 0x165667B19E3779F9ull, 0xD6E8FEB86659FD93ull,
                             0xA0761D6478BD642Full, 0xE7037ED1A0B428DBull, 0x8EBC6AF09C88C6E3ull, 0x589965CC75374CC3ull,
                             0x1D8E4E27C47D124Full};
    u64 h = kHashSeed + m * kMul[8];
#pragma unroll
    for (u32 j = 0; j < 8; ++j) h += r[j] * kMul[j];  // (entries past the children are 0)
    return mix64(h);
}

// A merge hash cut to its low `bits` bits, in both the tag and the slot position, so that distinct
// keys collide (bits = 0: the full hash).  Builds use it only to exercise collision detection.
__device__ inline u64 weaken_hash(u64 h, u32 bits) {
    if (!bits) return h;
    const u32 t = (u32)h & ((1u << bits) - 1u);
    return ((u64)t << 32) | t;
}

// Run heads are bounded by the level's n nodes where they are used as indices:
// past a level's emitted children (counts that exceed them, which the host then reports) the
// entries were never written.
struct LeafEq {
    const u32* mask;
    const u64* leafm;     // a run's first node's partial leafmasks: the row at that node's index
    const u32* runhead;   // when set, a node's key is read from its run's first node
    u32 n;                // nodes of the leaf level
    __device__ bool operator()(u32 a, u32 b) const {
        if (runhead) {
            const u32 ha = runhead[a], hb = runhead[b];
            a = (ha < n) ? ha : a;
            b = (hb < n) ? hb : b;
            if (a == b) return true;
        }
        const u32 m = mask[a], mb = mask[b];
        if (m != mb) return false;
        const u32 k = num_children(m);
        const u64* pa = leafm + (size_t)a * 8;
        const u64* pb = leafm + (size_t)b * 8;
        bool eq = true;
#pragma unroll
        for (u32 j = 0; j < 8; ++j)
            if (j < k) eq = eq && (pa[j] == pb[j]);
        return eq;
    }
};
struct InnerEq {
    const u32* mask;
    const u32* cstart;
    const u32* child_id;  // null at the deepest level
    u32 child_n;
    __device__ bool operator()(u32 a, u32 b) const {
        // Masks and first-child indices are loaded together (one round trip before the identities).
        const u32 m = mask[a], mb = mask[b];
        const u32 ca = cstart[a], cb = cstart[b];
        if (m != mb) return false;
        const u32 k = child_id ? num_children(m) : 0u;
        if (!k) return true;
        u32 ra[8], rb[8];
#pragma unroll
        for (u32 j = 0; j < 8; ++j) {
            ra[j] = (j < k) ? child_id[min(ca + j, child_n - 1)] : 0u;
            rb[j] = (j < k) ? child_id[min(cb + j, child_n - 1)] : 0u;
        }
        bool eq = true;
#pragma unroll
        for (u32 j = 0; j < 8; ++j) eq = eq && (ra[j] == rb[j]);
        return eq;
    }
};

// Open addressing, linear probing.  Large groups of equal keys hit one slot, so the slot is read
// first, and only an empty slot or a larger index costs an atomic.  A slot only ever goes from
// empty to one tag, and its index only decreases, so a stale read merely leads to an atomic that
// was not needed.  The read is an agent-scope load, which is served coherently across the XCDs:
// each XCD's L2 would otherwise keep showing a slot as empty after another XCD's atomic (atomics
// are performed at memory) had filled it, and every later insert of that key from the XCD would
// pay an atomic round trip.  Measured at 8192^2: leaf insert 77 -> 55 µs, inner inserts 137 ->
// 104 µs against a plain load.
// A probe gives up after kMaxProbes occupied slots (a table too small for its keys: the leaf
// level's table is sized for a quarter of its nodes), counts that in *full and returns a slot in
// range; the host then builds again with a larger table (whatever a slot holds is bounded where it is
// used as an index).
// occ: a node that the slot held (equal keys, unless hashes collide: the caller compares), or kNoRep
// when this one took it first.  Every node of a slot is compared with one that came before it, so
// compares that all hold make all the slot's keys equal.
constexpr u32 kMaxProbes = 256;
__device__ inline u32 table_insert(u64* tab, u32 S, u64 h, u32 i, u32* full, u32& occ) {
    occ = kNoRep;
    const u32 tag = (u32)(h >> 32);
    const u64 mine = ((u64)tag << 32) | i;
    u32 slot = __umulhi((u32)(h ^ (h >> 31)) * 0x9E3779B1u, S);
    for (u32 probe = 0; probe < kMaxProbes; ++probe) {
        u64 cur = __hip_atomic_load(tab + slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (cur == kEmptySlot) {
            cur = atomicCAS(reinterpret_cast<unsigned long long*>(tab + slot), (unsigned long long)kEmptySlot,
                            (unsigned long long)mine);
            if (cur == kEmptySlot) return slot;
        }
        if ((u32)(cur >> 32) == tag) {
            occ = (u32)cur;
            if ((u32)cur > i) atomicMin(reinterpret_cast<unsigned long long*>(tab + slot), (unsigned long long)mine);
            return slot;
        }
        if (++slot == S) slot = 0;
    }
    atomicAdd(full, 1u);
    return slot;
}

constexpr u32 kLeafInsertThreads = 256;
constexpr u32 kInnerTwoMin = 1u << 20, kInnerSmallMax = 1u << 18;

// Threads per workgroup of the write kernels (at 8192^2, 128 and 256 tie; 512 and 1024 are slower).
constexpr u32 kNodeThreads = 256;

// A workgroup's nodes have consecutive ranks, so their words are one run of the level.  Each thread puts
// its n words (at offset o of the level, the first thread's at o0) in LDS, and the run goes out side by
// side; stores by node touched 64 lines each.  cap: words that fit at out (nothing is written past).
// Every thread calls it (barriers); n = 0: no node.  8192^2 42 -> 39 us, 32 maps 122 -> 102.
constexpr u32 kStageWords = 17 * kNodeThreads;
__device__ inline void stage_words(u32* s_out, u32 o0, u32 o, u32 n, const u32 (&w)[17], u32* out, u32 cap) {
    __shared__ u32 s_end;
    if (threadIdx.x == 0) s_end = 0;
    __syncthreads();
    if (n) {
#pragma unroll
        for (u32 j = 0; j < 17; ++j)
            if (j < n && o - o0 + j < kStageWords) s_out[o - o0 + j] = w[j];
    }
    const u32 end = wave_reduce(n ? o - o0 + n : 0u, OpMax{});
    if ((threadIdx.x & (kWave - 1)) == 0) atomicMax(&s_end, end);
    __syncthreads();
    const u32 m = min(min(s_end, kStageWords), o0 < cap ? cap - o0 : 0u);
    for (u32 j = threadIdx.x; j < m; j += kNodeThreads) out[o0 + j] = s_out[j];
    __syncthreads();
}

// A leaf node's k leafmasks as words (lo, hi of each), from its row.
__device__ inline void leaf_row(const u64* row, u32 k, u32* w) {
#pragma unroll
    for (u32 j = 0; j < 8; j += 2) {
        ulonglong2 x = make_ulonglong2(0ull, 0ull);
        if (j < k) x = *reinterpret_cast<const ulonglong2*>(row + j);
        w[2 * j] = (u32)x.x, w[2 * j + 1] = (u32)(x.x >> 32), w[2 * j + 2] = (u32)x.y, w[2 * j + 3] = (u32)(x.y >> 32);
    }
}

// Segment start of each sorted position: max-scan of (key differs from predecessor ? p : 0).
struct SegHeadIn {
    const u32* skey;
    __device__ u32 operator()(u32 p) const { return (p == 0 || skey[p] != skey[p - 1]) ? p : 0u; }
};
struct SegStartOut {
    u32* seg;
    __device__ void operator()(u32 p, u32 ex, u32 v) const { seg[p] = ex > v ? ex : v; }
};

// Representative (first occurrence) of each node.  Within a segment of equal 32-bit keys the
// stable sort keeps node indices ascending, so the head is the smallest index.
template <class Eq>
__global__ __launch_bounds__(256) void k_representative(const u32* __restrict__ sval, const u32* __restrict__ seg, u32 count,
                                                        Eq eq, u32* __restrict__ rep, u32* __restrict__ collisions) {
    const u32 p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= count) return;
    const u32 i = sval[p];
    const u32 s = seg[p];
    const u32 head = sval[s];
    u32 r = head;
    if (head != i && !eq(i, head)) {
        atomicAdd(collisions, 1u);
        r = i;
        for (u32 q = s + 1; q < p; ++q) {
            const u32 j = sval[q];
            if (eq(i, j)) {
                r = j;
                break;
            }
        }
    }
    rep[i] = r;
}


// Device metadata block (u32 words).
enum : int {
    kMetaU = 0,                          // uniques per level
    kMetaS = kMaxLevels,                 // words per level
    kMetaB = 2 * kMaxLevels,             // level base offsets
    kMetaC = 3 * kMaxLevels,             // children emitted per level (scan totals)
    kMetaW = 4 * kMaxLevels,             // total words
    kMetaColl = 4 * kMaxLevels + 1,      // key collisions in the hash table (table merge)
    kMetaRoot = 4 * kMaxLevels + 2,      // root mask
    kMetaSortColl = 4 * kMaxLevels + 3,  // 32-bit key collisions resolved by a scan (sort merge)
    kMetaFull = 4 * kMaxLevels + 4,      // table inserts that found no free slot (table merge)
    kMetaSlow = 4 * kMaxLevels + 5,      // leaf columns left to the wave-per-column kernel
    kMetaWords = 4 * kMaxLevels + 6,
};


// Launches over this many columns walk them one per lane (a map's are then at least 16 x 16).
constexpr u64 kLaneLeafMin = 1u << 15;
constexpr u32 kSlowWaves = 8192;  // waves that stride over a list of columns: the chip's 32 per CU
inline u32 list_waves(u32 most) { return most < kSlowWaves ? (most + kXcds - 1) / kXcds * kXcds : kSlowWaves; }

// Slots for n keys, at most two thirds full.
inline u32 table_slots(u64 n) {
    const u64 S = n + n / 2 + 1;
    return S < 1024 ? 1024u : (u32)(S < 0xFFFFFFFFull ? S : 0xFFFFFFFFull);
}
// Large levels repeat their nodes (8192^2: 5% of the leaves and 15% of the nodes above them are
// distinct, 1024^2 25-40%), and a table that is not needed costs its clear and, spread wide, a cache
// miss for every probe and look-up: from 2^20 nodes on a leaf level gets slots for a quarter of its
// nodes and an inner level for half.  A table found too small (maps of mostly distinct leaves, such
// as white noise) is reported, and the build runs again with small = false.
constexpr u32 kSmallTableMin = 1u << 20;
inline u32 leaf_table_slots(u64 c, bool small) { return table_slots((small && c >= kSmallTableMin) ? c / 4 : c); }
// Small inner levels' tables are at most a quarter full: each probe is a read from memory, and where
// every key is distinct (the upper levels of a forest, whose keys hold the DAG's index) the longest run
// of occupied slots in a two-thirds table is tens of probes (32 maps: 3 K nodes 22.9 -> 9.9 us, 18 K
// nodes 14.7 -> 9.5; the batch 2047 -> 2011, a server's burst 360 -> 351).
constexpr u32 kSparseTableMax = 1u << 17;
inline u32 inner_table_slots(u64 c, bool small) {
    return c < kSparseTableMax ? table_slots(c * 8 / 3) : table_slots((small && c >= kSmallTableMin) ? c / 2 : c);
}

}  // namespace cpvs
