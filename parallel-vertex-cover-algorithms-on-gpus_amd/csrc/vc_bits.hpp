// vc_bits.hpp -- search of a small remainder (at most 256 live vertices) in
// registers; included by vc_kernels.hip.
//
// Once a tree node has at most 64 K live vertices (K = 1, 2 or 4), its whole
// subtree is searched on the induced subgraph: vertex i of the remainder
// (live vertices in increasing order) belongs to lane i % 64, slot i / 64,
// and the lane holds its adjacency row as 2 K words.  A node of that subtree
// is then one wave-uniform mask of K 64-bit words (the vertices not in the
// cover) in scalar registers:
//   degree      popcount of row & mask, per lane
//   leaf rule   one test per lane: row & (mask of degree-1 vertices)
//   take a set  mask &= ~set (no neighbour is touched)
//   stack       8 K bytes of mask instead of 8 bytes per vertex
// so a node needs no LDS, no atomics and no node-state copies, and there is
// room for a much better bound (clique_cover).
#pragma once

#include <type_traits>

namespace vcg {

// largest remainder the search takes (vertices), and the largest when the
// workgroup's LDS has no room for that
constexpr uint32_t kBitsMax = 256u, kBitsMaxSmall = 128u;

__device__ __forceinline__ uint64_t uni64(uint64_t x)
{
    return ((uint64_t)uni((uint32_t)(x >> 32)) << 32) | uni((uint32_t)x);
}

// A wave-uniform mask as a per-lane truth value.
__device__ __forceinline__ bool lane_in(uint64_t mask) { return __builtin_amdgcn_inverse_ballot_w64(mask); }

// Minimum over the 64 lanes: row_shr 1/2/4/8, then row_bcast 15/31; lane 63
// holds the result.
__device__ __forceinline__ uint32_t wave_umin(uint32_t x)
{
    int v = (int)x;
    const int id = -1;  // the identity, for lanes without a source
#define VC_DPP_MIN(ctrl, rows) \
    v = (int)min((uint32_t)v, (uint32_t)__builtin_amdgcn_update_dpp(id, v, ctrl, rows, 0xF, false))
    VC_DPP_MIN(0x111, 0xF);
    VC_DPP_MIN(0x112, 0xF);
    VC_DPP_MIN(0x114, 0xF);
    VC_DPP_MIN(0x118, 0xF);
    VC_DPP_MIN(0x142, 0xA);
    VC_DPP_MIN(0x143, 0xC);
#undef VC_DPP_MIN
    return (uint32_t)__builtin_amdgcn_readlane(v, 63);
}

// Word k of a mask of the first c vertices.
__device__ __forceinline__ uint64_t low_bits(uint32_t c, uint32_t k)
{
    return c >= 64u * k + 64u ? ~0ull : c > 64u * k ? (1ull << (c - 64u * k)) - 1ull : 0ull;
}

template <int K>
struct BitMask {
    uint64_t w[K];
    __device__ __forceinline__ uint32_t half(int j) const { return (uint32_t)(w[j >> 1] >> (32 * (j & 1))); }
    __device__ __forceinline__ bool any() const
    {
        uint64_t x = 0;
#pragma unroll
        for (int k = 0; k < K; ++k) x |= w[k];
        return x != 0;
    }
    __device__ __forceinline__ uint32_t count() const
    {
        uint32_t c = 0;
#pragma unroll
        for (int k = 0; k < K; ++k) c += (uint32_t)__popcll(w[k]);
        return c;
    }
    __device__ __forceinline__ void clear()
    {
#pragma unroll
        for (int k = 0; k < K; ++k) w[k] = 0;
    }
    __device__ __forceinline__ void set(uint32_t i)
    {
#pragma unroll
        for (int k = 0; k < K; ++k)
            if (i / 64u == (uint32_t)k) w[k] |= 1ull << (i & 63u);
    }
    __device__ __forceinline__ void reset(uint32_t i)
    {
#pragma unroll
        for (int k = 0; k < K; ++k)
            if (i / 64u == (uint32_t)k) w[k] &= ~(1ull << (i & 63u));
    }
    __device__ __forceinline__ void drop(const BitMask &o)
    {
#pragma unroll
        for (int k = 0; k < K; ++k) w[k] &= ~o.w[k];
    }
    __device__ __forceinline__ void keep(const BitMask &o)
    {
#pragma unroll
        for (int k = 0; k < K; ++k) w[k] &= o.w[k];
    }
    __device__ __forceinline__ void add(const BitMask &o)
    {
#pragma unroll
        for (int k = 0; k < K; ++k) w[k] |= o.w[k];
    }
    // highest member; the mask is not empty
    __device__ __forceinline__ uint32_t last() const
    {
        uint32_t i = 0;
#pragma unroll
        for (int k = 0; k < K; ++k)
            if (w[k]) i = 64u * k + 63u - (uint32_t)__builtin_clzll(w[k]);
        return i;
    }
    // lowest member; the mask is not empty
    __device__ __forceinline__ uint32_t first() const
    {
        uint32_t i = 0;
#pragma unroll
        for (int k = K - 1; k >= 0; --k)
            if (w[k]) i = 64u * k + (uint32_t)__builtin_ctzll(w[k]);
        return i;
    }
};

// Adjacency rows: r[k][j] = bits 32 j .. 32 j + 31 of the row of vertex
// 64 k + lane.
template <int K>
struct BitRows {
    uint32_t r[K][2 * K];

    // does the lane's vertex of slot k have a neighbour in m?
    __device__ __forceinline__ bool hits(int k, const BitMask<K> &m) const
    {
        uint32_t t = 0;
#pragma unroll
        for (int j = 0; j < 2 * K; ++j) t |= r[k][j] & m.half(j);
        return t != 0;
    }
    __device__ __forceinline__ uint32_t degree(int k, const BitMask<K> &m) const
    {
        uint32_t t = 0;
#pragma unroll
        for (int j = 0; j < 2 * K; ++j) t += (uint32_t)__popc(r[k][j] & m.half(j));
        return t;
    }
    // the row of vertex i (wave-uniform)
    __device__ __forceinline__ BitMask<K> row(uint32_t i) const
    {
        BitMask<K> m;
        const int lane = (int)(i & 63u);
#pragma unroll
        for (int h = 0; h < K; ++h) {
            uint32_t lo = r[0][2 * h], hi = r[0][2 * h + 1];
#pragma unroll
            for (int k = 1; k < K; ++k) {
                // both read before the choice: a choice of addresses would
                // put the rows into memory
                const uint32_t lo_k = r[k][2 * h], hi_k = r[k][2 * h + 1];
                const bool here = i / 64u == (uint32_t)k;
                lo = here ? lo_k : lo;
                hi = here ? hi_k : hi;
            }
            m.w[h] = (uint32_t)__builtin_amdgcn_readlane((int)lo, lane) |
                     ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)hi, lane) << 32);
        }
        return m;
    }
};

// Contexts.  A search runs on a context: the rows of its remainder and the
// vertices' ids.  The vertices of a context are ordered by increasing degree at
// the time it was made, because clique_cover takes them in index order.  As a
// search goes deeper and its remainder shrinks to the next size of ctx_cap,
// it makes a smaller context from the current node (derive): fewer words per
// row, and the order follows the degrees again (with the order of the first
// context alone the searches visit 2-4 times as many nodes as with every
// node's own order, with new ones at 128 and 64 vertices 1.4 times, at the
// sizes below 1.2 times).
//
// A worker holds one context per size in LDS; an entry on its stack names its
// size, and sizes only fall along the stack, so a size's area is free when a
// deeper node needs it.  The cover outside a context is not kept: it follows
// from the masks that led to it (cover_words).  Another worker cannot read
// this worker's LDS, so the first donation from a context copies it, with the
// cover outside it, to the worker's area of that size in HBM (publish).  A
// donated subtree refers to that copy, which counts its users (the owner and
// every donated subtree) and is only overwritten once it has none.  Like a
// worklist slot the copies are written and read with agent-coherent accesses
// only.  (With the contexts themselves in HBM making one cost 20,000 cycles,
// four dependent round trips, and returning to one 6,500.)
constexpr uint32_t kCtxLevels = 6;
// 256 128 96 64 48 32
__host__ __device__ constexpr uint32_t ctx_cap(uint32_t level)
{
    return level == 0u ? 256u : level == 1u ? 128u : level == 2u ? 96u : level == 3u ? 64u : level == 4u ? 48u : 32u;
}
__device__ __forceinline__ uint32_t ctx_level(uint32_t c)
{
    return c > 128u ? 0u : c > 96u ? 1u : c > 64u ? 2u : c > 48u ? 3u : c > 32u ? 4u : 5u;
}
// slots per lane of a level
__device__ __forceinline__ uint32_t ctx_slots(uint32_t level) { return level == 0u ? 4u : level < 3u ? 2u : 1u; }
// LDS per worker: rows of levels 1 to 5 (8 K bytes per vertex) | their ids
// (4 bytes each) | per level a parent mask (32 bytes) | per level (vertices,
// parent level) | 512 bytes of scratch | rows of level 0 | its ids.
// The part before level 0 is what a worker needs with kBitsMaxSmall.  A load
// of 64 K rows may run past its level's rows, into the next level's or the ids;
// those lanes' vertices are in no mask.
constexpr uint32_t kCtxIds = 4736, kCtxMask = kCtxIds + 4u * 368u, kCtxMeta = kCtxMask + 32u * kCtxLevels,
                   kCtxOrder = kCtxMeta + 8u * kCtxLevels, kCtxRows0 = kCtxOrder + 512u, kCtxIds0 = kCtxRows0 + 8192u,
                   kCtxLdsSmall = kCtxRows0, kCtxLdsBytes = kCtxIds0 + 1024u;
static_assert(kCtxLdsBytes % 16u == 0u && kCtxLdsSmall % 16u == 0u, "the node storage after it is 16-byte aligned");
__device__ __forceinline__ uint32_t ctx_rows(uint32_t level)
{
    return level == 0u ? kCtxRows0 : level == 1u ? 0u : level == 2u ? 2048u : level == 3u ? 3584u : level == 4u ? 4096u : 4480u;
}
__device__ __forceinline__ uint32_t ctx_ids(uint32_t level)
{
    return level == 0u ? kCtxIds0
                       : kCtxIds + 4u * (level == 1u ? 0u : level == 2u ? 128u : level == 3u ? 224u : level == 4u ? 288u : 336u);
}
// HBM per worker: user counts (a line) | vertex counts (a line) | the same
// rows and ids | a cover bitmap per level.
constexpr uint32_t kHbmCount = 64, kHbmBase = 128, kHbmCover = (kHbmBase + kCtxLdsBytes + 63u) / 64u * 64u;
__device__ __forceinline__ uint32_t ctx_cover(const SolveArgs &a, uint32_t level)
{
    return kHbmCover + level * ((a.ctx_bytes - kHbmCover) / kCtxLevels);
}
// a published context's name: worker * kCtxLevels + level
__device__ __forceinline__ __amdgpu_buffer_rsrc_t ctx_rsrc(const SolveArgs &a, uint32_t ctx)
{
    return slot_rsrc(a.ctx + (size_t)(ctx / kCtxLevels) * a.ctx_bytes, a.ctx_bytes);
}
__device__ __forceinline__ uint32_t *ctx_users(const SolveArgs &a, uint32_t ctx)
{
    return reinterpret_cast<uint32_t *>(a.ctx + (size_t)(ctx / kCtxLevels) * a.ctx_bytes) + ctx % kCtxLevels;
}

// One worker's contexts in LDS.
struct BitsLds {
    char *base;
    __device__ __forceinline__ char *row(uint32_t level, uint32_t i) const
    {
        return base + ctx_rows(level) + i * (8u * ctx_slots(level));
    }
    __device__ __forceinline__ uint32_t &id(uint32_t level, uint32_t i) const
    {
        return reinterpret_cast<uint32_t *>(base + ctx_ids(level))[i];
    }
    // vertices of the parent context that were not in the cover when the
    // level's context was made
    __device__ __forceinline__ uint64_t &parent_mask(uint32_t level, uint32_t k) const
    {
        return reinterpret_cast<uint64_t *>(base + kCtxMask)[4u * level + k];
    }
    // a search of a whole graph: what its first reductions put in the cover
    // (level 0 has no parent)
    __device__ __forceinline__ uint64_t &root_cover(uint32_t k) const { return parent_mask(0u, k); }
    __device__ __forceinline__ uint32_t &count(uint32_t level) const
    {
        return reinterpret_cast<uint32_t *>(base + kCtxMeta)[2u * level];
    }
    __device__ __forceinline__ uint32_t &parent(uint32_t level) const  // kNone: the search's first context
    {
        return reinterpret_cast<uint32_t *>(base + kCtxMeta)[2u * level + 1u];
    }
    // scratch, a byte per vertex each
    __device__ __forceinline__ uint8_t *order() const { return reinterpret_cast<uint8_t *>(base + kCtxOrder); }
    __device__ __forceinline__ uint8_t *claim() const { return reinterpret_cast<uint8_t *>(base + kCtxOrder + 256u); }
};

template <int K>
__device__ __forceinline__ void load_rows(const BitsLds &lds, uint32_t level, BitRows<K> &rows)
{
    const char *const p = lds.base + ctx_rows(level);
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const char *const q = p + (64u * k + lane_id()) * (8u * K);
        if constexpr (K == 1) {
            const uint2 x = *reinterpret_cast<const uint2 *>(q);
            rows.r[k][0] = x.x;
            rows.r[k][1] = x.y;
        } else {
#pragma unroll
            for (int j = 0; j < 2 * K; j += 4) {
                const uint4 x = *reinterpret_cast<const uint4 *>(q + 4 * j);
                rows.r[k][j] = x.x;
                rows.r[k][j + 1] = x.y;
                rows.r[k][j + 2] = x.z;
                rows.r[k][j + 3] = x.w;
            }
        }
    }
}

// The remainder of the node in w (nq live vertices) into the LDS context of
// `level`, in id order.  Positions of live vertices go to bytes over w.s2, which
// the subtree does not use (of the node's state only the degrees' signs are read
// again, for covers).
template <int K, class N>
__device__ __forceinline__ void build_rows(const N &w, const BitsLds &lds, uint32_t level, uint32_t nq)
{
    uint8_t *const pos = reinterpret_cast<uint8_t *>(w.s2);
    uint32_t c = 0;
    w.sync();
    for (uint32_t base = 0, nv = uni(w.n); base < nv; base += kWave) {
        const uint32_t v = base + lane_id();
        const bool live = deg_or_none(w, v, nv) > 0;
        const uint64_t m = __ballot(live);
        if (live) {
            const uint32_t p = c + lanes_below(m);
            lds.id(level, p) = v;
            pos[v] = (uint8_t)p;
        }
        c = uni(c + (uint32_t)__popcll(m));
    }
    w.sync();
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const uint32_t i = 64u * k + lane_id();
        if (64u * k >= nq) break;
        uint32_t r[2 * K];
#pragma unroll
        for (int j = 0; j < 2 * K; ++j) r[j] = 0;
        uint32_t x = 0, e = 0;
        if (i < nq) {
            const uint32_t v = lds.id(level, i);
            x = w.off(v);
            e = w.off(v + 1u);
        }
        // eight neighbours in flight
        for (; x < e; x += 8u) {
            uint32_t t[8];
#pragma unroll
            for (uint32_t q = 0; q < 8u; ++q) t[q] = w.nb(min(x + q, e - 1u));
#pragma unroll
            for (uint32_t q = 0; q < 8u; ++q) {
                // a repeated last neighbour sets its bit again
                if (w.deg(t[q]) > 0) {
                    const uint32_t p = pos[t[q]];
                    const uint32_t bit = 1u << (p & 31u);
#pragma unroll
                    for (int j = 0; j < 2 * K; ++j) r[j] |= (p >> 5) == (uint32_t)j ? bit : 0u;
                }
            }
        }
        if (i < nq)
#pragma unroll
            for (int j = 0; j < 2 * K; ++j) reinterpret_cast<uint32_t *>(lds.row(level, i))[j] = r[j];
    }
    if (lane_id() == 0) {
        lds.count(level) = nq;
        lds.parent(level) = kNone;
    }
    w.sync();
}

// The whole graph in w (at most 64 K vertices) as the LDS context of `level`.
template <int K, class N>
__device__ __forceinline__ void build_whole(const N &w, const BitsLds &lds, uint32_t level)
{
    const uint32_t n = uni(w.n);
#pragma unroll
    for (int k = 0; k < K; ++k) {
        if (64u * k >= n) break;
        const uint32_t i = 64u * k + lane_id();
        uint32_t r[2 * K];
#pragma unroll
        for (int j = 0; j < 2 * K; ++j) r[j] = 0;
        uint32_t x = 0, e = 0;
        if (i < n) {
            x = w.off(i);
            e = w.off(i + 1u);
        }
        // eight neighbours in flight
        for (; x < e; x += 8u) {
            uint32_t t[8];
#pragma unroll
            for (uint32_t q = 0; q < 8u; ++q) t[q] = w.nb(min(x + q, e - 1u));
#pragma unroll
            for (uint32_t q = 0; q < 8u; ++q) {
                const uint32_t bit = 1u << (t[q] & 31u);
#pragma unroll
                for (int j = 0; j < 2 * K; ++j) r[j] |= (t[q] >> 5) == (uint32_t)j ? bit : 0u;
            }
        }
        if (i < n) {
            lds.id(level, i) = i;
#pragma unroll
            for (int j = 0; j < 2 * K; ++j) reinterpret_cast<uint32_t *>(lds.row(level, i))[j] = r[j];
        }
    }
    if (lane_id() == 0) {
        lds.count(level) = n;
        lds.parent(level) = kNone;
#pragma unroll
        for (uint32_t k = 0; k < 4u; ++k) lds.root_cover(k) = 0ull;
    }
    nsync<false>();
}

// Makes the context of level `to` for a node of level `from`: its nq vertices
// with a live edge in order of increasing degree (deg: the node's degrees),
// ties in the old order.  `first`: the new context replaces `from` as the
// search's first one (what the node has covered is kept in root_cover);
// otherwise to == from sorts a context whose vertices are all in the node.  One row (2 K readlanes) per vertex of the new context, no memory
// access but LDS.
template <int K>
__device__ __forceinline__ void derive(const BitsLds &lds, const BitRows<K> &rows, const BitMask<K> &live,
                                       const uint32_t (&deg)[K], uint32_t nq, uint32_t from, uint32_t to, bool first)
{
    const uint32_t lane = lane_id(), slots = ctx_slots(to);
    // rank of every vertex: degree by degree, in index order
    uint32_t rank[K], ids[K];
    BitMask<K> left;
#pragma unroll
    for (int k = 0; k < K; ++k) {
        left.w[k] = __ballot(deg[k] != 0u);
        rank[k] = kNone;
        ids[k] = 64u * k + lane < ctx_cap(K == 4 ? 0u : K == 2 ? 1u : 3u) ? lds.id(from, 64u * k + lane) : 0u;
    }
    uint32_t next = 0;
    while (next < nq) {
        uint32_t x = kNone;
#pragma unroll
        for (int k = 0; k < K; ++k) x = min(x, lane_in(left.w[k]) ? deg[k] : kNone);
        x = wave_umin(x);
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const uint64_t m = __ballot(deg[k] == x);
            if (deg[k] == x) rank[k] = next + lanes_below(m);
            next = uni(next + (uint32_t)__popcll(m));
            left.w[k] &= ~m;
        }
    }
    // order[r] = the old index of the vertex of rank r
    uint8_t *const order = lds.order();
    nsync<false>();
#pragma unroll
    for (int k = 0; k < K; ++k)
        if (rank[k] != kNone) {
            order[rank[k]] = (uint8_t)(64u * k + lane);
            lds.id(to, rank[k]) = ids[k];
        }
    if (lane == 0 && (first || to != from)) {
        lds.count(to) = nq;
        lds.parent(to) = first ? kNone : from;
    }
    if (lane == 0 && !first && to != from) {
#pragma unroll
        for (int k = 0; k < K; ++k) lds.parent_mask(to, k) = live.w[k];
    }
    nsync<false>();
    // column j of the new rows = the old row of order[j], seen from every
    // old vertex; each vertex then stores its new row at its rank
#pragma unroll
    for (int j = 0; j < 2 * K; ++j) {
        if (32u * j >= nq) break;
        const uint32_t mine = order[32u * j + (lane & 31u)];
        uint32_t acc[K];
#pragma unroll
        for (int k = 0; k < K; ++k) acc[k] = 0;
        const uint32_t cols = min(32u, nq - 32u * j);
        for (uint32_t q = 0; q < cols; ++q) {
            const BitMask<K> m = rows.row((uint32_t)__builtin_amdgcn_readlane((int)mine, (int)q));
#pragma unroll
            for (int k = 0; k < K; ++k) acc[k] |= lane_in(m.w[k]) ? 1u << q : 0u;
        }
#pragma unroll
        for (int k = 0; k < K; ++k)
            if (rank[k] != kNone) reinterpret_cast<uint32_t *>(lds.row(to, rank[k]))[j] = acc[k];
    }
    // words past the last column
    for (uint32_t j = (nq + 31u) / 32u; j < 2u * slots; ++j)
#pragma unroll
        for (int k = 0; k < K; ++k)
            if (rank[k] != kNone) reinterpret_cast<uint32_t *>(lds.row(to, rank[k]))[j] = 0u;
    nsync<false>();
}

// Greedy clique cover of the nq vertices in q.  A clique of s vertices needs
// s - 1 of them in any cover, so the cover grows by at least lb = nq - cliques.
// Ends early (returns true) once lb > room, the most vertices the cover may
// still take.
//
// In order of the vertices: each clique starts at the first unassigned vertex
// and takes the first common neighbour of its members until none is left.
// That is one vertex after the other, some 200 cycles each (a row by
// readlanes, then scalar instructions, no memory access).  In a sparse
// remainder most of it is done by kRounds rounds for all lanes at once first:
// vertices that are each other's first unassigned neighbour become a pair, and
// each pair takes its first unassigned common neighbour (of several pairs that
// want the same vertex one gets it).  Three rounds leave 14-23% of a sparse
// remainder for the serial part and the searches visit as many nodes as
// without them; dense remainders, whose cliques are larger, take the serial
// part alone (with rounds the searches visit a fifth more nodes at half of all
// edges).
//
// When lb <= room: any cover of at most `room` more vertices leaves at least
// nq - room vertices out, no two in one clique, and nq - lb - r cliques with
// r = room - lb + 1 can hold only nq - room - 1 of them; so among the other r
// cliques at least one vertex stays out.  `branch` receives, in a sparse
// remainder, the vertices of r cliques, singletons first, then pairs, when
// these are at most kFewBranch vertices, and is left empty otherwise.  One such
// vertex: it stays out, its neighbours are in, nothing is left to branch on.
// In a dense remainder it receives all that the first nq - room - 1 cliques
// leave over, and the cover ends there: the cliques are large, so many children
// of one node (each much smaller than the node) replace a chain of nodes that
// each take one vertex and make the cover again.  At a density of a half and
// above that halves the nodes of a search (three graphs of n = 225..250: 11.8
// -> 8.2 ms); sparse remainders leave so much over that the search grows by
// two thirds (n = 140, mean degree 6: 1,161 -> 1,924 nodes).
constexpr uint32_t kRounds = 3;
constexpr uint32_t kSerialOnly = 16;  // a rest this small is left to the serial part
constexpr uint32_t kFewBranch = 4;

// The first vertex of p (not empty): off q, and p keeps its neighbours.  One
// uniform branch per slot instead of selects: the slot's registers and mask
// words are then known.
template <int K>
__device__ __forceinline__ uint32_t take_first(const BitRows<K> &rows, BitMask<K> &p, BitMask<K> &q)
{
    uint32_t i = 0;
    auto at = [&](auto slot) {
        constexpr int k = decltype(slot)::value;
        const int lane = (int)__builtin_ctzll(p.w[k]);
        i = 64u * k + (uint32_t)lane;
        q.w[k] &= ~(1ull << lane);
#pragma unroll
        for (int h = 0; h < K; ++h)
            p.w[h] &= (uint32_t)__builtin_amdgcn_readlane((int)rows.r[k][2 * h], lane) |
                      ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)rows.r[k][2 * h + 1], lane) << 32);
    };
    if constexpr (K == 1) {
        at(std::integral_constant<int, 0>{});
    } else if constexpr (K == 2) {
        if (p.w[0])
            at(std::integral_constant<int, 0>{});
        else
            at(std::integral_constant<int, 1>{});
    } else {
        if (p.w[0])
            at(std::integral_constant<int, 0>{});
        else if (p.w[1])
            at(std::integral_constant<int, 1>{});
        else if (p.w[2])
            at(std::integral_constant<int, 2>{});
        else
            at(std::integral_constant<int, 3>{});
    }
    return i;
}

template <int K>
__device__ __forceinline__ bool clique_cover(const BitsLds &lds, const char *my_rows, const BitRows<K> &rows, BitMask<K> q,
                                             uint32_t nq, uint32_t room, bool sparse, BitMask<K> &branch, uint32_t &nbranch)
{
    const uint32_t lane = lane_id();
    BitMask<K> one, pair_a, pair_b;  // singletons, the serial part's last two pairs
    BitMask<K> leads;                // first vertices of the rounds' pairs
    uint32_t mate[K];                // of those
    one.clear();
    pair_a.clear();
    pair_b.clear();
    leads.clear();
    uint32_t lb = 0, left = nq, pairs = 0;
    branch.clear();
    nbranch = 0;
#pragma unroll
    for (int k = 0; k < K; ++k) mate[k] = 0;
    if (sparse) {
        uint8_t *const wants = lds.order(), *const claim = lds.claim();
        for (uint32_t round = 0; round < kRounds && left > kSerialOnly; ++round) {
            if (lb + left + kFewBranch <= room) return false;
            uint32_t first[K], third[K];
#pragma unroll
            for (int k = 0; k < K; ++k) {
                const uint32_t v = 64u * k + lane;
                uint32_t p = kNone;
#pragma unroll
                for (int j = 2 * K - 1; j >= 0; --j) {
                    const uint32_t x = rows.r[k][j] & q.half(j);
                    if (x) p = 32u * j + (uint32_t)__builtin_ctz(x);
                }
                first[k] = lane_in(q.w[k]) ? p : kNone;
                if (lane_in(q.w[k])) {
                    wants[v] = (uint8_t)(p != kNone ? p : v);
                    claim[v] = 255u;  // (no pair's first vertex)
                }
            }
            nsync<false>();
            BitMask<K> paired, lead;
#pragma unroll
            for (int k = 0; k < K; ++k) {
                const uint32_t v = 64u * k + lane, p = first[k];
                const bool mutual = (p != kNone) & (wants[p != kNone ? p : 0u] == v);
                paired.w[k] = __ballot(mutual);
                lead.w[k] = __ballot(mutual & (v < p));
            }
            if (!paired.any()) break;
            q.drop(paired);
            const uint32_t made = lead.count();
            left -= 2u * made;
            lb += made;
            // each pair's first unassigned common neighbour
#pragma unroll
            for (int k = 0; k < K; ++k) {
                third[k] = kNone;
                const uint32_t p = lane_in(lead.w[k]) ? first[k] : 0u;
                const uint32_t *const other = reinterpret_cast<const uint32_t *>(my_rows + p * (8u * K));
#pragma unroll
                for (int j = 2 * K - 1; j >= 0; --j) {
                    const uint32_t x = rows.r[k][j] & other[j] & q.half(j);
                    if (x) third[k] = 32u * j + (uint32_t)__builtin_ctz(x);
                }
                if (!lane_in(lead.w[k])) third[k] = kNone;
                if (third[k] != kNone) claim[third[k]] = (uint8_t)(64u * k + lane);
            }
            nsync<false>();
            BitMask<K> joined;
#pragma unroll
            for (int k = 0; k < K; ++k) {
                const uint32_t v = 64u * k + lane;
                joined.w[k] = __ballot(claim[v] != 255u) & q.w[k];
                const bool got = (third[k] != kNone) & (claim[third[k] != kNone ? third[k] : 0u] == v);
                const uint64_t alone = lead.w[k] & ~__ballot(got);
                leads.w[k] |= alone;
                if (lane_in(alone)) mate[k] = first[k];
            }
            nsync<false>();
            q.drop(joined);
            const uint32_t more = joined.count();
            left -= more;
            lb += more;
            if (lb > room) return true;
        }
        pairs = leads.count();
    }
    const int stop = sparse ? (int)room - (int)kFewBranch : (int)room + 1;
    while (left) {
        if ((int)(lb + left) <= stop) {
            // sparse: even one clique of all that is left leaves more than
            // kFewBranch cliques to branch in; dense: nq - room - 1 cliques
            // are made (or any nq vertices may be covered: no branch set)
            if (!sparse && nq > room) {
                branch = q;
                nbranch = left;
            }
            return false;
        }
        BitMask<K> p = q;
        const uint32_t v = take_first<K>(rows, p, q);
        uint32_t size = 1, last = v;
        while (p.any()) {
            last = take_first<K>(rows, p, q);
            ++size;
        }
        left -= size;
        lb += size - 1u;
        if (lb > room) return true;
        if (size == 1u) {
            one.set(v);
        } else if (size == 2u) {
            ++pairs;
            pair_b = pair_a;
            pair_a.clear();
            pair_a.set(v);
            pair_a.set(last);
        }
    }
    const uint32_t r = room - lb + 1u, cliques = nq - lb, singles = one.count();
    if (r >= cliques) return false;
    if (r <= singles) {
        if (r > kFewBranch) return false;
        // the last r singletons (of the highest degrees)
        for (uint32_t i = 0; i < r; ++i) {
            const uint32_t v = one.last();
            one.reset(v);
            branch.set(v);
        }
        nbranch = r;
    } else {
        const uint32_t two = r - singles;
        if (two > pairs || two > 2u || singles + 2u * two > kFewBranch) return false;
        branch = one;
        for (uint32_t i = 0; i < two; ++i) {
            // the serial part's pairs first, then the rounds'
            if (i == 0u && pair_a.any()) {
                branch.add(pair_a);
            } else if (i == 1u && pair_b.any()) {
                branch.add(pair_b);
            } else {
                const uint32_t v = leads.last();
                leads.reset(v);
                uint32_t u = 0;
#pragma unroll
                for (int k = 0; k < K; ++k) {
                    const uint32_t mate_k = (uint32_t)__builtin_amdgcn_readlane((int)mate[k], (int)(v & 63u));
                    u = v / 64u == (uint32_t)k ? mate_k : u;
                }
                branch.set(v);
                branch.set(u);
            }
        }
        nbranch = singles + 2u * two;
    }
    return false;
}

// One worker's bitset search: what it shares with the main loop, and the node
// it is at.
struct BitsWorker {
    char *stk;           // the worker's stack: a bitset entry takes one slot
    uint2 *stk_meta;     // (d, level) of a bitset entry
    uint32_t slot_bytes, wid;
    int top, bot;
    uint64_t pending, total_nodes, donations;
    uint32_t moved, flush_every;
    int base;            // stack entries above this one are the search's own
    uint32_t d;          // cover size of the node
    uint32_t level;      // its context's level
    uint32_t home;       // the published context the search started from, or kNone (the node in w)
    uint32_t fresh;      // 1 = the first context is in id order (just built)
    uint32_t published;  // levels whose context has a valid copy in HBM, held by this search
    uint32_t whole;      // 1 = the first context is the graph itself
    uint32_t since, want; // branches since the last donation, items missing at the next
    uint32_t rnd;        // random state (next_random)
    uint32_t best;       // the search looks for covers smaller than this
    uint64_t live[4], settled[4];  // the node's masks (K words each)
};

// Every control value of the search is wave-uniform.  The compiler loses sight
// of that where it merges values behind a branch on the lane number, and then
// keeps masks in vector registers and runs loops under exec masks; so they
// are made uniform again at every node (no instruction where they are).
__device__ __forceinline__ void make_uniform(BitsWorker &b)
{
    b.top = (int)uni((uint32_t)b.top);
    b.bot = (int)uni((uint32_t)b.bot);
    b.base = (int)uni((uint32_t)b.base);
    b.pending = uni64(b.pending);
    b.total_nodes = uni64(b.total_nodes);
    b.donations = uni64(b.donations);
    b.moved = uni(b.moved);
    b.flush_every = uni(b.flush_every);
    b.level = uni(b.level);
    b.home = uni(b.home);
    b.fresh = uni(b.fresh);
    b.published = uni(b.published);
    b.whole = uni(b.whole);
    b.since = uni(b.since);
    b.want = uni(b.want);
    b.rnd = uni(b.rnd);
    b.best = uni(b.best);
}

// Word i of a bitset entry's masks (live, then settled) in lane i into b.
__device__ __forceinline__ void unpack_masks(BitsWorker &b, uint32_t x)
{
    const uint32_t slots = ctx_slots(b.level);
#pragma unroll
    for (uint32_t k = 0; k < 4u; ++k) {
        b.live[k] = b.settled[k] = 0ull;
        if (k < slots) {
            b.live[k] = (uint32_t)__builtin_amdgcn_readlane((int)x, (int)(2u * k)) |
                        ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)x, (int)(2u * k + 1u)) << 32);
            b.settled[k] = (uint32_t)__builtin_amdgcn_readlane((int)x, (int)(2u * slots + 2u * k)) |
                           ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)x, (int)(2u * slots + 2u * k + 1u)) << 32);
        }
    }
}

// A search donates at its first branch, then whenever it has a full batch
// or this many branches after the last time: 1, 2 and 4 take 1.55, 1.47 and
// 1.55 ms for four 3-regular graphs of n = 108..120.
constexpr uint32_t kDonateEvery = 2;

// What bit_level asks its caller for.
enum BitsNext : uint32_t {
    kBitsDone,    // the search has ended (or was stopped: the stack is empty)
    kBitsNode,    // go on with the node in b, at b.level
    kBitsDonate,  // donate the oldest entry, then go on with the node in b
    kBitsCover,   // the node in b is a cover of size b.d: record it, then pop
};

// Searches at one context, from the node in b or, with `pop`, from the stack's
// top entry, until it ends, goes on at another level or needs something off
// the common path (which is kept out of here: the loop should stay small
// enough for the instruction cache).
template <int K, bool STAGED>
__device__ __forceinline__ uint32_t bit_level(const SolveArgs &a, const BitsLds &lds, const GDesc &gd, uint32_t g,
                                              BitsWorker &b, bool pop)
{
    GState *const gs = &a.gstate[g];
    const bool mvc = uni(gd.instance) == 0u;
    const uint32_t lane = lane_id();
    make_uniform(b);
    BitRows<K> rows;
    BitMask<K> live, settled;  // settled: degree-2 vertices whose neighbours are not adjacent
    uint32_t d = uni(b.d);
#pragma unroll
    for (int k = 0; k < K; ++k) {
        live.w[k] = uni64(b.live[k]);
        settled.w[k] = uni64(b.settled[k]);
    }
    load_rows<K>(lds, b.level, rows);
    const char *const my_rows = lds.base + ctx_rows(b.level);
    auto leave = [&](uint32_t what) {
        b.d = d;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            b.live[k] = live.w[k];
            b.settled[k] = settled.w[k];
        }
        return what;
    };

    bool dead = pop;
    for (;;) {
        make_uniform(b);
        if (uni(dead ? 1u : 0u)) {
            // the search's next entry
            if (b.top <= b.base || b.top < b.bot) return kBitsDone;
            const uint32_t ts = (uint32_t)b.top % a.depth;
            const uint2 m = b.stk_meta[ts];
            uint32_t x = 0;
            if (lane < 16u) x = reinterpret_cast<const uint32_t *>(b.stk + (size_t)ts * b.slot_bytes)[lane];
            --b.top;
            b.moved += 16u * K;
            d = uni(m.x);
            const uint32_t level = uni(m.y);
            if (level != b.level) {
                b.level = level;
                b.d = d;
                unpack_masks(b, x);
                return kBitsNode;
            }
#pragma unroll
            for (int k = 0; k < K; ++k) {
                live.w[k] = (uint32_t)__builtin_amdgcn_readlane((int)x, 2 * k) |
                            ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)x, 2 * k + 1) << 32);
                settled.w[k] = (uint32_t)__builtin_amdgcn_readlane((int)x, 2 * K + 2 * k) |
                               ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)x, 2 * K + 2 * k + 1) << 32);
            }
        }
        // one node: (live, settled, d)
        d = uni(d);
#pragma unroll
        for (int k = 0; k < K; ++k) {
            live.w[k] = uni64(live.w[k]);
            settled.w[k] = uni64(settled.w[k]);
        }
        // the stop flag and the incumbent, and the launch's counter, are read
        // at the node's start and used at its end, so the node does not wait
        // for them
        const unsigned long long state_next = ld_rlx(reinterpret_cast<unsigned long long *>(&gs->best));
        unsigned long long counter_next = 0;
        if (a.version == 1u) counter_next = ld_rlx(&a.glob->counter);
        if (++b.pending >= b.flush_every) {
            b.total_nodes += b.pending;
            flush_nodes<STAGED>(a, gd, g, b.pending, b.moved, b.flush_every, false);
            uint32_t stop_all = 0;
            if (lane == 0) stop_all = ld_rlx(&a.glob->cancel) || past_deadline(a);
            if (uni(stop_all)) {
                b.top = -1;
                b.bot = 0;
                return kBitsDone;
            }
        }
        const uint32_t T = b.best;
        uint32_t deg[K];
        dead = false;
        for (;;) {
            // rule fixpoint (reduce_node's rules on masks)
            if (d >= T) {
                dead = true;
                break;
            }
            BitMask<K> m, take;
#pragma unroll
            for (int k = 0; k < K; ++k) {
                const uint32_t x = rows.degree(k, live);
                deg[k] = lane_in(live.w[k]) ? x : 0u;
                m.w[k] = __ballot(deg[k] == 1u);
            }
            if (m.any()) {
                // leaf rule: every live vertex with a leaf neighbour, of an
                // isolated edge only the lower end
#pragma unroll
                for (int k = 0; k < K; ++k) {
                    uint32_t t = 0;
#pragma unroll
                    for (int j = 2 * k; j < 2 * K; ++j) {
                        uint32_t x = rows.r[k][j] & m.half(j);
                        if (j == 2 * k) x &= lane < 32u ? ~((2u << lane) - 1u) : 0u;
                        if (j == 2 * k + 1) x &= lane < 32u ? ~0u : ~((2u << (lane - 32u)) - 1u);
                        t |= x;  // leaf neighbours above this vertex
                    }
                    const bool in = lane_in(live.w[k]) & (deg[k] == 1u ? t != 0u : rows.hits(k, m));
                    take.w[k] = __ballot(in);
                }
            } else {
#pragma unroll
                for (int k = 0; k < K; ++k) m.w[k] = __ballot(deg[k] == 2u) & ~settled.w[k];
                take.clear();
                if (m.any()) {
                    // triangle rule, every unexamined degree-2 vertex in its
                    // lane: are its two neighbours lo < hi adjacent (one word
                    // of lo's row, from LDS)?  Of adjacent vertices that fire
                    // the lowest does.
                    BitMask<K> fires;
#pragma unroll
                    for (int k = 0; k < K; ++k) {
                        uint32_t lo = 0, hi = 0;
#pragma unroll
                        for (int j = 2 * K - 1; j >= 0; --j) {
                            const uint32_t x = rows.r[k][j] & live.half(j);
                            if (x) lo = 32u * j + (uint32_t)__builtin_ctz(x);
                        }
#pragma unroll
                        for (int j = 0; j < 2 * K; ++j) {
                            const uint32_t x = rows.r[k][j] & live.half(j);
                            if (x) hi = 32u * j + 31u - (uint32_t)__builtin_clz(x);
                        }
                        const uint32_t word = reinterpret_cast<const uint32_t *>(my_rows + lo * (8u * K))[hi >> 5];
                        fires.w[k] = __ballot((word >> (hi & 31u)) & 1u) & m.w[k];
                        settled.w[k] |= m.w[k] & ~fires.w[k];
                    }
                    if (fires.any()) {
                        BitMask<K> first;
#pragma unroll
                        for (int k = 0; k < K; ++k) {
                            uint32_t t = 0;
#pragma unroll
                            for (int j = 0; j <= 2 * k + 1; ++j) {
                                uint32_t x = rows.r[k][j] & fires.half(j);
                                if (j == 2 * k) x &= lane < 32u ? (1u << lane) - 1u : ~0u;
                                if (j == 2 * k + 1) x &= lane < 32u ? 0u : (1u << (lane - 32u)) - 1u;
                                t |= x;  // neighbours below this vertex that fire
                            }
                            first.w[k] = __ballot(t == 0u) & fires.w[k];
                        }
#pragma unroll
                        for (int k = 0; k < K; ++k) take.w[k] = __ballot(lane_in(live.w[k]) & rows.hits(k, first));
                    }
                }
                if (!take.any()) {
                    // high-degree rule
                    const uint32_t need = T - d;
#pragma unroll
                    for (int k = 0; k < K; ++k) take.w[k] = __ballot(deg[k] >= need);
                }
            }
            if (!take.any()) break;
            live.drop(take);
            d += take.count();
        }
        BitMask<K> branch;
        uint32_t nbranch = 0;
        if (!dead) {
            // degree levels: x = 1, 2, ...: vertices of degree >= x
            const uint32_t room = T - 1u - d;
            uint32_t e2 = 0, cap = 0, nq = 0, md = 0;
            constexpr uint32_t kLevels = 24;
            for (uint32_t x = 1; x <= kLevels; ++x) {
                uint32_t cnt = 0;
#pragma unroll
                for (int k = 0; k < K; ++k) cnt += (uint32_t)__popcll(__ballot(deg[k] >= x));
                if (cnt == 0u) break;
                if (x == 1u) nq = cnt;
                md = x;
                e2 += cnt;
                cap += min(cnt, room);
            }
            if (md == kLevels) {
                // dense: maximum and sum over the lanes, `room` vertices of
                // maximum degree
                uint32_t s = 0, x = 0;
#pragma unroll
                for (int k = 0; k < K; ++k) {
                    s += deg[k];
                    x = max(x, deg[k]);
                }
                md = ~wave_umin(~x);
                e2 = (uint32_t)wave_sum((int)s);
                cap = room * md;
            }
            if (nq == 0u) return leave(kBitsCover);  // every live vertex is isolated: a cover of size d < T
            BitMask<K> q;
#pragma unroll
            for (int k = 0; k < K; ++k) q.w[k] = __ballot(deg[k] != 0u);
            if (e2 > 2u * cap) {
                // `room` vertices cannot cover the edges, whichever they are
                dead = true;
            } else if (md <= 2u) {
                // cycles only: some minimum cover holds any one vertex
                live.reset(q.first());
                d += 1u;
            } else {
                const uint32_t level = ctx_level(nq);
                const bool first = b.fresh != 0u && b.whole != 0u;
                const bool sort = b.fresh != 0u && level == b.level &&
                                  (first || (nq == live.count() && nq == uni(lds.count(b.level))));
                if (level > b.level || sort) {
                    // the remainder fits a smaller context (or its context is
                    // in id order still): go on there; the node is not
                    // counted twice
                    if (first && lane == 0) {
                        const uint32_t all = lds.count(b.level);
#pragma unroll
                        for (int k = 0; k < K; ++k) lds.root_cover(k) = low_bits(all, k) & ~live.w[k];
                    }
                    derive<K>(lds, rows, live, deg, nq, b.level, level, first);
                    if ((b.published >> level) & 1u) {
                        // the copy in HBM was of the old context
                        if (lane == 0) fetch_add(ctx_users(a, b.wid * kCtxLevels + level), 0xFFFFFFFFu);
                        b.published &= ~(1u << level);
                    }
                    b.level = level;
                    b.d = d;
                    b.pending -= 1u;
                    b.fresh = 0u;
#pragma unroll
                    for (uint32_t k = 0; k < 4u; ++k) {
                        b.live[k] = low_bits(nq, k);
                        b.settled[k] = 0ull;
                    }
                    return kBitsNode;
                }
                dead = clique_cover<K>(lds, my_rows, rows, q, nq, room, 4u * e2 <= nq * nq, branch, nbranch);
                if (!dead) {
                    // children: stack all but the last
                    auto push = [&](const BitMask<K> &m, uint32_t dm) {
                        if (dm >= T) return;
                        ++b.top;
                        const uint32_t ts = (uint32_t)b.top % a.depth;
                        uint32_t x = 0;
#pragma unroll
                        for (int k = 0; k < K; ++k) {
                            x = lane_in(1ull << (2 * k)) ? (uint32_t)m.w[k] : x;
                            x = lane_in(1ull << (2 * k + 1)) ? (uint32_t)(m.w[k] >> 32) : x;
                            x = lane_in(1ull << (2 * K + 2 * k)) ? (uint32_t)settled.w[k] : x;
                            x = lane_in(1ull << (2 * K + 2 * k + 1)) ? (uint32_t)(settled.w[k] >> 32) : x;
                        }
                        if (lane < 4u * K) reinterpret_cast<uint32_t *>(b.stk + (size_t)ts * b.slot_bytes)[lane] = x;
                        if (lane == 0) b.stk_meta[ts] = make_uint2(dm, b.level);
                        b.moved += 16u * K;
                    };
                    if (nbranch == 0u) {
                        // the first vertex of maximum degree: its neighbours
                        // in, then itself in
                        uint32_t v = 0;
#pragma unroll
                        for (int k = K - 1; k >= 0; --k) {
                            const uint64_t top_k = __ballot(deg[k] == md);
                            if (top_k) v = 64u * k + (uint32_t)__builtin_ctzll(top_k);
                        }
                        BitMask<K> r = live;
                        r.drop(rows.row(v));
                        push(r, d + md);
                        live.reset(v);
                        d += 1u;
                    } else {
                        // one of the branch vertices stays out: the i-th child
                        // covers the ones before it and the i-th's neighbours
                        for (uint32_t i = 0; i < nbranch; ++i) {
                            const uint32_t u = branch.last();
                            branch.reset(u);
                            BitMask<K> r = live, m = rows.row(u);
                            m.keep(live);
                            r.drop(m);
                            const uint32_t dm = d + m.count();
                            if (i + 1u == nbranch) {
                                live = r;
                                d = dm;
                            } else {
                                push(r, dm);
                                live.reset(u);
                                d += 1u;
                            }
                        }
                    }
                    ++b.since;
                    if (a.version == 1u && b.top >= b.bot &&
                        (b.since >= kDonateEvery || b.top - b.bot + 1 >= (int)kDonateBatch)) {
                        b.want = wants_donation<true>(a, counter_next, b.rnd);
                        if (b.want != 0u && uni((uint32_t)(state_next >> 32)) == 0u) return leave(kBitsDonate);
                    }
                }
            }
        }
        if (uni((uint32_t)(state_next >> 32))) {
            b.top = -1;
            b.bot = 0;
            return kBitsDone;
        }
        if (mvc) b.best = min(b.best, uni((uint32_t)state_next));
    }
}

// The cover of a node of the search, one bitmap word after the other to
// put(i, word): at its level the vertices missing from `live` (kNone: none),
// at the levels above those missing from the mask that led down, and the cover
// outside the first context (the home context's copy, root_cover, or the node
// in w).
// w.mark (all zero between passes) holds the search's part while it is built.
template <class N, class F>
__device__ __forceinline__ void cover_words(const SolveArgs &a, const N &w, const BitsLds &lds, uint32_t home, bool whole, uint32_t n,
                                            uint32_t level, const uint64_t *live, F &&put)
{
    const uint32_t words = ((n + 63u) / 64u) * 2u;
    w.sync();
    uint64_t m[4] = {~0ull, ~0ull, ~0ull, ~0ull};
    if (live)
        for (uint32_t k = 0; k < 4u; ++k) m[k] = live[k];
    for (;;) {
        const uint32_t c = uni(lds.count(level));
#pragma unroll
        for (uint32_t k = 0; k < 4u; ++k) {
            const uint32_t i = 64u * k + lane_id();
            if (i < c && !((m[k] >> lane_id()) & 1ull)) {
                const uint32_t v = lds.id(level, i);
                __hip_atomic_fetch_or(&w.mark[v >> 5], 1u << (v & 31u), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
            }
        }
        const uint32_t up = uni(lds.parent(level));
        if (up == kNone) break;
        const uint32_t slots = ctx_slots(up);
#pragma unroll
        for (uint32_t k = 0; k < 4u; ++k) m[k] = k < slots ? lds.parent_mask(level, k) : 0ull;
        level = up;
    }
    w.sync();
    if (whole) {
        if (lane_id() < words)
            put(lane_id(), (uint32_t)(lds.root_cover(lane_id() / 2u) >> (32u * (lane_id() & 1u))) | w.mark[lane_id()]);
    } else if (home == kNone) {
        for (uint32_t base = 0; base < n; base += kWave) {
            const uint32_t v = base + lane_id();
            const uint64_t cm = __ballot(v < n && w.deg(v < n ? v : 0u) < 0);
            if (lane_id() < 2u) {
                const uint32_t i = base / 32u + lane_id();
                put(i, (uint32_t)(cm >> (32u * lane_id())) | w.mark[i]);
            }
        }
    } else {
        const __amdgpu_buffer_rsrc_t cb = ctx_rsrc(a, home);
        for (uint32_t i = lane_id(); i < words; i += kWave)
            put(i, (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(cb, ctx_cover(a, home % kCtxLevels) + 4u * i, 0, kCoherent) |
                       w.mark[i]);
    }
    w.sync();
    for (uint32_t i = lane_id(); i < words; i += kWave) w.mark[i] = 0u;
    w.sync();
}

// Copies the LDS context of `level` to this worker's area in HBM, with one
// user, the search itself; handoff_publish orders it before a donation's
// ticket.
template <class N>
__device__ __forceinline__ void publish(const SolveArgs &a, const N &w, const BitsLds &lds, const BitsWorker &b, uint32_t n,
                                        uint32_t level)
{
    const uint32_t ctx = b.wid * kCtxLevels + level, c = uni(lds.count(level)), lane = lane_id();
    const __amdgpu_buffer_rsrc_t cb = ctx_rsrc(a, ctx);
    const uint32_t row_words = c * 2u * ctx_slots(level);
    for (uint32_t i = lane; i < row_words; i += kWave)
        __builtin_amdgcn_raw_buffer_store_b32(reinterpret_cast<const uint32_t *>(lds.base + ctx_rows(level))[i], cb,
                                              kHbmBase + ctx_rows(level) + 4u * i, 0, kCoherent);
    for (uint32_t i = lane; i < c; i += kWave)
        __builtin_amdgcn_raw_buffer_store_b32(lds.id(level, i), cb, kHbmBase + ctx_ids(level) + 4u * i, 0, kCoherent);
    if (lane == 0) __builtin_amdgcn_raw_buffer_store_b32(c, cb, kHbmCount + 4u * level, 0, kCoherent);
    cover_words(a, w, lds, b.home, b.whole != 0u, n, level, nullptr, [&](uint32_t i, uint32_t word) {
        __builtin_amdgcn_raw_buffer_store_b32(word, cb, ctx_cover(a, level) + 4u * i, 0, kCoherent);
    });
    if (lane == 0) st_rlx(ctx_users(a, ctx), 1u);
}

// The published context b.home into this worker's LDS, as the search's first.
__device__ __forceinline__ void fetch_home(const SolveArgs &a, const BitsLds &lds, const BitsWorker &b)
{
    const uint32_t level = b.home % kCtxLevels, lane = lane_id();
    const __amdgpu_buffer_rsrc_t cb = ctx_rsrc(a, b.home);
    const uint32_t cap = ctx_cap(level), row_words = cap * 2u * ctx_slots(level);
    const uint32_t c = __builtin_amdgcn_raw_buffer_load_b32(cb, kHbmCount + 4u * level, 0, kCoherent);
    // Eight row words and the ids in flight per lane: the round trip, some two
    // microseconds, is what a fetch costs.  (Rows and ids past the context's
    // vertices are read too, and not used.)
    uint32_t id[4];
#pragma unroll
    for (uint32_t q = 0; q < 4u; ++q)
        id[q] = q * kWave < cap ? __builtin_amdgcn_raw_buffer_load_b32(cb, kHbmBase + ctx_ids(level) + 4u * (lane + q * kWave), 0, kCoherent) : 0u;
    for (uint32_t i = lane; i < row_words; i += 8u * kWave) {
        uint32_t x[8];
#pragma unroll
        for (uint32_t q = 0; q < 8u; ++q)
            x[q] = __builtin_amdgcn_raw_buffer_load_b32(cb, kHbmBase + ctx_rows(level) + 4u * (i + q * kWave), 0, kCoherent);
#pragma unroll
        for (uint32_t q = 0; q < 8u; ++q)
            if (i + q * kWave < row_words) reinterpret_cast<uint32_t *>(lds.base + ctx_rows(level))[i + q * kWave] = x[q];
    }
#pragma unroll
    for (uint32_t q = 0; q < 4u; ++q)
        if (lane + q * kWave < cap) lds.id(level, lane + q * kWave) = id[q];
    if (lane == 0) {
        lds.count(level) = c;
        lds.parent(level) = kNone;
    }
    nsync<false>();
}

// Searches one subtree to its end (or until the graph or the launch stops,
// which empties the stack): with nq > 0 the remainder of the node in w, which
// has nq live vertices, else the donated one in shared.home (its masks in
// `word`).  Entries above the stack's top at the call are the search's own;
// the ones below are whole node states and stay, except that donations take
// the oldest entry of either kind.
template <bool STAGED, class N>
__device__ __forceinline__ void bit_search(uint64_t args, const N &w, const BitsLds &lds, const GDesc &gd, uint32_t g,
                                           uint32_t nq, uint32_t word, BitsWorker &shared)
{
    // the launch arguments are read where the kernel got them (constant
    // memory, scalar loads)
    typedef const SolveArgs __attribute__((address_space(4))) *ConstArgs;
    const SolveArgs &a = *(const SolveArgs *)(ConstArgs)uni64(args);
    BitsWorker b = shared;
    b.stk = (char *)uni64((uint64_t)b.stk);
    b.stk_meta = (uint2 *)uni64((uint64_t)b.stk_meta);
    b.slot_bytes = uni(b.slot_bytes);
    b.wid = uni(b.wid);
    b.base = b.top;
    b.published = 0u;
    b.level = 0u;
    b.fresh = 0u;
    b.since = kDonateEvery;
    b.want = 0u;
    make_uniform(b);
    g = uni(g);
    nq = uni(nq);
    const uint32_t n = uni(gd.n);
    b.best = uni(gd.instance) == 0u ? uni((uint32_t)ld_rlx(&a.gstate[g].best)) : uni(gd.k) + 1u;
    if (nq != 0u) {
        b.level = ctx_level(nq);
        b.fresh = 1u;
        if (b.whole) {
            if (nq <= 64u)
                build_whole<1>(w, lds, b.level);
            else if (nq <= 128u)
                build_whole<2>(w, lds, b.level);
            else
                build_whole<4>(w, lds, b.level);
        } else {
            if (nq <= 64u)
                build_rows<1>(w, lds, b.level, nq);
            else if (nq <= 128u)
                build_rows<2>(w, lds, b.level, nq);
            else
                build_rows<4>(w, lds, b.level, nq);
            b.pending -= 1u;  // the node was counted before its context was made
        }
#pragma unroll
        for (uint32_t k = 0; k < 4u; ++k) {
            b.live[k] = low_bits(nq, k);
            b.settled[k] = 0ull;
        }
    } else {
        b.level = b.home % kCtxLevels;
        fetch_home(a, lds, b);
        unpack_masks(b, word);
    }
    bool pop = false;
    for (;;) {
        b.level = uni(b.level);
        const uint32_t slots = ctx_slots(b.level);
        uint32_t next;
        if (slots == 1u)
            next = bit_level<1, STAGED>(a, lds, gd, g, b, pop);
        else if (slots == 2u)
            next = bit_level<2, STAGED>(a, lds, gd, g, b, pop);
        else
            next = bit_level<4, STAGED>(a, lds, gd, g, b, pop);
        next = uni(next);
        make_uniform(b);
        pop = false;
        if (next == kBitsDone) break;
        if (next == kBitsCover) {
            const uint32_t level = b.level;
            record_cover(a, gd, g, uni(b.d), [&] {
                uint32_t *const cw = a.covers + gd.off_cover;
                cover_words(a, w, lds, b.home, b.whole != 0u, n, level, b.live, [&](uint32_t i, uint32_t x) { cw[i] = x; });
            });
            if (uni(gd.instance) == 0u) b.best = min(b.best, b.d);
            pop = true;
        } else if (next == kBitsDonate) {
            // the oldest entry, as in the main loop
            const uint32_t bs = (uint32_t)b.bot % a.depth;
            const uint2 m = b.stk_meta[bs];
            const uint32_t dm = uni(m.x), level = uni(m.y);
            bool sent = false;
            if (b.bot <= b.base) {
                sent = uni(try_enqueue(a, w, b.stk + (size_t)bs * b.slot_bytes, g, dm, level, b.slot_bytes)) != 0u;
                if (sent) b.moved += 2u * copy_bytes<N>(w.n);
            } else {
                const bool is_home = b.home != kNone && b.home % kCtxLevels == level;
                const uint32_t ctx = is_home ? b.home : b.wid * kCtxLevels + level;
                if (!is_home && !((b.published >> level) & 1u) && uni(ld_rlx(ctx_users(a, ctx))) == 0u) {
                    publish(a, w, lds, b, n, level);
                    b.published |= 1u << level;
                }
                b.published = uni(b.published);
                if (is_home || ((b.published >> level) & 1u)) {
                    // the oldest entries of this level, as many as are
                    // missing, and at most half of the stack (with all of it
                    // 1,024 uneven graphs took 17.9 ms instead of 17.3)
                    const uint32_t words = 4u * ctx_slots(level);
                    const uint32_t most = min(min(kDonateBatch, b.want), (uint32_t)(b.top - b.bot + 2) / 2u);
                    uint32_t other = 0;
                    if (lane_id() < most) other = b.stk_meta[((uint32_t)b.bot + lane_id()) % a.depth].y != level;
                    const uint64_t differ = __ballot(other);
                    const uint32_t count = uni(differ ? min(most, (uint32_t)__builtin_ctzll(differ)) : most);
                    if (lane_id() == 0) fetch_add(ctx_users(a, ctx), count);
                    if (uni(try_enqueue_bits(a, g, ctx, words, count, b.stk, b.stk_meta, (uint32_t)b.bot, b.slot_bytes)) != 0u) {
                        b.bot += (int)count - 1;
                        b.donations += count - 1u;
                        b.moved += 8u * words * count;
                        sent = true;
                    } else if (lane_id() == 0) {
                        fetch_add(ctx_users(a, ctx), 0u - count);
                    }
                }
            }
            b.since = 0u;
            if (sent) {
                ++b.bot;
                ++b.donations;
            }
        }
    }
    // the search's use of the copies ends with its last access
    if (b.published != 0u || b.home != kNone) {
        handoff_publish();
        if (lane_id() < kCtxLevels && ((b.published >> lane_id()) & 1u))
            fetch_add(ctx_users(a, b.wid * kCtxLevels + lane_id()), 0xFFFFFFFFu);
        if (b.home != kNone && lane_id() == 0) fetch_add(ctx_users(a, b.home), 0xFFFFFFFFu);
    }
    shared = b;
}

}  // namespace vcg
