// single.h -- perft of one root when only its total is wanted (pg_perft):
// breadth-first, equal boards of a level collapsed into one with a weight.
//
// Every board of a level is kept with the number of paths that reach it, so
// the total is the weighted sum of the last boards' perft(2) and nothing has
// to come back up the levels.  Two boards are merged only when they are the
// same board (compared in full, not by a key), so the total is exact.
//
// No planning or scan kernels: a work-group reserves the output range of its
// tile with one atomic on the level's counter, and every kernel derives the
// arrays' places from the counters its predecessors left.  A depth-d search
// takes 1 launch for d <= 4, 2 for d = 5 and 4 + 3 (d - 5) above (a search
// with a plan and a scan per ply took 6 per ply).
//
// Measured against that search without merging, one MI355X, averages over
// random positions: depth 3 (ply 0-60) 67 -> 26 us, depth 5 (ply 5-80) 213 ->
// 92 us, depth 6 (ply 10-60) 570 -> 364 us, three plies into the game depth 7
// 6.3 -> 1.6 ms and depth 8 67 -> 18 ms.  Of a depth-8 search of 15 ms the
// fused leaf takes 10.3 ms (integer VALU), the last ply's collapse 3.8 ms.
#pragma once
#include "kernels.h"

namespace pg {

constexpr int S_MAX_PLY = 16;
constexpr int S_MOVES = 218;  // most moves of a position

// A kept board: the paths that reach it are w, or, until the level kernel has
// run, w + set[slot].w (the paths merged into it by the collapse).
struct __align__(64) SNode {
    Pos b;
    u64 w;
    u32 slot;  // S_NO_SLOT: w is complete
    u32 pad;
};
static_assert(sizeof(SNode) == 64, "a kept board is one 64-byte line");
constexpr u32 S_NO_SLOT = 0xFFFFFFFFu;

// Collapse-set slot: id = tag << 48 | move << 32 | parent word of the owner,
// from which its board can be made again (never 0, since a piece moves);
// 0 = free; w = paths merged into the owner.
struct __align__(16) SSlot {
    u64 id, w;
};

// A listed move carries its parent's node and the moving piece in one word.
constexpr u32 S_NODE_BITS = 29;
constexpr u64 S_NODE_MAX = (1ULL << S_NODE_BITS) - 1;
constexpr u64 S_ITEM_MAX = 3400000000ULL;  // s_slots of as many items: slot numbers are 32 bits

// Device state of a search.  All counters are zero between calls: the last
// work-group of a search publishes them to the host and clears them.  Every
// work-group of the last kernel adds into acc, items, paths and done, which
// therefore lie in lines of their own (atomics on one address take about 6 ns
// each, one after the other).
struct SPlan {
    alignas(128) u64 nNode[S_MAX_PLY];  // boards kept per ply
    alignas(128) u64 nList[S_MAX_PLY];  // moves listed per ply (the boards of that ply before the collapse)
    alignas(128) u64 paths[S_MAX_PLY];  // perft(ply): the listed moves, each with its parent's weight
    alignas(128) u64 acc;
    alignas(128) u64 items;
    alignas(128) u32 done;
    alignas(128) u32 tile;              // next tile of the last kernel
    alignas(128) u32 overflow, err, ovf;
};

// What the host reads, in pinned memory; seq is written last.
struct SResult {
    u64 acc, items;
    u64 boards;             // boards of the last materialized ply
    u64 paths[S_MAX_PLY];
    u32 overflow, err, ovf, pad;
    u64 seq;
};

// The root and its moves, listed on the host: a kernel argument.
struct SRoot {
    Pos b;
    u32 n;
    u16 mv[S_MOVES + 2];
    u8 piece[S_MOVES + 2];
};

// The arena is used as two halves: ply l lives in half l & 1 as its nodes,
// then the moves listed from them (ply l + 1), then, when ply l + 1 is
// collapsed, its set.  Collapsing ply l + 1 writes its nodes to the other
// half, over ply l - 1, which is done with.
struct SRegion {
    u8 *half[2];
    u64 bytes;      // per half
    u64 node2;      // nodes reserved for ply 2 (its count is not known while its list is written)
    u64 collapse;   // bit l: ply l is collapsed
};
struct SLevel {
    SNode *node;
    u16 *mv;
    u32 *par;
    SSlot *set;
    u64 cap;        // most moves the list holds
};

PG_HD u64 s_align(u64 x) { return (x + 255) & ~255ULL; }
PG_HD u64 s_slots(u64 m) { return m + m / 4 + 64; }

// places of ply l's nodes and of the list and set of ply l + 1, given the
// number of nodes; the set of a full list fits behind it
PG_HD SLevel s_level(const SRegion &r, int l, u64 nodes) {
    SLevel L;
    u8 *h = r.half[l & 1];
    const u64 a = s_align((l == 2 ? r.node2 : nodes) * sizeof(SNode));
    const u64 per = (r.collapse >> (l + 1)) & 1 ? 2 + 4 + 20 : 2 + 4;
    const u64 slack = 4096;  // alignment of the three arrays and the set's constant part
    u64 cap = a + slack < r.bytes ? (r.bytes - a - slack) / per : 0;
    if (cap > S_ITEM_MAX) cap = S_ITEM_MAX;
    L.node = (SNode *)h;
    L.mv = (u16 *)(h + a);
    L.par = (u32 *)(h + a + s_align(2 * cap));
    L.set = (SSlot *)(h + a + s_align(2 * cap) + s_align(4 * cap));
    L.cap = cap;
    return L;
}
PG_HD u64 s_node_cap(const SRegion &r) {
    const u64 c = r.bytes / sizeof(SNode);
    return c < S_NODE_MAX ? c : S_NODE_MAX;
}

// ---------------------------------------------------------------- tiles
// A work-group's boards and the moves they generate (the fused leaf's window;
// 40 KB, so that four work-groups share a CU's LDS).
constexpr int S_CAP = 6800;
struct STile {
    Pos b[LEAF_WG];
    u16 mv[S_CAP];
    u16 tag[S_CAP];  // owner | moving piece << 8
    u32 per[LEAF_WG];
    u32 next;
    u64 base;
};

// Boards per tile.  Whole waves of boards keep the lanes of the tile's
// expansion full; a level of too few boards for that on every CU is dealt out
// 8 boards or more at a time, for the time of its longest tile.  (The fused
// leaf of a depth-5 search, 2e4 boards: 84 us in tiles of 256, 47 us so.)
constexpr u32 S_RESIDENT = 1024;  // work-groups the chip holds (four per CU)
__device__ __forceinline__ u32 s_tile_boards(u64 n) {
    if (n < 64 * S_RESIDENT) return n < 8 * S_RESIDENT ? 8u : (u32)((n + S_RESIDENT - 1) / S_RESIDENT);
    const u64 t = n / (8 * S_RESIDENT) / 64 * 64;
    return t < 64 ? 64u : t > LEAF_WG ? (u32)LEAF_WG : (u32)t;
}

// *acc += the work-group's sum of s, one atomic; sums may need all 64 bits,
// and *ovf is raised when a total passes them
__device__ __forceinline__ void s_add(u64 *acc, u64 s, u32 *ovf) {
    __shared__ u64 part[LEAF_WG / 64][2];
    const u64 lo = wave_sum(s & 0xFFFFFFFFULL), hi = wave_sum(s >> 32);
    if ((threadIdx.x & 63) == 0) {
        part[threadIdx.x >> 6][0] = lo;
        part[threadIdx.x >> 6][1] = hi;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        u64 l = 0, h = 0;
        for (int i = 0; i < LEAF_WG / 64; i++) {
            l += part[i][0];
            h += part[i][1];
        }
        h += l >> 32;
        if (h >> 32) atomicOr(ovf, 1u);
        if (l | h) add_checked(acc, (h << 32) | (l & 0xFFFFFFFFULL), ovf);
    }
    __syncthreads();
}
// s += w * c with a carry check
__device__ __forceinline__ void s_mad(u64 *s, u64 w, u64 c, bool *carry) {
    const u64 v = w * c;
    *s += v;
    *carry |= __umul64hi(w, c) != 0 || *s < v;
}

// The moves of the tile's boards (lane tid: s.b[tid] with c legal moves, 0 for
// an idle lane), a window at a time: f(first, last, start) handles the listed
// moves first..last, of which slot j - start holds number j.
template <int V, class F>
__device__ __forceinline__ u32 s_windows(STile &s, u32 c, u32 *err, const Tables &t, F &&f, u32 pos, u32 total) {
    const int tid = threadIdx.x;
    u32 start = 0;
    while (start < total) {
        const u32 end = start + S_CAP;
        if (tid == 0) s.next = total;
        __syncthreads();
        if (c && pos >= start && pos + c <= end) {
            const u32 g = generate_any<V>(s.b[tid], t, s.mv + (pos - start), c, s.tag + (pos - start), (u32)tid);
            if (g != c) atomicOr(err, 2u);
        } else if (c && pos >= start) {
            atomicMin(&s.next, pos);
        }
        __syncthreads();
        const u32 wend = s.next;
        f(start, wend);
        __syncthreads();
        start = wend;
    }
    return total;
}

struct SSum {
    u64 total = 0, items = 0, paths = 0;
    bool carry = false, wide = false;
};

// perft(2) of the tile's boards times their weights
template <int V>
__device__ __forceinline__ void s_leaf_tile(STile &s, bool live, const Pos &b, u64 w, SSum &sum, u32 *err,
                                            const Tables &t) {
    const int tid = threadIdx.x;
    u32 c = 0;
    if (live) {
        c = count_any<V>(b, t);
        s.b[tid] = b;
    }
    s.per[tid] = 0;
    u64 total;
    const u32 pos = (u32)block_excl_scan<LEAF_WG>(c, &total);
    s_windows<V>(
        s, c, err, t,
        [&](u32 start, u32 wend) {
            for (u32 j = start + tid; j < wend; j += LEAF_WG) {
                const u32 tg = s.tag[j - start];
                const u32 o = tg & 255;
                atomicAdd(&s.per[o], count_after_as<V>(s.b[o], s.mv[j - start], (int)(tg >> 8), t));
            }
        },
        pos, (u32)total);
    if (live) {
        s_mad(&sum.total, w, s.per[tid], &sum.carry);
        s_mad(&sum.paths, w, c, &sum.wide);
        sum.items += c;
    }
    __syncthreads();
}

// the tile's moves into the list of the next ply; node = the first board's
// place.  False when the list is full.
template <int V>
__device__ __forceinline__ void s_list_tile(STile &s, bool live, const Pos &b, u64 w, u32 node, u64 *counter,
                                            const SLevel &L, SPlan *P, SSum &sum, const Tables &t) {
    const int tid = threadIdx.x;
    u32 c = 0;
    if (live) {
        c = count_any<V>(b, t);
        s.b[tid] = b;
        s_mad(&sum.paths, w, c, &sum.wide);
    }
    u64 total64;
    const u32 pos = (u32)block_excl_scan<LEAF_WG>(c, &total64);
    if (tid == 0) {
        s.base = atomicAdd(counter, total64);
        if (s.base + total64 > L.cap) P->overflow = 1;
    }
    __syncthreads();
    const u64 base = s.base;
    if (base + total64 <= L.cap)
        s_windows<V>(
            s, c, &P->err, t,
            [&](u32 start, u32 wend) {
                for (u32 j = start + tid; j < wend; j += LEAF_WG) {
                    const u32 tg = s.tag[j - start];
                    L.mv[base + j] = s.mv[j - start];
                    L.par[base + j] = (node + (tg & 255)) | (tg >> 8) << S_NODE_BITS;
                }
            },
            pos, (u32)total64);
    __syncthreads();
}

__device__ __forceinline__ Pos s_made(Pos p, u16 mv, int piece, const Tables &t) {
    if (pos_side(p)) make_move_as<BLACK, false>(p, mv, piece, nullptr, t);
    else make_move_as<WHITE, false>(p, mv, piece, nullptr, t);
    return p;
}
__device__ __forceinline__ Pos s_child(const SNode *nodes, u32 par, u16 mv, const Tables &t) {
    return s_made(nodes[par & S_NODE_MAX].b, mv, (int)(par >> S_NODE_BITS), t);
}

__device__ __forceinline__ u64 s_load(const u64 *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ u32 s_load(const u32 *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// whether an earlier kernel of the search found that a level does not fit
// (one answer for the whole work-group)
__device__ __forceinline__ bool s_stopped(const SPlan *P) {
    __shared__ u32 stop;
    if (threadIdx.x == 0) stop = s_load(&P->overflow);
    __syncthreads();
    return stop != 0;
}

// Ends the last kernel of a search: adds the work-group's sums, and the last
// work-group to arrive hands the counters to the host and clears them.  What
// the last one reads was written by atomics that had returned before the
// writer arrived, so waiting for one's own is enough (a release fence would
// write the L2 back once per work-group).
__device__ __forceinline__ void s_finish(SPlan *P, const SSum &sum, int depth, u64 bias, SResult *out, u64 seq) {
    s_add(&P->acc, sum.total, &P->ovf);
    s_add(&P->paths[depth - 1], sum.paths, &P->overflow);
    s_add(&P->items, sum.items, &P->overflow);
    if (sum.carry) atomicOr(&P->ovf, 1u);
    if (sum.wide) atomicOr(&P->overflow, 1u);
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x) return;
    if (atomicAdd(&P->done, 1u) + 1 != gridDim.x) return;
    const u64 acc = s_load(&P->acc);
    out->acc = acc + bias;
    out->ovf = s_load(&P->ovf) | (acc + bias < bias);
    out->overflow = s_load(&P->overflow);
    out->err = s_load(&P->err);
    out->items = s_load(&P->items);
    const int last = depth >= 2 ? depth - 2 : 0;
    const u64 kept = s_load(&P->nNode[last]);
    out->boards = kept ? kept : s_load(&P->nList[last]);
    for (int l = 0; l < S_MAX_PLY; l++) {
        out->paths[l] = s_load(&P->paths[l]);
        P->nNode[l] = P->nList[l] = P->paths[l] = 0;
    }
    P->acc = P->items = 0;
    P->overflow = P->err = P->ovf = P->done = P->tile = 0;
    __hip_atomic_store(&out->seq, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

#define S_LEAF_BOUNDS(V) __launch_bounds__(LEAF_WG) __attribute__((amdgpu_waves_per_eu((V) == SL_KOGGE ? 4 : 5, 8)))

// ---------------------------------------------------------------- kernels
// perft(1) and perft(2): one work-group
template <int V>
__global__ __launch_bounds__(LEAF_WG) void ks_one(SRoot r, SPlan *P, int depth, u64 bias, SResult *out, u64 seq, Tables t) {
    SSum sum;
    const u32 tid = threadIdx.x;
    if (depth == 1) {
        if (tid == 0) sum.total = sum.paths = count_any<V>(r.b, t);
    } else if (tid < r.n) {
        sum.total = count_after_as<V>(r.b, r.mv[tid], r.piece[tid], t);
        sum.items = sum.paths = 1;
    }
    s_finish(P, sum, depth, bias, out, seq);
}

// perft(3): the fused leaf over the root's children, 8 per work-group, so
// that each work-group's children's moves are one pass of its lanes
constexpr int S_SMALL_TILE = 8;
template <int V>
__global__ S_LEAF_BOUNDS(V) void ks_three(SRoot r, SPlan *P, u64 bias, SResult *out, u64 seq, Tables t) {
    __shared__ STile s;
    SSum sum;
    const u32 i = blockIdx.x * S_SMALL_TILE + threadIdx.x;
    const bool live = threadIdx.x < S_SMALL_TILE && i < r.n;
    Pos b{};
    if (live) b = s_made(r.b, r.mv[i], r.piece[i], t);
    s_leaf_tile<V>(s, live, b, 1, sum, &P->err, t);
    if (blockIdx.x == 0 && threadIdx.x == 0) atomicAdd(&P->paths[1], (u64)r.n);
    s_finish(P, sum, 3, bias, out, seq);
}

// The children of the root's move number blockIdx / PARTS, part blockIdx %
// PARTS of them: every work-group lists the moves of its child of the root
// itself (one lane), which spares the kernel and the round through memory
// that a list of ply 2 would take.
template <int V, int PARTS>
__device__ __forceinline__ bool s_grandchild(STile &s, const SRoot &r, SPlan *P, u32 *n2, Pos *b, const Tables &t) {
    const u32 i = blockIdx.x / PARTS, part = blockIdx.x % PARTS;
    const Pos c = s_made(r.b, r.mv[i], r.piece[i], t);
    if (threadIdx.x == 0) s.next = generate_any<V>(c, t, s.mv, 256, s.tag, 0);
    __syncthreads();
    const u32 n = s.next < 256 ? s.next : 256;
    const u32 lo = n * part / PARTS, hi = n * (part + 1) / PARTS;
    const u32 j = lo + threadIdx.x;
    const bool live = j < hi;
    if (live) *b = s_made(c, s.mv[j], s.tag[j] >> 8, t);
    if (blockIdx.x == 0 && threadIdx.x == 0) atomicAdd(&P->paths[1], (u64)r.n);
    if (part == 0 && threadIdx.x == 0) atomicAdd(&P->paths[2], (u64)n);
    *n2 = hi - lo;
    __syncthreads();
    return live;
}

// perft(4): the fused leaf over the root's grandchildren
constexpr int S_FOUR_PARTS = 4, S_TOP_PARTS = 2;
template <int V>
__global__ S_LEAF_BOUNDS(V) void ks_four(SRoot r, SPlan *P, u64 bias, SResult *out, u64 seq, Tables t) {
    __shared__ STile s;
    SSum sum;
    Pos b{};
    u32 n;
    const bool live = s_grandchild<V, S_FOUR_PARTS>(s, r, P, &n, &b, t);
    s_leaf_tile<V>(s, live, b, 1, sum, &P->err, t);
    s_finish(P, sum, 4, bias, out, seq);
}

// plies 1 to 3 of a deeper search: the nodes of ply 2 and the list of ply 3
template <int V>
__global__ S_LEAF_BOUNDS(V) void ks_top(SRoot r, SPlan *P, SRegion rg, Tables t) {
    __shared__ STile s;
    __shared__ u32 first;
    SSum sum;
    Pos b{};
    u32 n;
    const bool live = s_grandchild<V, S_TOP_PARTS>(s, r, P, &n, &b, t);
    const SLevel L = s_level(rg, 2, 0);
    if (threadIdx.x == 0) first = (u32)atomicAdd(&P->nNode[2], (u64)n);
    __syncthreads();
    if (first + n > rg.node2) {  // cannot happen: node2 is the root's moves times the most a position has
        if (threadIdx.x == 0) P->overflow = 1;
        return;
    }
    if (live) L.node[first + threadIdx.x] = SNode{b, 1, S_NO_SLOT, 0};
    s_list_tile<V>(s, live, b, 1, first, &P->nList[3], L, P, sum, t);
    s_add(&P->paths[3], sum.paths, &P->overflow);
}

// empties the set of ply l (whose size follows from its list)
static __global__ __launch_bounds__(256) void ks_clear(SPlan *P, SRegion rg, int l) {
    if (s_stopped(P)) return;
    const SLevel L = s_level(rg, l - 1, P->nNode[l - 1]);
    const u64 n = s_slots(P->nList[l]);
    ulonglong2 *set = reinterpret_cast<ulonglong2 *>(L.set);
    PG_GRID_LOOP(i, n) set[i] = make_ulonglong2(0, 0);
}

// 64-bit mix of a board (equal boards, equal values): the six words, each
// folded so that its high bits reach all of the product, times odd constants
__device__ __forceinline__ u64 s_hash(const Pos &p) {
    auto fold = [](u64 x) { return x ^ (x >> 32); };
    u64 h = fold(p.white) * 0x9E3779B97F4A7C15ULL + fold(p.pawns) * 0xC2B2AE3D27D4EB4FULL +
            fold(p.knights) * 0x165667B19E3779F9ULL + fold(p.bishopQueens) * 0xD6E8FEB86659FD93ULL +
            fold(p.rookQueens) * 0xA0761D6478BD642FULL + fold(p.kings) * 0xE7037ED1A0B428DBULL;
    h ^= h >> 32;
    h *= 0xBF58476D1CE4E5B9ULL;
    return h ^ (h >> 29);
}

// Collapse of ply l: each listed move is made, and inserted in an
// open-addressing set; the first of equal boards owns the slot and becomes a
// node, the others add their weight to the slot.  A slot holds 32 bits of the
// hash beside the owner's item, so only a probable match is compared: the
// owner is made again from the list and compared board for board.  Bound by
// the random accesses to the set (one line per board, two operations on it
// for a merged one): about 110 ps per listed move once the set is past the
// caches.  Every work-group reserves its nodes with one atomic per pass on one
// counter, hence the largest work-group: 1024 lanes take 326 us for the 1.9e6
// moves of an opening's ply 5, 512 take 363 and 256 take 414.
constexpr int S_COLLAPSE_WG = 1024;
static __global__ __launch_bounds__(S_COLLAPSE_WG) void ks_collapse(SPlan *P, SRegion rg, int l, Tables t) {
    if (s_stopped(P)) return;
    __shared__ u64 sBase;
    const SLevel L = s_level(rg, l - 1, P->nNode[l - 1]);
    SNode *out = (SNode *)rg.half[l & 1];
    const u64 n = P->nList[l], slots = s_slots(n), cap = s_node_cap(rg);
    for (u64 base = (u64)blockIdx.x * S_COLLAPSE_WG; base < n; base += (u64)gridDim.x * S_COLLAPSE_WG) {
        const u64 i = base + threadIdx.x;
        bool own = i < n;
        SNode nd{};
        u64 at = 0;
        if (own) {
            const u32 par = L.par[i];
            const u16 mv = L.mv[i];
            const SNode &p = L.node[par & S_NODE_MAX];
            nd.w = p.w;
            nd.b = s_made(p.b, mv, (int)(par >> S_NODE_BITS), t);
            const u64 h = s_hash(nd.b);
            const u64 id = (h << 48) | (u64)mv << 32 | par;
            at = __umul64hi(h, slots);
            u64 cur = atomicCAS(&L.set[at].id, 0ULL, id);
            for (u64 step = 0; cur; step++) {
                if ((cur ^ id) >> 48 == 0) {
                    const Pos q = s_child(L.node, (u32)cur, (u16)(cur >> 32), t);
                    if (q.white == nd.b.white && q.pawns == nd.b.pawns && q.knights == nd.b.knights &&
                        q.bishopQueens == nd.b.bishopQueens && q.rookQueens == nd.b.rookQueens && q.kings == nd.b.kings) {
                        atomicAdd(&L.set[at].w, nd.w);
                        own = false;
                        break;
                    }
                }
                if (step >= slots) { P->err = 3; break; }
                at = at + 1 < slots ? at + 1 : 0;
                cur = atomicCAS(&L.set[at].id, 0ULL, id);
            }
            nd.slot = (u32)at;
        }
        u64 total;
        u64 pos = block_excl_scan<S_COLLAPSE_WG>(own, &total);
        if (threadIdx.x == 0) {
            sBase = atomicAdd(&P->nNode[l], total);
            if (sBase + total > cap) P->overflow = 1;
        }
        __syncthreads();
        pos += sBase;
        if (own && pos < cap) out[pos] = nd;
        __syncthreads();
    }
}

// Board number i of ply l and its weight: a node of the collapse (its weight
// completed here), or (LIST) the listed move i made from its parent, kept as
// node i for the next ply when KEEP.
template <bool LIST, bool KEEP>
__device__ __forceinline__ Pos s_board(const SRegion &rg, const SLevel &A, SNode *node, u64 i, u64 *w, const Tables &t) {
    if constexpr (LIST) {
        const u32 par = A.par[i];
        *w = A.node[par & S_NODE_MAX].w;
        const Pos b = s_child(A.node, par, A.mv[i], t);
        if (KEEP) node[i] = SNode{b, *w, S_NO_SLOT, 0};
        return b;
    } else {
        const SNode nd = node[i];
        *w = nd.w;
        if (nd.slot != S_NO_SLOT) *w += A.set[nd.slot].w;
        if (KEEP) {
            node[i].w = *w;
            node[i].slot = S_NO_SLOT;
        }
        return nd.b;
    }
}

// ply l's boards to the list of ply l + 1
template <int V, bool LIST>
__global__ S_LEAF_BOUNDS(V) void ks_level(SPlan *P, SRegion rg, int l, Tables t) {
    __shared__ STile s;
    if (s_stopped(P)) return;
    const SLevel A = s_level(rg, l - 1, P->nNode[l - 1]);
    const u64 n = LIST ? P->nList[l] : P->nNode[l];
    if (LIST && n > s_node_cap(rg)) {
        if (threadIdx.x == 0) P->overflow = 1;
        return;
    }
    const SLevel L = s_level(rg, l, n);
    if (LIST && blockIdx.x == 0 && threadIdx.x == 0) P->nNode[l] = n;
    const u32 T = s_tile_boards(n);
    SSum sum;
    for (u64 tile = blockIdx.x; tile * T < n; tile += gridDim.x) {
        const u64 i = tile * T + threadIdx.x;
        const bool live = threadIdx.x < T && i < n;
        Pos b{};
        u64 w = 0;
        if (live) b = s_board<LIST, true>(rg, A, L.node, i, &w, t);
        s_list_tile<V>(s, live, b, w, (u32)(tile * T), &P->nList[l + 1], L, P, sum, t);
    }
    s_add(&P->paths[l + 1], sum.paths, &P->overflow);
    if (sum.wide) P->overflow = 1;
}

// the last plies: perft(2) of ply depth - 2's boards
template <int V, bool LIST>
__global__ S_LEAF_BOUNDS(V) void ks_leaf(SPlan *P, SRegion rg, int depth, u64 bias, SResult *out, u64 seq, Tables t) {
    __shared__ STile s;
    __shared__ u32 next;
    SSum sum;
    const int l = depth - 2;
    if (!s_stopped(P)) {
        const SLevel A = s_level(rg, l - 1, P->nNode[l - 1]);
        const u64 n = LIST ? P->nList[l] : P->nNode[l];
        SNode *node = (SNode *)rg.half[l & 1];
        const u32 T = s_tile_boards(n);
        // the first tiles are dealt out, the others taken as work-groups get done
        for (u64 tile = blockIdx.x; tile * T < n;) {
            if (threadIdx.x == 0) next = atomicAdd(&P->tile, 1u) + gridDim.x;
            const u64 i = tile * T + threadIdx.x;
            const bool live = threadIdx.x < T && i < n;
            Pos b{};
            u64 w = 0;
            if (live) b = s_board<LIST, false>(rg, A, node, i, &w, t);
            s_leaf_tile<V>(s, live, b, w, sum, &P->err, t);
            tile = next;
            __syncthreads();
        }
    }
    s_finish(P, sum, depth, bias, out, seq);
}

}  // namespace pg
