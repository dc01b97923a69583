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
// Measured against that search without merging and with a leaf that counted
// every reply from scratch, one MI355X, averages over random positions, in
// us: depth 3 (ply 0-60) 65 -> 21, depth 5 (ply 5-80) 197 -> 61, depth 6 (ply
// 10-60) 1098 -> 449, three plies into the game depth 7 4059 -> 743 and depth
// 8 72788 -> 5539.  Of a depth-8 search of 8 ms the fused leaf takes 4.3 ms
// (integer VALU), the collapses 3.3 ms.
#pragma once
#include "kernels.h"

namespace pg {

constexpr int S_MAX_PLY = 16;
constexpr int S_MOVES = 218;  // most moves of a position in a game

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
// work-group of the last kernel adds into acc, paths, items and done.  Atomics
// on one line take about 6 ns each, one after the other, so each of these is
// spread over banks (work-group i adds to bank i % S_BANKS).
constexpr u32 S_BANKS = 32;
struct SPlan {
    alignas(128) u64 nNode[S_MAX_PLY];  // boards kept per ply
    alignas(128) u64 nList[S_MAX_PLY];  // moves listed per ply (the boards of that ply before the collapse)
    alignas(128) u64 paths[S_MAX_PLY];  // perft(ply): the listed moves, each with its parent's weight
    struct alignas(128) Bank {
        u64 acc, paths, items;          // of the last kernel; paths: of its ply
        u32 done;
        u32 tile;                       // tiles of the bank taken
    } bank[S_BANKS];
    alignas(128) u32 done;              // banks that are complete
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
// Boards per tile of the leaf (a wave each) and of the level kernel (a
// work-group each): a level of too few boards for whole tiles on every CU is
// dealt out a few at a time, for the time of its longest tile.
constexpr u32 S_RESIDENT = 1024;  // work-groups of the level kernel the chip holds (four per CU)
__device__ __forceinline__ u32 s_tile_boards(u64 n, u32 tiles, u32 least, u32 most) {
    const u64 t = (n + tiles - 1) / tiles;
    return t < least ? least : t > most ? most : (u32)t;
}

// the wave's sum of v; *wide: it passed 64 bits
__device__ __forceinline__ u64 s_wave_total(u64 v, bool *wide) {
    const u64 lo = wave_sum(v & 0xFFFFFFFFULL), hi = wave_sum(v >> 32) + (lo >> 32);
    *wide |= hi >> 32 != 0;
    return hi << 32 | (lo & 0xFFFFFFFFULL);
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

struct SSum {
    u64 total = 0, items = 0, paths = 0;
    bool carry = false, wide = false;
};

// *s += the wave's sum of w * c, all in scalar registers: the leaf leaves no
// vector register for a lane's sums.  *wide: the sum passed 64 bits.
__device__ __forceinline__ void s_wave_mad(u64 *s, u64 w, u32 c, bool *wide) {
    const u64 v = w * c;
    u64 lo, hi = 0;
    if (__ballot(v >> 26) == 0 && __ballot(w >> 32) == 0) {
        lo = wave_sum32((u32)v);
    } else {
        lo = uniform64(wave_sum((w & 0xFFFFFFFFULL) * c));
        hi = uniform64(wave_sum((w >> 32) * c));
        hi += lo >> 32;
        lo = hi << 32 | (lo & 0xFFFFFFFFULL);
    }
    *s += lo;
    *wide |= hi >> 32 != 0 || *s < lo;
}

// The moves of a work-group's boards (this lane: board b when live, of weight
// w) into the list of the next ply; node = the first board's place.  They are
// staged in LDS so that the list is written by consecutive lanes, a window at
// a time; a list that is full raises overflow.
constexpr int S_CAP = 6912;
struct ListTile {
    Pos b[LEAF_WG];
    u32 word[S_CAP];
    u32 next;
    u64 base;
};
template <int V>
__device__ __forceinline__ void s_list_tile(ListTile &s, bool live, const Pos &b, u64 w, u32 node, u64 *counter,
                                            const SLevel &L, SPlan *P, SSum &sum, const Tables &t) {
    u32 c = 0;
    if (live) {
        s.b[threadIdx.x] = b;
        c = count_any<V>(b, t);
        s_mad(&sum.paths, w, c, &sum.wide);
    }
    u64 total64;
    const u32 pos = (u32)block_excl_scan<LEAF_WG>(c, &total64);
    const u32 total = (u32)total64;
    if (threadIdx.x == 0) {
        s.base = atomicAdd(counter, total64);
        if (s.base + total > L.cap) P->overflow = 1;
    }
    __syncthreads();
    const u64 base = s.base;
    for (u32 start = 0; base + total <= L.cap && start < total;) {
        if (threadIdx.x == 0) s.next = total;
        __syncthreads();
        if (c && pos >= start && pos + c <= start + S_CAP) {
            if (generate_words<V>(s.b[threadIdx.x], t, s.word + (pos - start), c, threadIdx.x) != c) P->err = 2;
        } else if (c && pos >= start) {
            atomicMin(&s.next, pos);
        }
        __syncthreads();
        const u32 end = s.next;
        for (u32 j = start + threadIdx.x; j < end; j += LEAF_WG) {
            const u32 m = s.word[j - start];
            L.mv[base + j] = (u16)m;
            L.par[base + j] = (node + (m >> 16 & 255)) | (u32)piece_code(m >> 24) << S_NODE_BITS;
        }
        __syncthreads();
        start = end;
    }
    __syncthreads();
}

__device__ __forceinline__ Pos s_child(const SNode *nodes, u32 par, u16 mv, const Tables &t) {
    return made(nodes[par & S_NODE_MAX].b, mv, (int)(par >> S_NODE_BITS), t);
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
    const u32 bank = blockIdx.x % S_BANKS, banks = gridDim.x < S_BANKS ? gridDim.x : S_BANKS;
    SPlan::Bank &B = P->bank[bank];
    s_add(&B.acc, sum.total, &P->ovf);
    s_add(&B.paths, sum.paths, &P->overflow);
    s_add(&B.items, sum.items, &P->overflow);
    if (sum.carry) atomicOr(&P->ovf, 1u);
    if (sum.wide) atomicOr(&P->overflow, 1u);
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __syncthreads();
    __shared__ u32 last;
    if (threadIdx.x == 0) {
        last = 0;
        const u32 members = (gridDim.x - bank + S_BANKS - 1) / S_BANKS;
        if (atomicAdd(&B.done, 1u) + 1 == members) last = atomicAdd(&P->done, 1u) + 1 == banks;
    }
    __syncthreads();
    if (!last || threadIdx.x >= 64) return;
    // the last work-group's first wave: the banks' sums, with carries
    const u32 lane = threadIdx.x;
    u64 acc = 0, paths = 0, items = 0;
    if (lane < banks) {
        SPlan::Bank &L = P->bank[lane];
        acc = s_load(&L.acc);
        paths = s_load(&L.paths);
        items = s_load(&L.items);
        L.acc = L.paths = L.items = 0;
        L.done = L.tile = 0;
    }
    bool accWide = false, pathsWide = false;
    acc = s_wave_total(acc, &accWide);
    paths = s_wave_total(paths, &pathsWide);
    items = wave_sum(items);
    if (lane) return;
    out->acc = acc + bias;
    out->ovf = s_load(&P->ovf) | accWide | (acc + bias < bias);
    out->overflow = s_load(&P->overflow) | pathsWide;
    out->err = s_load(&P->err);
    out->items = items;
    const int l2 = depth >= 2 ? depth - 2 : 0;
    const u64 kept = s_load(&P->nNode[l2]);
    out->boards = kept ? kept : s_load(&P->nList[l2]);
    for (int l = 0; l < S_MAX_PLY; l++) {
        out->paths[l] = s_load(&P->paths[l]) + (l == depth - 1 ? paths : 0);
        P->nNode[l] = P->nList[l] = P->paths[l] = 0;
    }
    P->overflow = P->err = P->ovf = P->done = 0;
    __hip_atomic_store(&out->seq, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// ---------------------------------------------------------------- kernels
// perft(1) and perft(2): one work-group
template <int V>
__global__ __launch_bounds__(LEAF_WG) void ks_one(SRoot r, SPlan *P, int depth, u64 bias, SResult *out, u64 seq, Tables t) {
    SSum sum;
    const u32 tid = threadIdx.x;
    if (depth == 1) {
        if (tid == 0) sum.total = sum.paths = count_any<V>(r.b, t);
    } else if (tid < r.n) {
        sum.total = count_any<V>(made(r.b, r.mv[tid], r.piece[tid], t), t);
        sum.items = sum.paths = 1;
    }
    s_finish(P, sum, depth, bias, out, seq);
}

// perft(3): a wave per child of the root
constexpr u32 S_WAVES = LEAF_WG / 64;
template <int V>
__global__ __launch_bounds__(LEAF_WG) void ks_three(SRoot r, SPlan *P, u64 bias, SResult *out, u64 seq, Tables t) {
    __shared__ u32 list[S_WAVES][WAVE_LIST];
    SSum sum;
    const u32 wave = wave_number(), i = blockIdx.x * S_WAVES + wave;
    if (i < r.n) {
        u32 moves;
        sum.total = wave_perft2<V>(uniform_pos(made(r.b, r.mv[i], r.piece[i], t)), list[wave], &moves, &P->overflow, t);
        if ((threadIdx.x & 63) == 0) sum.items = sum.paths = moves;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) atomicAdd(&P->paths[1], (u64)r.n);
    s_finish(P, sum, 3, bias, out, seq);
}

// Plies 1 and 2 of a deeper search: the waves of work-group blockIdx list the
// moves of the child of the root by its move number blockIdx / parts, each by
// itself, which spares the kernel and the round through memory that a list of
// ply 2 would take.  The work-group's share is number blockIdx % parts of
// them, *lo to *hi.
template <int V>
__device__ __forceinline__ Pos s_child_moves(u32 *list, const SRoot &r, SPlan *P, u32 parts, u32 *lo, u32 *hi,
                                             const Tables &t) {
    const u32 i = blockIdx.x / parts, part = blockIdx.x % parts;
    const Pos c = uniform_pos(made(r.b, r.mv[i], r.piece[i], t));
    const u32 n = wave_words<V>(c, t, list, WAVE_LIST, &P->overflow);
    wave_sync();
    if (threadIdx.x == 0) {
        if (blockIdx.x == 0) atomicAdd(&P->paths[1], (u64)r.n);
        if (part == 0) atomicAdd(&P->paths[2], (u64)n);
    }
    *lo = n * part / parts;
    *hi = n * (part + 1) / parts;
    return c;
}

// perft(4): a wave per board of ply 2 (a few where a child has many moves)
constexpr u32 S_FOUR_PARTS = 8, S_TOP_PARTS = 8;
template <int V>
__global__ __launch_bounds__(LEAF_WG) void ks_four(SRoot r, SPlan *P, u64 bias, SResult *out, u64 seq, Tables t) {
    __shared__ u32 child[S_WAVES][WAVE_LIST], list[S_WAVES][WAVE_LIST];
    SSum sum;
    const u32 wave = wave_number();
    u32 lo, hi;
    const Pos c = s_child_moves<V>(child[wave], r, P, S_FOUR_PARTS, &lo, &hi, t);
    for (u32 j = lo + wave; j < hi; j += S_WAVES) {
        u32 moves;
        sum.total += wave_perft2<V>(wave_made(c, child[wave], j, t), list[wave], &moves, &P->overflow, t);
        if ((threadIdx.x & 63) == 0) {
            sum.items += moves;
            sum.paths += moves;
        }
    }
    s_finish(P, sum, 4, bias, out, seq);
}

// plies 1 to 3 of a deeper search: the nodes of ply 2 and the list of ply 3,
// a wave per board of ply 2
template <int V>
__global__ __launch_bounds__(LEAF_WG) void ks_top(SRoot r, SPlan *P, SRegion rg, Tables t) {
    __shared__ u32 child[S_WAVES][WAVE_LIST], list[S_WAVES][WAVE_LIST];
    __shared__ u32 first, count[S_WAVES];
    __shared__ u64 base;
    const u32 wave = wave_number(), lane = threadIdx.x & 63;
    u32 lo, hi;
    const Pos c = s_child_moves<V>(child[wave], r, P, S_TOP_PARTS, &lo, &hi, t);
    const SLevel L = s_level(rg, 2, 0);
    u64 paths = 0;
    if (threadIdx.x == 0) first = lo < hi ? (u32)atomicAdd(&P->nNode[2], (u64)(hi - lo)) : 0;
    __syncthreads();
    if (first + (hi - lo) > rg.node2) {  // node2 is for games, in which no child has more than S_MOVES moves
        if (threadIdx.x == 0) P->overflow = 1;
        return;
    }
    for (u32 j0 = lo; j0 < hi; j0 += S_WAVES) {
        const u32 j = j0 + wave, node = first + j - lo;
        u32 m = 0;
        if (j < hi) {
            const Pos b = wave_made(c, child[wave], j, t);
            m = wave_words<V>(b, t, list[wave], WAVE_LIST, &P->overflow);
            if (lane == 0) L.node[node] = SNode{b, 1, S_NO_SLOT, 0};
        }
        if (lane == 0) count[wave] = m;
        __syncthreads();
        u32 before = 0, total = 0;
        for (u32 w = 0; w < S_WAVES; w++) {
            if (w < wave) before += count[w];
            total += count[w];
        }
        if (threadIdx.x == 0) {
            base = atomicAdd(&P->nList[3], (u64)total);
            if (base + total > L.cap) P->overflow = 1;
        }
        __syncthreads();
        if (base + total <= L.cap)
            for (u32 k = lane; k < m; k += 64) {
                const u32 w = list[wave][k];
                L.mv[base + before + k] = (u16)w;
                L.par[base + before + k] = node | (u32)piece_code(w >> 24) << S_NODE_BITS;
            }
        paths += total;
        __syncthreads();
    }
    if (threadIdx.x == 0 && paths) atomicAdd(&P->paths[3], paths);
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
// node, the others add their weight to the slot.  A slot holds 16 bits of the
// hash beside the owner's item, so that of the unequal boards met one in 65536
// is compared: the owner is made again from the list and compared board for board.  Bound by
// the random accesses to the set and to the owners' parents, and by their
// latency: a work-group waits for its longest probe sequence before it
// reserves its nodes with one atomic (all on one counter, hence large
// work-groups), so two of 768 per CU, at 80 registers, beat one of 1024: 300
// us against 330 for the 1.9e6 moves of an opening's ply 5, which is 160 ps
// per move; 110 ps for the 30e6 of ply 6.
constexpr int S_COLLAPSE_WG = 768;
static __global__ __launch_bounds__(S_COLLAPSE_WG, 6) void ks_collapse(SPlan *P, SRegion rg, int l, Tables t) {
    if (s_stopped(P)) return;
    __shared__ u64 sBase;
    const SLevel L = s_level(rg, l - 1, uniform64(P->nNode[l - 1]));
    SNode *out = (SNode *)rg.half[l & 1];
    const u64 n = uniform64(P->nList[l]), slots = s_slots(n), cap = s_node_cap(rg);
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
            nd.b = made(p.b, mv, (int)(par >> S_NODE_BITS), t);
            const u64 h = s_hash(nd.b);
            const u64 id = (h << 48) | (u64)mv << 32 | par;
            at = __umul64hi(h, slots);
            u64 cur = slot_claim(&L.set[at].id, slot_look(&L.set[at].id), id);
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
                cur = slot_claim(&L.set[at].id, slot_look(&L.set[at].id), id);
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
template <bool LIST>
__device__ __forceinline__ u64 s_weight(const SLevel &A, const SNode *node, u64 i) {
    if constexpr (LIST) return A.node[A.par[i] & S_NODE_MAX].w;
    const SNode &nd = node[i];
    return nd.slot != S_NO_SLOT ? nd.w + A.set[nd.slot].w : nd.w;
}
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

// The moves of a few boards, each listed by a wave: up to S_FEW_BOARDS in a row
// per wave, then one reservation for the work-group.  For so few boards the
// kernel is one chain of latencies, and the listing by one lane each is the
// longest link: 30 us for the 12000 boards of an opening's ply 3 against 37.
constexpr u32 S_FEW_BOARDS = 4;
template <int V, bool LIST>
__device__ __forceinline__ void s_few_boards(u32 *word, const SRegion &rg, const SLevel &A, const SLevel &L, u64 n,
                                             u64 *counter, SPlan *P, SSum &sum, const Tables &t) {
    __shared__ u32 count[S_WAVES];
    __shared__ u64 first;
    const u32 wave = wave_number(), lane = threadIdx.x & 63;
    static_assert(S_WAVES * S_FEW_BOARDS * WAVE_LIST <= S_CAP, "the waves' lists share the window");
    u32 *const list = word + wave * S_FEW_BOARDS * WAVE_LIST;
    const u32 each = s_tile_boards(n, S_RESIDENT * S_WAVES, 1, S_FEW_BOARDS);
    for (u64 i0 = (u64)blockIdx.x * S_WAVES * each; i0 < n; i0 += (u64)gridDim.x * S_WAVES * each) {
        const u64 mine = i0 + wave * each;
        u32 m[S_FEW_BOARDS], total = 0;
#pragma unroll
        for (u32 k = 0; k < S_FEW_BOARDS; k++) {
            m[k] = 0;
            if (k < each && mine + k < n) {
                u64 w;
                const Pos b = uniform_pos(s_board<LIST, true>(rg, A, L.node, mine + k, &w, t));
                m[k] = wave_words<V>(b, t, list + k * WAVE_LIST, WAVE_LIST, &P->overflow);
                if (lane == 0) s_mad(&sum.paths, w, m[k], &sum.wide);
            }
            total += m[k];
        }
        if (lane == 0) count[wave] = total;
        __syncthreads();
        u32 before = 0, all = 0;
        for (u32 v = 0; v < S_WAVES; v++) {
            if (v < wave) before += count[v];
            all += count[v];
        }
        if (threadIdx.x == 0) {
            first = atomicAdd(counter, (u64)all);
            if (first + all > L.cap) P->overflow = 1;
        }
        __syncthreads();
        u64 at = first + before;
        if (first + all <= L.cap)
#pragma unroll
            for (u32 k = 0; k < S_FEW_BOARDS; k++) {
                for (u32 j = lane; j < m[k]; j += 64) {
                    const u32 w = list[k * WAVE_LIST + j];
                    L.mv[at + j] = (u16)w;
                    L.par[at + j] = (u32)(mine + k) | (u32)piece_code(w >> 24) << S_NODE_BITS;
                }
                at += m[k];
            }
        __syncthreads();
    }
}

// ply l's boards to the list of ply l + 1
template <int V, bool LIST>
__global__ __launch_bounds__(LEAF_WG) void ks_level(SPlan *P, SRegion rg, int l, Tables t) {
    __shared__ ListTile s;
    if (s_stopped(P)) return;
    const SLevel A = s_level(rg, l - 1, uniform64(P->nNode[l - 1]));
    const u64 n = uniform64(LIST ? P->nList[l] : P->nNode[l]);
    if (LIST && n > s_node_cap(rg)) {
        if (threadIdx.x == 0) P->overflow = 1;
        return;
    }
    const SLevel L = s_level(rg, l, n);
    if (LIST && blockIdx.x == 0 && threadIdx.x == 0) P->nNode[l] = n;
    SSum sum;
    const bool few = n <= (u64)S_RESIDENT * S_WAVES * S_FEW_BOARDS;
    if (few) s_few_boards<V, LIST>(s.word, rg, A, L, n, &P->nList[l + 1], P, sum, t);
    const u32 T = s_tile_boards(n, S_RESIDENT, 8, LEAF_WG);
    for (u64 tile = blockIdx.x; !few && tile * T < n; tile += gridDim.x) {
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
__global__ PG_LEAF_BOUNDS void ks_leaf(SPlan *P, SRegion rg, int depth, u64 bias, SResult *out, u64 seq, Tables t) {
    __shared__ LeafTile tiles[S_WAVES];
    u64 total = 0, paths = 0, items = 0;  // the wave's
    bool carry = false, wide = false;
    const int l = depth - 2;
    if (!s_stopped(P)) {
        const u32 wave = wave_number();
        LeafTile &s = tiles[wave];
        const u32 lane = threadIdx.x & 63, waves = gridDim.x * S_WAVES;
        const SLevel A = s_level(rg, l - 1, uniform64(P->nNode[l - 1]));
        const u64 n = uniform64(LIST ? P->nList[l] : P->nNode[l]);
        SNode *node = (SNode *)rg.half[l & 1];
        const u32 T = leaf_tile_boards(n, waves);
        // the first tiles are dealt out, the others (if any) taken as waves
        // get done, from as many counters as there are banks: with one, its
        // atomics (12 ns each) were all that perft(8) from the start without
        // merging waited for, 21.9 ms
        const u32 banks = gridDim.x < S_BANKS ? gridDim.x : S_BANKS, bank = blockIdx.x % banks;
        const u32 mine = ((gridDim.x - bank + banks - 1) / banks) * S_WAVES;  // the bank's waves
        const bool more = (u64)waves * T < n;
        for (u64 tile = (u64)(blockIdx.x / banks * S_WAVES + wave) * banks + bank; tile * T < n;) {
            u32 next = 0;
            if (more && lane == 0) next = atomicAdd(&P->bank[bank].tile, 1u) + mine;
            const u64 i = tile * T + lane;
            const bool live = lane < T && i < n;
            Pos b{};
            u64 w;
            if (live) b = s_board<LIST, false>(rg, A, node, i, &w, t);
            tile = more ? (u64)(u32)__builtin_amdgcn_readfirstlane((int)next) * banks + bank : n;
            const u32 c = leaf_expand<V>(s, live, b, &P->err, t);
            w = 0;
            if (live) w = s_weight<LIST>(A, node, i);  // again: there is no register to keep it in
            s_wave_mad(&total, w, live ? s.per[lane] : 0, &carry);
            s_wave_mad(&paths, w, c, &wide);
            items += wave_sum32(c);
            wave_sync();
        }
    }
    SSum sum;
    if ((threadIdx.x & 63) == 0) sum = SSum{total, items, paths, carry, wide};
    s_finish(P, sum, depth, bias, out, seq);
}

}  // namespace pg
