// dloop.h -- device-driven level loop: the breadth-first perft of a batch of
// roots with no host round trip between levels, so the whole search can be
// captured once into a HIP graph and replayed.
//
// Sizes and array pointers of every level live in a Plan in device memory.
// The work-group that ends a level's scan reads the total, carves the next
// level's arrays out of a bump region (stack discipline: transient
// move/parent/set arrays are released after expansion) and publishes the
// level's size; the work kernels are persistent grid-stride loops that read
// their size from the plan.  A kernel of a small level takes 4 to 5 us
// whatever it does, so a level takes few: scan and plan; moves, their offsets
// and the empty duplicate set; children; duplicates.  If a level does not
// fit, the plan raises `overflow` and publishes size 0, every later kernel
// becomes a no-op, and the host reruns the batch in halves.  Per-root results
// come back up the levels by segmented sums (children of a board are
// contiguous), as in the TT path.
#pragma once
#include "tt.h"

namespace pg {

struct DLevel {
    u64 n;            // boards at this level
    Pos *b;
    Key128 *k;
    u32 *cnt;
    u64 *off;         // n + 1 exclusive offsets of the children
    u64 *perft;
    u8 *state;
    u32 *dup;
    u64 *tiles;       // children before each tile of GEN_WG boards
    u64 kids;         // children of the level
    u32 *live;        // leaf level: the boards with moves (kd_live), when there was room
    u16 *mv;          // moves / parents of the children: transient, or kept (keep) when
    u32 *par;         //   the children's boards are not stored (the leaf makes them)
    u32 *set;         // transient: duplicate set
    u64 setMask;
    u64 release;      // bump top to return to after expansion
    u32 keep;         // mv / par outlive the expansion
};

struct Plan {
    u8 *base;
    u64 cap, top;
    u32 overflow, err;  // overflow: a level did not fit the region
    u64 leafItems;
    u64 acc;
    u64 bias;           // test hook: starting value of every root's total
    u32 ovf;            // a 64-bit total wrapped
    u64 peak;           // highest bump top reached (bytes of the region used)
    u64 liveN;          // entries of the leaf level's live list
    u64 began;          // device clock at the search's start
    u32 arrived[TT_MAX_DEPTH];  // work-groups done with a level's kd_scan
    // A root that no game leads to was seen (pos_regular): nothing is searched,
    // and the host runs the search again with the plain leaf.  Not among what
    // kd_begin copies: set by it, cleared by kd_end.
    u64 irregular;
    DLevel lv[TT_MAX_DEPTH];
};

// A search's inputs and results in pinned host memory, which its first and
// last kernels read and write themselves: copies on the stream cost 8 to 10 us
// each, of which a search would need five.
struct Link {
    Plan plan;          // as the search begins; the last kernel updates the counters
    const Pos *b;       // roots and keys (null: already on the device)
    const Key128 *k;
    u64 *out;           // the roots' perfts (null: left on the device)
    u64 ticks;          // device clock ticks from the first kernel to the last
    u64 want, seq;      // seq = want is written last
};

__device__ __forceinline__ void *plan_alloc(Plan *P, u64 bytes) {
    const u64 a = (P->top + 255) & ~255ULL;
    if (a + bytes > P->cap) {
        P->overflow = 1;
        return nullptr;
    }
    P->top = a + bytes;
    if (P->top > P->peak) P->peak = P->top;
    return P->base + a;
}

// as plan_alloc, for an optional array: no room leaves the plan as it was
__device__ __forceinline__ void *plan_try_alloc(Plan *P, u64 bytes) {
    const u64 a = (P->top + 255) & ~255ULL;
    if (a + bytes > P->cap) return nullptr;
    P->top = a + bytes;
    if (P->top > P->peak) P->peak = P->top;
    return P->base + a;
}

// room for the offsets of a level that will be expanded
__device__ __forceinline__ void plan_offsets(Plan *P, DLevel &L) {
    L.off = nullptr;
    L.tiles = nullptr;
    if (L.n == 0) return;
    L.off = (u64 *)plan_alloc(P, (L.n + 1) * 8);
    L.tiles = L.off ? (u64 *)plan_alloc(P, ((L.n + GEN_WG - 1) / GEN_WG) * 8) : nullptr;
    if (!L.tiles) L.n = 0;
}

// The first kernel: the plan and the roots come from the host, the roots are
// counted (deeper levels get their counts from the expansion) and the table
// of depth D is probed: hits are resolved before the expansion.  check: the
// leaf counts replies by difference, which not every root allows.
template <int V>
__global__ __launch_bounds__(wg_size<V>()) void kd_begin(Plan *P, const Link *H, TTView tt, int D, TTCounters *ctr,
                                                         int small, int check, Tables t) {
    stage_tables<V>(t);
    if (blockIdx.x == 0) {
        const u64 *from = (const u64 *)&H->plan;
        for (u32 i = threadIdx.x; i < sizeof(Plan) / 8; i += blockDim.x)
            if (i != offsetof(Plan, irregular) / 8) ((u64 *)P)[i] = from[i];
        __syncthreads();
        if (threadIdx.x == 0) {
            P->began = wall_clock64();
            if (!small) plan_offsets(P, P->lv[0]);
        }
    }
    const DLevel L = H->plan.lv[0];
    const u64 bias = H->plan.bias;
    const Pos *const hb = H->b;
    const Key128 *const hk = H->k;
    PG_GRID_LOOP(i, L.n) {
        const Pos b = hb ? hb[i] : L.b[i];
        if (hb) {
            L.b[i] = b;
            if (L.k) L.k[i] = hk[i];
        }
        if (check && !pos_regular(b)) atomicOr(&P->irregular, 1ULL);
        if (small) {
            L.perft[i] = bias;
            continue;
        }
        u64 v = 0;
        const bool probe = D >= 2 && tt.base[D] && L.k;
        const bool hit = probe && tt_probe(tt, D, L.k[i], &v);
        if (ctr) {
            ctr_count(ctr, D, 0, probe);
            ctr_count(ctr, D, 1, hit);
        }
        // the roots are left untouched so that a rerun after an overflow sees
        // the same input; a hit is recorded in state/perft and expands to nothing
        L.state[i] = hit ? ST_HIT : ST_LIVE;
        L.perft[i] = v;
        L.cnt[i] = hit ? 0 : count_any<V>(b, t);
    }
}

// The last kernel, one work-group: results and counters to the host.
static __global__ __launch_bounds__(1024) void kd_end(Plan *P, Link *H) {
    const DLevel L = P->lv[0];
    u64 *const out = H->out;
    if (out)
        for (u64 i = threadIdx.x; i < L.n; i += blockDim.x) out[i] = L.perft[i];
    if (threadIdx.x == 0) {
        Plan &h = H->plan;
        h.overflow = P->overflow;
        h.err = P->err;
        h.ovf = P->ovf;
        h.leafItems = P->leafItems;
        h.peak = P->peak;
        h.irregular = P->irregular;
        P->irregular = 0;
        H->ticks = wall_clock64() - P->began;
    }
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x == 0) __hip_atomic_store(&H->seq, H->want, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// level-0 move counts of a total-only search (the byte-lookup variant)
static __global__ __launch_bounds__(wg_size<SL_BYTE>()) void kd_count(Plan *P, Tables t) {
    stage_tables<SL_BYTE>(t);
    const DLevel L = P->lv[0];
    if (blockIdx.x == 0 && threadIdx.x == 0) plan_offsets(P, P->lv[0]);
    PG_GRID_LOOP(i, L.n) L.cnt[i] = count_any<SL_BYTE>(L.b[i], t);
}

static __global__ __launch_bounds__(256) void kd_root_store(Plan *P, TTView tt, int D, TTCounters *ctr) {
    const DLevel L = P->lv[0];
    if (P->overflow || P->bias) return;  // a biased test total is not a perft
    PG_GRID_LOOP(i, L.n) {
        const bool st = D >= 2 && L.k && L.state[i] == ST_LIVE && tt_store(tt, D, L.k[i], L.perft[i]);
        if (ctr) ctr_count(ctr, D, 2, st);
    }
}

// release the transient arrays of level l (after its children are made)
__device__ __forceinline__ void release_level(Plan *P, int l) {
    DLevel &L = P->lv[l];
    if (P->lv[l + 1].n) P->top = L.release;
    if (!L.keep) {
        L.mv = nullptr;
        L.par = nullptr;
    }
    L.set = nullptr;
}

__device__ void plan_children(Plan *P, int l, int wantKeys, int wantSet, int total, int expand);

// The children before each tile of GEN_WG boards of level l, and the plan of
// level l + 1.  The work-group that arrives last scans the tile sums and
// plans: what it reads was written by atomics that had returned before the
// writer arrived.  (expand: level l + 1 will be expanded in its turn.)
constexpr int PLAN_IPT = 8;
static __global__ __launch_bounds__(GEN_WG) void kd_scan(Plan *P, int l, int wantKeys, int wantSet, int total, int expand) {
    __shared__ u32 last;
    constexpr u32 WAVES = GEN_WG / 64;
    const u32 tid = threadIdx.x, lane = tid & 63;
    const DLevel L = P->lv[l];
    const u64 tiles = (L.n + GEN_WG - 1) / GEN_WG;
    // work-groups without a tile do not take part (arrivals take 6 ns each)
    const u64 need = tiles ? (tiles + WAVES - 1) / WAVES : 1;
    const u32 members = need < gridDim.x ? (u32)need : gridDim.x;
    if (blockIdx.x >= members) return;
    for (u64 tile = (u64)blockIdx.x * WAVES + wave_number(); tile < tiles; tile += (u64)members * WAVES) {
        u32 c = 0;
#pragma unroll
        for (u32 k = 0; k < WAVES; k++) {
            const u64 i = tile * GEN_WG + k * 64 + lane;
            c += i < L.n ? L.cnt[i] : 0;
        }
        const u64 sum = wave_sum32(c);
        if (lane == 0) __hip_atomic_store(&L.tiles[tile], sum, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (tid == 0) last = atomicAdd(&P->arrived[l], 1u) + 1 == members;
    __syncthreads();
    if (!last) return;
    u64 carry = 0;
    for (u64 first = 0; first < tiles; first += GEN_WG * PLAN_IPT) {
        const u64 at = first + tid * PLAN_IPT;
        u64 v[PLAN_IPT], sum = 0;
#pragma unroll
        for (int j = 0; j < PLAN_IPT; j++) {
            v[j] = at + j < tiles ? __hip_atomic_load(&L.tiles[at + j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0;
            sum += v[j];
        }
        u64 all;
        u64 run = carry + block_excl_scan<GEN_WG>(sum, &all);
#pragma unroll
        for (int j = 0; j < PLAN_IPT; j++) {
            if (at + j < tiles) L.tiles[at + j] = run;
            run += v[j];
        }
        carry += all;
    }
    if (tid == 0) {
        P->lv[l].kids = carry;
        if (l > 0) release_level(P, l - 1);
        plan_children(P, l, wantKeys, wantSet, total, expand);
    }
}

// The offsets of a tile's boards' children (all threads): this thread's board
// is number first + threadIdx.x; returns its offset and *c, its count.
__device__ __forceinline__ u64 tile_offsets(const DLevel &L, u64 first, u32 *c) {
    const u64 i = first + threadIdx.x;
    *c = i < L.n ? L.cnt[i] : 0;
    u64 sum;
    const u64 o = L.tiles[first / GEN_WG] + block_excl_scan<GEN_WG>(*c, &sum);
    if (i < L.n) L.off[i] = o;
    if (i + 1 == L.n) L.off[L.n] = o + *c;
    return o;
}
// the offsets for the byte-lookup variant, whose tables leave the generate
// kernel no room for a scan
static __global__ __launch_bounds__(GEN_WG) void kd_offsets(Plan *P, int l) {
    const DLevel L = P->lv[l];
    if (P->lv[l + 1].n == 0) return;
    u32 c;
    for (u64 first = (u64)blockIdx.x * GEN_WG; first < L.n; first += (u64)gridDim.x * GEN_WG) (void)tile_offsets(L, first, &c);
}

// allocate level l+1 (children of l) and the transient arrays; a total-only
// search (total == 1) keeps just boards and counts per level.
// total == 3: the last level of a search with per-board results and keys
// keeps no boards or counts, only keys, perfts, states and owners; the moves
// and parents stay until the leaf, which makes the children from them.
__device__ void plan_children(Plan *P, int l, int wantKeys, int wantSet, int total, int expand) {
    DLevel &L = P->lv[l];
    DLevel &C = P->lv[l + 1];
    memset(&C, 0, sizeof(C));
    L.keep = 0;
    const u64 m = L.n ? L.kids : 0;
    if (m == 0 || m > 0xFFFFFFFFULL || P->irregular) {
        if (m) P->overflow = 1;
        return;
    }
    if (total == 3) {
        C.perft = (u64 *)plan_alloc(P, m * 8);
        C.state = (u8 *)plan_alloc(P, m);
        C.dup = (u32 *)plan_alloc(P, m * 4);
        C.k = (Key128 *)plan_alloc(P, m * sizeof(Key128));
        L.mv = (u16 *)plan_alloc(P, m * 2);
        L.par = (u32 *)plan_alloc(P, m * 4);
        L.keep = 1;
        L.release = P->top;  // only the set goes after the expansion
        if (wantSet) {
            u64 s = 1;
            while (s < 2 * m) s <<= 1;
            L.set = (u32 *)plan_alloc(P, s * 4);
            L.setMask = s - 1;
        }
        if (P->overflow) {
            memset(&C, 0, sizeof(C));
            return;
        }
        C.n = m;
        return;
    }
    C.b = (Pos *)plan_alloc(P, m * sizeof(Pos));
    C.cnt = (u32 *)plan_alloc(P, m * 4);
    if (!total) {
        C.perft = (u64 *)plan_alloc(P, m * 8);
        C.state = (u8 *)plan_alloc(P, m);
        C.dup = (u32 *)plan_alloc(P, m * 4);
    }
    if (wantKeys) C.k = (Key128 *)plan_alloc(P, m * sizeof(Key128));
    C.n = m;
    if (expand) plan_offsets(P, C);
    L.release = P->top;
    L.mv = (u16 *)plan_alloc(P, m * 2);
    L.par = (u32 *)plan_alloc(P, m * 4);
    if (wantSet) {
        u64 s = 1;
        while (s < 2 * m) s <<= 1;
        L.set = (u32 *)plan_alloc(P, s * 4);
        L.setMask = s - 1;
    }
    if (P->overflow) {
        memset(&C, 0, sizeof(C));
        return;
    }
    C.n = m;
}

// the moves of level l, and its duplicate set emptied (graphs get no memset
// nodes)
template <int V>
__global__ __launch_bounds__(wg_size<V>()) void kd_generate(Plan *P, int l, Tables t) {
    stage_tables<V>(t);
    const DLevel L = P->lv[l];
    if (P->lv[l + 1].n == 0) return;
    if (L.set) PG_GRID_LOOP(i, L.setMask + 1) L.set[i] = 0;
    if constexpr (V == SL_BYTE) {
        PG_GRID_LOOP(i, L.n) {
            const u64 o = L.off[i];
            const u32 room = (u32)(L.off[i + 1] - o);
            if (room == 0) continue;
            const u32 c = generate_any<V>(L.b[i], t, L.mv + o, room);
            if (c != room) P->err = 1;
            for (u32 j = 0; j < room; j++) L.par[o + j] = (u32)i;
        }
    } else {
        generate_tiles<V>(L.b, L.n, L.mv, L.par, &P->err, t, [&](u64 first, u32 *c) { return tile_offsets(L, first, c); });
    }
}

// children: make (with key), probe the child depth's table, count moves
template <int V>
__global__ __launch_bounds__(wg_size<V>()) void kd_expand(Plan *P, int l, TTView tt, int rc, TTCounters *ctr, Tables t) {
    stage_tables<V>(t);
    const DLevel L = P->lv[l];
    const DLevel C = P->lv[l + 1];
    PG_GRID_LOOP(i, C.n) {
        const u32 pi = L.par[i];
        Pos p = L.b[pi];
        u64 v = 0;
        bool hit = false;
        if (C.k) {
            Key128 h = L.k[pi];
            make_any_hash(p, L.mv[i], h, t);
            C.k[i] = h;
            const bool probe = rc >= 2 && tt.base[rc];
            hit = probe && tt_probe(tt, rc, h, &v);
            if (ctr) {
                ctr_count(ctr, rc, 0, probe);
                ctr_count(ctr, rc, 1, hit);
            }
        } else {
            make_any(p, L.mv[i], t);
        }
        C.cnt[i] = hit ? 0 : count_any<V>(p, t);
        C.b[i] = p;
        if (C.state) {  // absent in a total-only search
            C.state[i] = hit ? ST_HIT : ST_LIVE;
            C.perft[i] = v;
            C.dup[i] = (u32)i;
        }
    }
}

// the last level when it keeps keys only (plan_children, total == 3): each
// child is made in registers for its key and its table probe
template <int V>
__global__ __launch_bounds__(wg_size<V>()) void kd_expand_keys(Plan *P, int l, TTView tt, int rc, TTCounters *ctr,
                                                      Tables t) {
    stage_tables<V>(t);
    const DLevel L = P->lv[l];
    const DLevel C = P->lv[l + 1];
    PG_GRID_LOOP(i, C.n) {
        const u32 pi = L.par[i];
        Pos p = L.b[pi];
        Key128 h = L.k[pi];
        make_any_hash(p, L.mv[i], h, t);
        u64 v = 0;
        const bool probe = rc >= 2 && tt.base[rc];
        const bool hit = probe && tt_probe(tt, rc, h, &v);
        if (ctr) {
            ctr_count(ctr, rc, 0, probe);
            ctr_count(ctr, rc, 1, hit);
        }
        C.k[i] = h;
        C.state[i] = hit ? ST_HIT : ST_LIVE;
        if (hit) C.perft[i] = v;  // the leaf writes the live children's; duplicates have their owners'
    }
}

// equal children of level l+1 when their boards are not stored: both made
// again from parent and move
__device__ __forceinline__ bool same_child(const DLevel &L, u64 a, u64 b, const Tables &t) {
    Pos pa = L.b[L.par[a]], pb = L.b[L.par[b]];
    make_any(pa, L.mv[a], t);
    make_any(pb, L.mv[b], t);
    return same_board(pa, pb);
}

// one child after its first probe (kd_dedup): follow the probe sequence
// until the child owns a slot or finds its equal
__device__ __forceinline__ void kd_dedup_finish(Plan *P, const DLevel &L, const DLevel &C, u64 i, bool live, u64 s,
                                                u32 cur, bool look, TTCounters *ctr, int rc, int keyOnly, const Tables &t) {
    bool isDup = false;
    if (live) {
        for (u64 step = 0;; step++) {
            if (cur == 0) break;
            const u32 o = cur - 1;
            if (C.k[o].lo == C.k[i].lo && C.k[o].hi == C.k[i].hi &&
                (keyOnly || (C.b ? same_board(C.b[o], C.b[i]) : same_child(L, o, i, t)))) {
                C.dup[i] = o;
                isDup = true;
                break;
            }
            if (step >= L.setMask) { P->err = 3; break; }
            s = (s + 1) & L.setMask;
            cur = slot_claim(&L.set[s], look ? slot_look(&L.set[s]) : 0, (u32)i + 1);
        }
    }
    if (ctr) ctr_count(ctr, rc, 3, isDup);
    if (isDup) {
        C.state[i] = ST_DUP;
        if (C.cnt) C.cnt[i] = 0;  // a level that keeps keys only has no counts
    }
}

// in-level duplicates of level l+1 (as k_dedup: two children per thread,
// both first probes in flight).  keyOnly (a search with a table, which
// accepts hits on the 128-bit key): equal keys are equal positions; without
// a table the boards are compared as well.
static __global__ __launch_bounds__(256) void kd_dedup(Plan *P, int l, TTCounters *ctr, int rc, int keyOnly, Tables t) {
    const DLevel L = P->lv[l];
    const DLevel C = P->lv[l + 1];
    if (!L.set) return;
    const u64 stride = (u64)gridDim.x * blockDim.x;
    // A set that the caches hold is claimed without a look first: the swap
    // waits less there, and the look is one more access in a row (32 MB set,
    // divide of an opening at depth 7: 1134 us per call without, 1170 with;
    // 1 GB set, 4096 positions at depth 5: 46.0 ms without, 45.2 with).
    const bool look = L.setMask >= 1u << 25;
    for (u64 i0 = (u64)blockIdx.x * blockDim.x + threadIdx.x; i0 < C.n; i0 += 2 * stride) {
        const u64 i1 = i0 + stride;
        const bool has1 = i1 < C.n;
        const bool l0 = C.state[i0] == ST_LIVE, l1 = has1 && C.state[i1] == ST_LIVE;
        const u64 s0 = (C.k[i0].lo >> 7) & L.setMask, s1 = l1 ? (C.k[i1].lo >> 7) & L.setMask : 0;
        u32 c0 = l0 && look ? slot_look(&L.set[s0]) : 0, c1 = l1 && look ? slot_look(&L.set[s1]) : 0;
        if (l0) c0 = slot_claim(&L.set[s0], c0, (u32)i0 + 1);
        if (l1) c1 = slot_claim(&L.set[s1], c1, (u32)i1 + 1);
        kd_dedup_finish(P, L, C, i0, l0, s0, c0, look, ctr, rc, keyOnly, t);
        if (has1) kd_dedup_finish(P, L, C, i1, l1, s1, c1, look, ctr, rc, keyOnly, t);
    }
}

// The live list of the leaf level l (as k_live_count / k_live_write, in one
// pass): boards resolved from the table or collapsed into an equal board
// have count 0, so the fused leaf runs over the boards with moves only.  A
// live board without moves gets its perft(2) = base here.  kd_plan_live
// makes room for the list (none: the leaf takes every board); each
// work-group lists a chunk of boards in order at an offset it reserves with
// one atomic, so chunks land in any order.
static __global__ void kd_plan_live(Plan *P, int l) {
    if (threadIdx.x || blockIdx.x) return;
    if (l > 0) release_level(P, l - 1);  // the moves, parents and set that made level l
    DLevel &L = P->lv[l];
    if (P->irregular) {
        P->overflow = 1;
        L.n = 0;
    }
    P->liveN = 0;
    L.live = L.n && L.n <= 0xFFFFFFFFULL ? (u32 *)plan_try_alloc(P, L.n * 4) : nullptr;
}

static __global__ __launch_bounds__(LIVE_WG) void kd_live(Plan *P, int l) {
    const DLevel L = P->lv[l];
    if (!L.live) return;
    __shared__ u64 sBase;
    const u64 base = l == 0 ? P->bias : 0;
    const u64 chunks = (L.n + LIVE_CHUNK - 1) / LIVE_CHUNK;
    for (u64 ch = blockIdx.x; ch < chunks; ch += gridDim.x) {
        // each thread takes LIVE_PER_THREAD consecutive boards, so the list
        // keeps the level's order (siblings stay neighbours in the leaf)
        const u64 first = ch * LIVE_CHUNK + (u64)threadIdx.x * LIVE_PER_THREAD;
        u32 f = 0, c = 0;
#pragma unroll
        for (int k = 0; k < LIVE_PER_THREAD; k++) {
            const u64 i = first + k;
            if (!L.cnt) {  // a level that keeps keys only: its live children, counted by the leaf
                const bool lv = i < L.n && L.state[i] == ST_LIVE;
                if (lv) f |= 1u << k;
                c += lv;
                continue;
            }
            const u32 n = i < L.n ? L.cnt[i] : 0;
            if (n) f |= 1u << k;
            c += n != 0;
            if (i < L.n && n == 0 && L.state[i] == ST_LIVE) L.perft[i] = base;
        }
        u64 total;
        const u64 pos = block_excl_scan<LIVE_WG>(c, &total);
        if (threadIdx.x == 0) sBase = total ? atomicAdd((unsigned long long *)&P->liveN, total) : 0;
        __syncthreads();
        u64 at = sBase + pos;
        for (; f; f &= f - 1) L.live[at++] = (u32)(first + __builtin_ctz(f));
        __syncthreads();
    }
}

// perft(2) of the boards of level l, fused (see leaf_tiles), per board into
// the level's perft array
template <int V, bool PLAIN>
__global__ PG_LEAF_BOUNDS void kd_leaf(Plan *P, int l, Tables t) {
    const DLevel L = P->lv[l];
    const bool listed = L.live;
    leaf_tiles<V, true, false, PLAIN>(L.b, L.cnt, listed ? P->liveN : L.n, &P->acc, &P->leafItems, L.perft, L.state,
                                      l == 0 ? P->bias : 0, &P->err, &P->ovf, t, listed ? L.live : nullptr);
}

// perft(2) of the children of level l-1 that form level l when level l keeps
// keys only: the leaf makes each listed child from its parent and move (or,
// without room for the list, every child, writing the live ones)
template <int V, bool PLAIN>
__global__ PG_LEAF_BOUNDS void kd_leaf_keys(
    Plan *P, int l, Tables t) {
    const DLevel L = P->lv[l];
    const DLevel A = P->lv[l - 1];
    const bool listed = L.live != nullptr;
    leaf_tiles<V, true, true, PLAIN>(A.b, nullptr, listed ? P->liveN : L.n, &P->acc, &P->leafItems, L.perft,
                                     listed ? nullptr : L.state, 0, &P->err, &P->ovf, t, listed ? L.live : nullptr,
                                     A.par, A.mv);
}

// Small searches without a table (depth 3 or 4): no levels in memory.  What the
// level loop spends on such a search is mostly its kernels of 3 to 5 us each,
// four per level and more.  kd_begin has set the results to the bias.  A board
// with more moves than a wave's list holds raises overflow, and the host runs
// the level loop.
//
// kd_tiny: so few roots that every board of ply D-2 can have a wave of its own
// (wave_perft2).
template <int V, int D>
__global__ __launch_bounds__(LEAF_WG) void kd_tiny(Plan *P, Tables t) {
    constexpr u32 WAVES = LEAF_WG / 64, PARTS = 32;
    __shared__ u32 list[WAVES][3][WAVE_LIST];
    __shared__ u32 items;
    const u32 wave = wave_number(), lane = threadIdx.x & 63;
    u32(&ls)[3][WAVE_LIST] = list[wave];
    if (threadIdx.x == 0) items = 0;
    __syncthreads();
    const DLevel L = P->lv[0];
    const u64 n = P->irregular ? 0 : L.n, units = uniform64(n) * (D == 3 ? PARTS : PARTS * PARTS);
    u32 listed = 0;
    for (u64 u = blockIdx.x * WAVES + wave; u < units; u += gridDim.x * WAVES) {
        const u64 ri = u / (units / L.n);
        const u32 part = (u32)(u % PARTS), part2 = (u32)(u / PARTS % PARTS);
        const Pos root = uniform_pos(L.b[ri]);
        const u32 n = wave_words<V>(root, t, ls[0], WAVE_LIST, &P->overflow);
        wave_sync();
        u32 sum = 0, moves;
        for (u32 i = part; i < n; i += PARTS) {
            const Pos c = wave_made(root, ls[0], i, t);
            if constexpr (D == 3) {
                sum += wave_perft2<V>(c, ls[1], &moves, &P->overflow, t);
                listed += moves;
            } else {
                const u32 m = wave_words<V>(c, t, ls[1], WAVE_LIST, &P->overflow);
                wave_sync();
                for (u32 j = part2; j < m; j += PARTS) {
                    sum += wave_perft2<V>(wave_made(c, ls[1], j, t), ls[2], &moves, &P->overflow, t);
                    listed += moves;
                }
            }
        }
        sum = wave_sum32(sum);
        if (lane == 0 && sum) add_checked(&P->lv[0].perft[ri], sum, &P->ovf);
        wave_sync();
    }
    if (lane == 0) atomicAdd(&items, listed);
    __syncthreads();
    if (threadIdx.x == 0 && items) atomicAdd(&P->leafItems, (u64)items);
}

// kd_small: a wave takes a part of a root's moves, lists the boards of ply D-2
// below them, a tile at a time (wave_words lists one board's moves), and hands
// the tile to the fused leaf.
template <int V, int D>
__global__ __launch_bounds__(LEAF_WG) __attribute__((amdgpu_waves_per_eu(2, 8))) void kd_small(Plan *P, Tables t) {
    static_assert(D == 3 || D == 4, "two plies end in the leaf");
    constexpr u32 WAVES = LEAF_WG / 64, MOST = D == 3 ? 8 : 32;
    __shared__ LeafTile tiles[WAVES];
    const u32 wave = wave_number(), lane = threadIdx.x & 63;
    LeafTile &s = tiles[wave];
    const u64 n = uniform64(P->irregular ? 0 : P->lv[0].n);
    const u32 waves = gridDim.x * WAVES < LEAF_RESIDENT ? gridDim.x * WAVES : LEAF_RESIDENT;
    u32 parts = 1;
    while (parts < MOST && n * parts * 2 <= waves) parts *= 2;
    u64 items = 0;
    for (u64 u = blockIdx.x * WAVES + wave; u < n * parts; u += gridDim.x * WAVES) {
        const u64 ri = u / parts;
        const u32 part = (u32)(u % parts);
        // read again for each listing: no registers to keep it in
        const Pos *const rp = P->lv[0].b + ri;
        u32 lo = 0, hi = 1, mine = 0, at = 0;
        u32 chunk = 0, rootMoves = 0;  // D == 4: the part's moves, 64 at a time, one in each lane
        do {
            if (D == 4) {
                rootMoves = wave_words<V>(opaque_pos(uniform_pos(*rp)), t, s.word, LEAF_CAP, &P->overflow);
                wave_sync();
                lo = rootMoves * part / parts + chunk;
                hi = rootMoves * (part + 1) / parts;
                if (lo + lane < hi) mine = s.word[lo + lane];
                wave_sync();
                if (hi > lo + 64) hi = lo + 64;
                hi = hi > lo ? hi - lo : 0;
                lo = 0;
            }
            // lo: the next board to list, at: its next move
            for (;;) {
                u32 fill = 0;
                Pos b{};
                while (fill < 64 && lo < hi) {
                    Pos p = opaque_pos(uniform_pos(*rp));
                    if (D == 4) {
                        const u32 w = (u32)__builtin_amdgcn_readlane((int)mine, (int)lo);
                        p = made(p, (u16)w, piece_code(w >> 24), t);
                    }
                    u32 m = wave_words<V>(p, t, s.word, LEAF_CAP, &P->overflow);
                    wave_sync();
                    if (D == 3) {
                        if (at == 0) at = m * part / parts;
                        m = m * (part + 1) / parts;
                    }
                    const u32 take = m - at < 64 - fill ? m - at : 64 - fill;
                    if (lane >= fill && lane < fill + take) {
                        const u32 w = s.word[at + lane - fill];
                        b = made(p, (u16)w, piece_code(w >> 24), t);
                    }
                    wave_sync();
                    fill += take;
                    at += take;
                    if (at >= m) {
                        lo++;
                        at = 0;
                    }
                }
                if (!fill) break;
                const u32 c = leaf_expand<V>(s, lane < fill, b, &P->err, t);
                items += wave_sum32(c);
                const u32 sum = wave_sum32(lane < fill ? s.per[lane] : 0);
                if (lane == 0) add_checked(&P->lv[0].perft[ri], sum, &P->ovf);
                wave_sync();
            }
            chunk += 64;
        } while (D == 4 && rootMoves * part / parts + chunk < rootMoves * (part + 1) / parts);
    }
    if (lane == 0 && items) atomicAdd(&P->leafItems, items);
}

// the plan's total += the move counts of level l (perft(1) of a total-only search)
static __global__ __launch_bounds__(256) void kd_sum_counts(Plan *P, int l) {
    const DLevel L = P->lv[l];
    u64 s = 0;
    PG_GRID_LOOP(i, L.n) s += L.cnt[i];
    s = wave_sum(s);
    if ((threadIdx.x & 63) == 0 && s) add_checked(&P->acc, s, &P->ovf);
}

static __global__ __launch_bounds__(256) void kd_perft1(Plan *P, int l) {
    const DLevel L = P->lv[l];
    const u64 base = l == 0 ? P->bias : 0;
    PG_GRID_LOOP(i, L.n) {
        if (L.state[i] != ST_LIVE) continue;
        const u64 v = base + L.cnt[i];
        if (v < base) P->ovf = 1;
        L.perft[i] = v;
    }
}

// level l's perfts from those of level l+1 (see k_up; rc: its remaining depth)
static __global__ __launch_bounds__(UP_WG) void kd_up(Plan *P, int l, TTView tt, int rc, TTCounters *ctr) {
    const DLevel L = P->lv[l];
    const DLevel C = P->lv[l + 1];
    if (P->overflow) return;
    const u64 base = l == 0 ? P->bias : 0;
    if (C.n == 0) {  // no moves at all, and no offsets
        PG_GRID_LOOP(i, L.n) if (L.state[i] == ST_LIVE) L.perft[i] = base;
        return;
    }
    const bool store = C.k && rc >= 2 && tt.base[rc];
    sum_children(L.n, L.off, base,
        [&](u64 j) {
            const u8 st = C.state[j];
            const u64 v = C.perft[st == ST_DUP ? C.dup[j] : j];
            bool stored = false;
            if (store && st == ST_LIVE) stored = tt_store(tt, rc, C.k[j], v);
            if (ctr) ctr_count(ctr, rc, 2, stored);
            return v;
        },
        [&](u64 i, u64 s, bool wide) {
            if (L.state[i] != ST_LIVE) return;
            L.perft[i] = s;
            if (wide) P->ovf = 1;
        });
}

}  // namespace pg
