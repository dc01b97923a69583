// kernels.h -- gfx950 kernels of the breadth-first perft.
//
// One level of the tree is expanded by four kernels (the reference's level
// loop, perft_bb.h:1071-1135, without device-side launches):
//   k_count     moves per board                        (countMoves)
//   scan        exclusive prefix sum of the counts     (ScanD, scan.cuh:329)
//   k_generate  move list + parent index per child     (generateMoves +
//               IntervalExpandDGenValues folded together, intervalmove.cuh:404)
//   k_expand    child board = make(parent, move), and the child's move count
//               (makemove_and_count_moves_single_level, perft_bb.h:601)
// and the last two plies by
//   k_leaf      sum over (parent, move) of countMoves(make(parent, move))
//               (makeMove_and_perft_single_level_indices, perft_bb.h:412)
// All kernels are grid-stride loops sized to the CU count, so one launch
// covers a level of any size; indices are 64-bit.
#pragma once
#include <type_traits>
#include "movegen.h"

namespace pg {

constexpr int kByteLdsBytes = FANCY_TABLE_SIZE + (BYTE_ROOK_SIZE + BYTE_BISHOP_SIZE) * 8 + 2 * 64 * 16 + 2 * 64 * 8;

__device__ __forceinline__ u64 wave_sum(u64 v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// *acc += s, raising *ovf when the 64-bit total wraps (a perft count that
// does not fit u64 is reported, never returned wrapped).  A wave's own sum
// cannot wrap: it counts at most a few million moves per lane.
__device__ __forceinline__ void add_checked(u64 *acc, u64 s, u32 *ovf) {
    const u64 old = atomicAdd(acc, s);
    if (old + s < old) atomicOr(ovf, 1u);
}

// per-call device state reset without memset nodes: total (with an optional
// starting bias), consumed leaf items, error and overflow flags
static __global__ void k_init_call(u64 *acc, u64 bias, u64 *items, u32 *err, u32 *ovf) {
    if (threadIdx.x || blockIdx.x) return;
    acc[0] = bias;
    acc[1] = 0;
    if (items) *items = 0;
    *err = 0;
    *ovf = 0;
}

// P[i] += base for n values, raising *ovf on a wrap (the count-bias test
// hook where a root's perft is not produced by a checked sum)
static __global__ void k_add_base(u64 *P, u64 n, u64 base, u32 *ovf) {
    for (u64 i = threadIdx.x; i < n; i += blockDim.x) {
        const u64 v = P[i] + base;
        if (v < base) *ovf = 1;
        P[i] = v;
    }
}

template <class T>
__device__ __forceinline__ void lds_copy(T *dst, const T *src, int count) {
    // 16-byte chunks; every table here is a multiple of 16 bytes
    const uint4 *s = reinterpret_cast<const uint4 *>(src);
    uint4 *d = reinterpret_cast<uint4 *>(dst);
    const int chunks = (int)(count * sizeof(T) / 16);
    for (int i = threadIdx.x; i < chunks; i += blockDim.x) d[i] = s[i];
}

// The byte-lookup variant keeps its whole working set (147 KiB) in LDS; the
// other variants read their tables through the L1/L2 caches.
template <int V>
__device__ __forceinline__ void stage_tables(Tables &t) {
    if constexpr (V == SL_BYTE) {
        __shared__ __align__(16) u8 sIdx[FANCY_TABLE_SIZE];
        __shared__ __align__(16) u64 sRook[BYTE_ROOK_SIZE];
        __shared__ __align__(16) u64 sBishop[BYTE_BISHOP_SIZE];
        __shared__ __align__(16) FancyEntry sRF[64], sBF[64];
        __shared__ __align__(16) u64 sRM[64], sBM[64];
        lds_copy(sIdx, t.byteIdx, FANCY_TABLE_SIZE);
        lds_copy(sRook, t.byteRook, BYTE_ROOK_SIZE);
        lds_copy(sBishop, t.byteBishop, BYTE_BISHOP_SIZE);
        lds_copy(sRF, t.rookFancy, 64);
        lds_copy(sBF, t.bishopFancy, 64);
        lds_copy(sRM, t.rookMask, 64);
        lds_copy(sBM, t.bishopMask, 64);
        __syncthreads();
        t.byteIdx = sIdx;
        t.byteRook = sRook;
        t.byteBishop = sBishop;
        t.rookFancy = sRF;
        t.bishopFancy = sBF;
        t.rookMask = sRM;
        t.bishopMask = sBM;
    }
}

template <int V> constexpr int wg_size() { return V == SL_BYTE ? 1024 : 256; }

#define PG_GRID_LOOP(i, n) \
    for (u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x; i < (n); i += (u64)gridDim.x * blockDim.x)

// number of legal moves of a board after one move, side-resolved once
template <int V>
__device__ __forceinline__ u32 count_after(Pos p, u16 mv, const Tables &t) {
    if (pos_side(p)) {
        make_move<BLACK, false>(p, mv, nullptr, t);
        return count_moves<WHITE, V>(p, t);
    }
    make_move<WHITE, false>(p, mv, nullptr, t);
    return count_moves<BLACK, V>(p, t);
}
template <int V>
__global__ __launch_bounds__(wg_size<V>()) void k_count(const Pos *__restrict__ b, u64 n, u32 *__restrict__ cnt, Tables t) {
    stage_tables<V>(t);
    PG_GRID_LOOP(i, n) cnt[i] = count_any<V>(b[i], t);
}

template <int V>
__global__ __launch_bounds__(wg_size<V>()) void k_count_sum(const Pos *__restrict__ b, u64 n, u64 *acc, u32 *ovf, Tables t) {
    stage_tables<V>(t);
    u64 s = 0;
    PG_GRID_LOOP(i, n) s += count_any<V>(b[i], t);
    s = wave_sum(s);
    if ((threadIdx.x & 63) == 0 && s) add_checked(acc, s, ovf);
}

static __global__ __launch_bounds__(256) void k_sum_u32(const u32 *__restrict__ c, u64 n, u64 *acc, u32 *ovf) {
    u64 s = 0;
    PG_GRID_LOOP(i, n) s += c[i];
    s = wave_sum(s);
    if ((threadIdx.x & 63) == 0 && s) add_checked(acc, s, ovf);
}

// Move lists and parent indices of boards [0, n) whose exclusive child
// offsets are off[0..n].  A work-group takes 256 consecutive boards, whose
// children form one contiguous output range: the boards generate into an LDS
// window (WordSink), then the work-group stores the window
// one lane per slot, so the HBM writes are coalesced and each byte is written
// once.  Boards that do not fit the window wait for the next pass.  err is
// set to 1 if a board generates a different number of moves than it counted
// (the two must agree for the level layout to be valid).
constexpr int GEN_WG = 256, GEN_WINDOW = 8192;

// offsets(first, &c): the offset of board first + threadIdx.x and its count
// (0: no moves, or resolved earlier)
template <int V, class Offsets>
__device__ __forceinline__ void generate_tiles(const Pos *__restrict__ b, u64 n, u16 *__restrict__ moves,
                                               u32 *__restrict__ parent, u32 *err, const Tables &t, Offsets &&offsets) {
    __shared__ u32 word[GEN_WINDOW];
    __shared__ u32 snext, stotal;
    __shared__ u64 sbase;
    const int tid = threadIdx.x;
    for (u64 tile = blockIdx.x; tile * GEN_WG < n; tile += gridDim.x) {
        const u64 first = tile * GEN_WG;
        const u64 i = first + tid;
        u32 c;
        const u64 off = offsets(first, &c);
        if (tid == 0) sbase = off;
        __syncthreads();
        const u64 base = sbase;
        const u32 pos = (u32)(off - base);
        if (tid == GEN_WG - 1) stotal = pos + c;
        __syncthreads();
        const u32 total = stotal;
        u32 start = 0;
        while (start < total) {
            const u32 end = start + GEN_WINDOW;
            if (tid == 0) snext = total;
            __syncthreads();
            if (c && pos >= start && pos + c <= end) {
                const u32 g = generate_words<V>(b[i], t, word + (pos - start), c, (u32)tid);
                if (g != c) *err = 1;
            } else if (c && pos >= start) {
                atomicMin(&snext, pos);
            }
            __syncthreads();
            const u32 wend = snext;
            for (u32 j = start + tid; j < wend; j += GEN_WG) {
                const u32 w = word[j - start];
                moves[base + j] = (u16)w;
                parent[base + j] = (u32)first + (w >> 16 & 255u);
            }
            __syncthreads();
            start = wend;
        }
    }
}

template <int V>
__global__ __launch_bounds__(wg_size<V>()) void k_generate(const Pos *__restrict__ b, u64 n, const u64 *__restrict__ off,
                                                           u16 *__restrict__ moves, u32 *__restrict__ parent, u32 *err,
                                                           Tables t) {
    stage_tables<V>(t);
    if constexpr (V == SL_BYTE) {
        // the byte-lookup tables fill the LDS: each lane writes its own list
        PG_GRID_LOOP(i, n) {
            const u64 o = off[i];
            const u32 room = (u32)(off[i + 1] - o);
            if (room == 0) continue;
            const u32 c = generate_any<V>(b[i], t, moves + o, room);
            if (c != room) *err = 1;
            for (u32 j = 0; j < room; j++) parent[o + j] = (u32)i;
        }
    } else {
        generate_tiles<V>(b, n, moves, parent, err, t, [&](u64 first, u32 *c) {
            const u64 i = first + threadIdx.x;
            *c = i < n ? (u32)(off[i + 1] - off[i]) : 0;
            return off[i < n ? i : n];
        });
    }
}

template <int V>
__global__ __launch_bounds__(wg_size<V>()) void k_expand(const Pos *__restrict__ parents, const u32 *__restrict__ pidx,
                                                         const u16 *__restrict__ moves, u64 m, Pos *__restrict__ children,
                                                         u32 *__restrict__ cnt, Tables t) {
    stage_tables<V>(t);
    PG_GRID_LOOP(i, m) {
        Pos p = parents[pidx[i]];
        make_any(p, moves[i], t);
        children[i] = p;
        cnt[i] = count_any<V>(p, t);
    }
}

template <int V>
__global__ __launch_bounds__(wg_size<V>()) void k_leaf(const Pos *__restrict__ parents, const u32 *__restrict__ pidx,
                                                       const u16 *__restrict__ moves, u64 m, u64 *acc, u32 *ovf, Tables t) {
    stage_tables<V>(t);
    u64 s = 0;
    PG_GRID_LOOP(i, m) s += count_after<V>(parents[pidx[i]], moves[i], t);
    s = wave_sum(s);
    if ((threadIdx.x & 63) == 0 && s) add_checked(acc, s, ovf);
}

// ---------------------------------------------------------------- scan helpers
constexpr int SCAN_WG = 256, SCAN_IPT = 8, SCAN_TILE = SCAN_WG * SCAN_IPT;

__device__ __forceinline__ u64 wave_incl_scan(u64 v) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const u64 y = __shfl_up(v, o, 64);
        if (lane >= o) v += y;
    }
    return v;
}

// exclusive scan across the work-group; *total gets the group sum
template <int WG>
__device__ __forceinline__ u64 block_excl_scan(u64 v, u64 *total) {
    __shared__ u64 waveTot[WG / 64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const u64 incl = wave_incl_scan(v);
    if (lane == 63) waveTot[w] = incl;
    __syncthreads();
    u64 base = 0, tot = 0;
#pragma unroll
    for (int i = 0; i < WG / 64; i++) {
        const u64 x = waveTot[i];
        if (i < w) base += x;
        tot += x;
    }
    __syncthreads();
    *total = tot;
    return base + incl - v;
}

// ---------------------------------------------------------------- sets
// What a set's slot holds before it is claimed for `mine` (0: it was empty and
// is now mine).  A slot is looked at first: a compare-and-swap that finds it
// taken is as dear as one that claims it, and those of equal items queue on
// one address.  With 2.5 items per value a set of 30 M items takes 43 ps per
// item this way and 93 without the look (48 when no two are equal).  A look
// may see a claimed slot as still empty; the swap then finds out.
template <class T> __device__ __forceinline__ T slot_look(const T *slot) {
    return __hip_atomic_load(slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
}
template <class T> __device__ __forceinline__ T slot_claim(T *slot, T seen, T mine) {
    return seen ? seen : atomicCAS(slot, (T)0, mine);
}

// ---------------------------------------------------------------- way back up
// done(i, base + sum of value(j) over i's children j, the sum passed 64 bits)
// for parents [0, n), whose children lie one after the other at off[0..n].
// Bound by memory: a work-group reads the children of 64 parents by
// consecutive lanes into LDS, where each parent's lane adds up its own.  A
// lane per parent that read its children itself, after a pass that copied the
// owners' values to the duplicates, took 3.2 ms for the 136 M children of the
// last level of 4096 positions at depth 5; this takes 1.1.
constexpr int UP_WG = 256, UP_PARENTS = 64, UP_WINDOW = 2048;
template <class Value, class Done>
__device__ __forceinline__ void sum_children(u64 n, const u64 *__restrict__ off, u64 base, Value &&value, Done &&done) {
    __shared__ u64 window[UP_WINDOW];
    __shared__ u64 at[UP_PARENTS + 1];
    const u32 tid = threadIdx.x;
    for (u64 first = (u64)blockIdx.x * UP_PARENTS; first < n; first += (u64)gridDim.x * UP_PARENTS) {
        const u32 np = n - first < UP_PARENTS ? (u32)(n - first) : UP_PARENTS;
        if (tid <= np) at[tid] = off[first + tid];
        __syncthreads();
        const u64 lo = at[0], hi = at[np];
        u64 s = base;
        bool carry = false;
        for (u64 c = lo; c < hi; c += UP_WINDOW) {
            const u64 e = c + UP_WINDOW < hi ? c + UP_WINDOW : hi;
            for (u64 j = c + tid; j < e; j += UP_WG) window[j - c] = value(j);
            __syncthreads();
            if (tid < np) {
                const u64 from = at[tid] > c ? at[tid] : c, to = at[tid + 1] < e ? at[tid + 1] : e;
                for (u64 j = from; j < to; j++) {
                    const u64 x = window[j - c];
                    s += x;
                    carry |= s < x;
                }
            }
            __syncthreads();
        }
        if (tid < np) done(first + tid, s, carry);
        __syncthreads();
    }
}

// ---------------------------------------------------------------- fused leaf
// The last two plies without touching HBM for the (parent, move) items.  A
// wave takes a tile of 64 boards of ply D-2, one per lane, and keeps them as
// kin in LDS, split by side.  Their moves fall into classes (leaf_eval):
//   quiet  neither square matters to any reply: all of a board's quiet moves
//          have the same number of replies, so they are counted, not listed
//   calm   the king's zone and the pins stay as they are: only the sliders,
//          pawns and knights that can reply differently are counted again
//   full   the others: the replies are counted from scratch
// In games from the start 59 to 74 % of the moves of the first twenty plies
// are quiet and 6 to 11 % full; later it is a quarter and a half.  Calm and
// full moves are listed into an LDS window, from its front and from its end,
// and counted a lane per move; boards that do not fit the window are worked
// out again for the next one.  Moves that are more than a piece leaving one
// square for another (castling, promotions, en passant) are put aside by the
// lanes that meet them and counted afterwards through make_move: as a branch
// in the main loop they would hold up nearly every wave.
//
// Bound by the issue of VALU instructions.  From the start position,
// perft(8) without merging (119 M boards, 3.2 G moves of ply 7) takes 20.1 ms,
// 21.9 while all waves took their tiles from one counter, as in the figures
// that follow.  As a count of every reply from a board that each lane made
// itself it took 50.1 ms, the same with the kin in LDS 44.9, and with quiet
// moves as well 23.7.
//
// No work-group barrier: working out the boards (a long chain, no listing)
// and counting the replies overlap between the waves of a SIMD.  Four waves'
// tiles of 7.4 KB of boards and 1488 window words are 53.5 KB, so that three
// work-groups share a CU's 160 KB (which is handed out in pieces of 1280
// bytes: 54.3 KB each no longer fit, 29.5 ms).  A tile of 64 boards lists 400
// to 1700 moves: windows of 608 words take 27.5 ms, 1216 words 23.7, 1408
// words 21.9.  Three waves per SIMD is also what the registers allow; for
// four the compiler spills, for two (209 registers) it takes 28.3 ms.
constexpr int LEAF_WG = 256, LEAF_TILE = 64, LEAF_CAP = 1488, LEAF_BLOCKS_PER_CU = 64;
constexpr u32 LEAF_LATE = 1u << 29;  // window word: a special move that found no room in the aside list

// a value that all lanes hold, in scalar registers
__device__ __forceinline__ u64 uniform64(u64 v) {
    return (u64)(u32)__builtin_amdgcn_readfirstlane((int)(v >> 32)) << 32 | (u32)__builtin_amdgcn_readfirstlane((int)v);
}
// the wave's sum of v, in scalar registers
__device__ __forceinline__ u32 wave_sum32(u32 v) {
    u32 x = v;
    x += (u32)__builtin_amdgcn_update_dpp(0, (int)x, 0x111, 0xF, 0xF, true);  // row_shr 1, 2, 4, 8
    x += (u32)__builtin_amdgcn_update_dpp(0, (int)x, 0x112, 0xF, 0xF, true);
    x += (u32)__builtin_amdgcn_update_dpp(0, (int)x, 0x114, 0xF, 0xF, true);
    x += (u32)__builtin_amdgcn_update_dpp(0, (int)x, 0x118, 0xF, 0xF, true);
    return (u32)(__builtin_amdgcn_readlane((int)x, 15) + __builtin_amdgcn_readlane((int)x, 31) +
                 __builtin_amdgcn_readlane((int)x, 47) + __builtin_amdgcn_readlane((int)x, 63));
}
// p after the move mv of its piece of code `piece`
__device__ __forceinline__ Pos made(Pos p, u16 mv, int piece, const Tables &t) {
    if (pos_side(p)) make_move_as<BLACK, false>(p, mv, piece, nullptr, t);
    else make_move_as<WHITE, false>(p, mv, piece, nullptr, t);
    return p;
}
__device__ __forceinline__ u32 lanes_below(u64 mask) {
    return __builtin_amdgcn_mbcnt_hi((u32)(mask >> 32), __builtin_amdgcn_mbcnt_lo((u32)mask, 0));
}
// orders a wave's LDS accesses (each wave's are carried out in order; this
// keeps the compiler from moving them)
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}
// a board that all lanes hold, in scalar registers
__device__ __forceinline__ Pos uniform_pos(Pos p) {
    u64 w[sizeof(Pos) / 8];
    memcpy(w, &p, sizeof(Pos));
#pragma unroll
    for (u32 i = 0; i < sizeof(Pos) / 8; i++) w[i] = uniform64(w[i]);
    memcpy(&p, w, sizeof(Pos));
    return p;
}

// the same, kept apart from earlier uses: nothing worked out from it stays in
// registers from one use to the next
__device__ __forceinline__ Pos opaque_pos(Pos p) {
    u64 w[sizeof(Pos) / 8];
    memcpy(w, &p, sizeof(Pos));
#pragma unroll
    for (u32 i = 0; i < sizeof(Pos) / 8; i++) asm volatile("" : "+s"(w[i]));
    memcpy(&p, w, sizeof(Pos));
    return p;
}

// The moves of one board listed by a whole wave.  The board is the same in
// all lanes: what concerns all of it is worked out by the scalar unit, and a
// lane works out the piece on its own square, an enemy slider's attacks or
// one's own moves.  One lane that lists a board by itself (generate_words)
// takes about four times as long, for it does one piece after the other.
// Like every writer it counts on past its cap and stores nothing there.
struct WaveSink {
    u32 *word;
    u32 cap, n, lane;
    __device__ void put(u32 at, u32 w) {
        if (at < cap) word[at] = w;
    }
    __device__ void add(u32 m, u32 piece) {
        if (lane == 0) put(n, m | piece << 24);
        n++;
    }
    template <class F> __device__ void squares(u64 m, u64, u32 piece, F &&f) {
        if (m >> lane & 1) put(n + lanes_below(m), f((int)lane) | piece << 24);
        n += (u32)popc(m);
    }
    __device__ void skipped(u64) {}
};
__device__ __forceinline__ u32 wave_or32(u32 x) {
    x |= (u32)__builtin_amdgcn_update_dpp(0, (int)x, 0x111, 0xF, 0xF, true);  // row_shr 1, 2, 4, 8
    x |= (u32)__builtin_amdgcn_update_dpp(0, (int)x, 0x112, 0xF, 0xF, true);
    x |= (u32)__builtin_amdgcn_update_dpp(0, (int)x, 0x114, 0xF, 0xF, true);
    x |= (u32)__builtin_amdgcn_update_dpp(0, (int)x, 0x118, 0xF, 0xF, true);
    return (u32)(__builtin_amdgcn_readlane((int)x, 15) | __builtin_amdgcn_readlane((int)x, 31) |
                 __builtin_amdgcn_readlane((int)x, 47) | __builtin_amdgcn_readlane((int)x, 63));
}
__device__ __forceinline__ u64 wave_or64(u64 x) { return (u64)wave_or32((u32)(x >> 32)) << 32 | wave_or32((u32)x); }

template <int C, int V>
__device__ __forceinline__ void wave_side_words(const Pos &p, const Tables &t, WaveSink &o) {
    const Sides s = sides_of<C>(p);
    const u32 sq = o.lane;
    const u64 here = bit((int)sq);
    const bool rook = (s.myRooks | s.eRooks) & here, bishop = (s.myBishops | s.eBishops) & here, enemy = s.enemy & here;
    const u64 occ = enemy ? s.occ ^ s.myKing : s.occ;  // enemy sliders look through the king
    u64 att = 0;
    if (rook) att = Sl<V>::rook(t, (int)sq, occ);
    if (bishop) att |= Sl<V>::bishop(t, (int)sq, occ);
    MoveCtx x;
    x.threatened = leaper_attacks<C>(s, t) | wave_or64(enemy ? att : 0);
    const KingRow &row = t.row[s.k];
    const bool line = or_and(row.rook & s.eRooks, row.bishop, s.eBishops) & here;
    u64 b = ~0ULL;  // what stands between an enemy slider and the king
    if (line) b = t.pin[s.k << 6 | (int)sq].between & s.occ;
    x.checkers = leaper_checks<C>(s, t, __ballot(b == 0));
    x.pinned = wave_or64(several(b) ? 0 : b) & s.mine;
    x.target = ~s.mine;
    if (x.checkers) x.target &= several(x.checkers) ? 0ULL : x.checkers | t.pin[s.k << 6 | ctz(x.checkers)].between;
    const Gen g{x.pinned, x.checkers, x.target, and_nor(row.king, s.mine, x.threatened), 0, 0, 0, 0, 0, 0, 0, 0, 0,
                castle_moves<C>(s, x)};
    if (!king_pawn_moves<C>(s, g, t, o)) return;
    const bool knight = s.myKnights & here;
    u64 m = (knight ? t.knight[sq] : enemy ? 0 : att) & x.target;
    if (m && x.pinned & here) m &= knight ? 0 : t.line[sq << 6 | (u32)s.k];
    const u32 piece = knight ? M_KNIGHT : (bishop ? M_BISHOP : 0u) | (rook ? M_ROOK : 0u);
    for (u64 left = __ballot(m != 0); left; left = __ballot(m != 0)) {
        if (m) {
            o.put(o.n + lanes_below(left), mk_move((int)sq, ctz(m), MF_QUIET) | piece << 24);
            m &= m - 1;
        }
        o.n += (u32)popc(left);
    }
}
// The number of words in out, which has room for cap.  A board with more moves
// than that (218 are the most in a game, but a caller may set up one with more
// queens than a game has) raises *full: the search is then to be run by the
// kernels whose lists are sized by the counted moves.
constexpr u32 WAVE_LIST = 256;
template <int V>
__device__ __forceinline__ u32 wave_words(const Pos &p, const Tables &t, u32 *out, u32 cap, u32 *full) {
    WaveSink o{out, cap, 0, threadIdx.x & 63};
    if (pos_side(p)) wave_side_words<BLACK, V>(p, t, o);
    else wave_side_words<WHITE, V>(p, t, o);
    const u32 n = (u32)__builtin_amdgcn_readfirstlane((int)o.n);
    if (n <= cap) return n;
    if (o.lane == 0) atomicOr(full, 1u);
    return cap;
}

// perft(2) of one board by a whole wave: its moves are listed (list: WAVE_LIST
// words), then counted a lane each.  Returns the lane's part; *moves: the
// board's moves.  A launch that does this takes 16 us (ks_three), where one
// with a tile of the fused leaf takes 28, but it is about ten times the
// instructions per board of a full tile.
template <int V>
__device__ __forceinline__ u32 wave_perft2(const Pos &b, u32 *list, u32 *moves, u32 *full, const Tables &t) {
    const u32 m = wave_words<V>(b, t, list, WAVE_LIST, full), lane = threadIdx.x & 63;
    wave_sync();
    u32 sum = 0;
    for (u32 k = lane; k < m; k += 64) sum += count_any<V>(made(b, (u16)list[k], piece_code(list[k] >> 24), t), t);
    wave_sync();
    *moves = m;
    return sum;
}
// the board after the move in list[i], in scalar registers
__device__ __forceinline__ Pos wave_made(const Pos &b, const u32 *list, u32 i, const Tables &t) {
    const u32 w = (u32)__builtin_amdgcn_readfirstlane((int)list[i]);
    return uniform_pos(made(b, (u16)w, piece_code(w >> 24), t));
}

// state of a board after expansion (TT and batch searches)
enum : u8 { ST_LIVE = 0, ST_HIT = 1, ST_DUP = 2 };

struct LeafTile {
    Kin k[LEAF_TILE];
    u32 word[LEAF_CAP];
    u32 per[LEAF_TILE];  // sum over a board's children
};

// this wave's number in its work-group, in a scalar register: what is
// addressed by it, and loops over it, then stay out of the vector registers
__device__ __forceinline__ u32 wave_number() { return (u32)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)); }

__device__ __forceinline__ u32 wave_excl_scan(u32 v, u32 *total) {
    const int lane = threadIdx.x & 63;
    u32 x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const u32 y = __shfl_up(x, o, 64);
        if (lane >= o) x += y;
    }
    *total = __shfl(x, 63, 64);
    return x - v;
}

// per[lane] = perft(2) of the wave's boards (lane's board b when live).
// Returns this lane's number of moves; all lanes of the wave call it.  err is
// set if a board lists a different number of moves than it counted.
template <int V>
__device__ __forceinline__ u32 leaf_expand(LeafTile &s, bool live, const Pos &b, u32 *err, const Tables &t) {
    const u32 lane = threadIdx.x & 63;
    if (live) s.k[lane] = kin_any(b, t);
    u32 moves = 0;
    for (u64 pending = __ballot(live); pending;) {
        // the boards still to do (one that did not fit the window is worked
        // out again: nothing of it is held while the others are counted)
        wave_sync();
        LeafEval q{};
        if (pending >> lane & 1) q = leaf_any(s.k[lane], t);
        const u32 list = q.calm + q.full;
        u32 totals;  // calm moves in the low half, the others in the high half
        const u32 at = wave_excl_scan(q.calm | q.full << 16, &totals), atCalm = at & 0xFFFF, atFull = at >> 16;
        // calm moves fill the window from its front, the others from its end
        const bool due = pending >> lane & 1, fits = due && atCalm + atFull + list <= LEAF_CAP;
        if (fits) {
            LeafSink o{s.word, LEAF_CAP, lane, atCalm, LEAF_CAP - 1 - atFull};
            generate_leaf<V>(s.k[lane], q.g, t, o);
            if (o.calm != atCalm + q.calm || o.full + atFull + q.full != LEAF_CAP - 1) atomicOr(err, 2u);
            s.per[lane] = q.quiet * q.c0;
            moves = list + q.quiet;
        }
        pending = __ballot(due && !fits);
        const u32 n = pending ? __shfl(at, __builtin_ctzll(pending), 64) : totals;
        const u32 nCalm = n & 0xFFFF, nFull = n >> 16;
        wave_sync();
        for (u32 j = lane; j < nCalm; j += 64) {
            const u32 w = s.word[j], o = w >> 16 & (LEAF_TILE - 1);
            atomicAdd(&s.per[o], count_calm_any(s.k[o], w, t));
        }
        wave_sync();
        u32 *const word = s.word + LEAF_CAP - 1;
        // special moves are put aside: their places, two to a word, in the
        // part of the window that is free again
        u16 *const aside = (u16 *)s.word;
        const u32 room = 2 * (LEAF_CAP - nFull);
        u32 asides = 0;
        for (u32 j0 = 0; j0 < nFull; j0 += 64) {
            const u32 j = j0 + lane;
            const u32 w = j < nFull ? word[-(int)j] : 0;
            const u64 special = __ballot(w >> 31);
            if (special) {
                if (w >> 31) {
                    const u32 a = asides + lanes_below(special);
                    if (a < room) aside[a] = (u16)j;
                    else word[-(int)j] = w | LEAF_LATE;
                }
                asides += (u32)__popcll(special);
            }
            if (j < nFull && !(w >> 31)) {
                const u32 o = w >> 16 & (LEAF_TILE - 1);
                atomicAdd(&s.per[o], count_child_any<V>(s.k[o], w, t));
            }
        }
        wave_sync();
        // those put aside, then (only if the list was full) the window's late ones
        const u32 m = asides < room ? asides : room, late = asides > room ? nFull : 0;
        for (u32 j = lane; j < m + late; j += 64) {
            const u32 w = word[-(int)(j < m ? aside[j] : j - m)], o = w >> 16 & (LEAF_TILE - 1);
            if (j < m || (w & LEAF_LATE)) atomicAdd(&s.per[o], count_made<V>(s.k[o], w, t));
        }
        wave_sync();
    }
    return moves;
}

// The same by making every move and counting the replies from scratch, for
// searches from a root no game leads to (pos_regular).  The window holds any
// board's moves: a square is entered by sliders from at most eight sides, by
// eight knights and by four pawn moves, three of which are four on the last
// rank, and one king moves, which makes fewer than 1400.
struct PlainTile {
    Pos b[LEAF_TILE];
    u32 word[LEAF_CAP];
    u32 per[LEAF_TILE];
};
static_assert(LEAF_CAP >= 1400, "a board that does not fit the window would be put off for ever");
template <int V>
__device__ __forceinline__ u32 leaf_plain(PlainTile &s, bool live, const Pos &b, u32 *err, const Tables &t) {
    const u32 lane = threadIdx.x & 63;
    s.b[lane] = b;
    s.per[lane] = 0;
    wave_sync();
    const u32 c = live ? count_any<V>(s.b[lane], t) : 0;
    u32 total;
    const u32 at = wave_excl_scan(c, &total);
    for (u32 start = 0; start < total;) {
        const bool due = c && at >= start, fits = due && at + c <= start + LEAF_CAP;
        wave_sync();
        if (fits && generate_words<V>(s.b[lane], t, s.word + (at - start), c, lane) != c) atomicOr(err, 2u);
        const u64 late = __ballot(due && !fits);
        const u32 end = late ? __shfl(at, __builtin_ctzll(late), 64) : total;
        wave_sync();
        for (u32 j = start + lane; j < end; j += 64) {
            const u32 w = s.word[j - start], o = w >> 16 & (LEAF_TILE - 1);
            atomicAdd(&s.per[o], count_any<V>(made(s.b[o], (u16)w, piece_code(w >> 24), t), t));
        }
        start = end;
    }
    wave_sync();
    return c;
}

// Boards per tile: too few boards for whole tiles on every CU are dealt out a
// few at a time, for the time of the longest tile (a launch of one tile of 4
// middle-game boards takes 28 us).
constexpr u32 LEAF_RESIDENT = 3072;  // waves the chip holds
__device__ __forceinline__ u32 leaf_tile_boards(u64 n, u32 waves) {
    if (waves > LEAF_RESIDENT) waves = LEAF_RESIDENT;
    const u64 t = (n + waves - 1) / waves;
    return t < 4 ? 4 : t > LEAF_TILE ? LEAF_TILE : (u32)t;
}

// The fused leaf over boards [0, n) with move counts cnt[]: PER = false adds
// every count to *acc; PER = true writes base + perft(2) to per[i] for live
// boards (state[i] == ST_LIVE when state is given, else a valid board).
// With idx, the boards are idx[0..n) (live boards with moves, listed by
// k_live_write) and per[] is written at those indices.
// MOVES: the n boards are not stored: board j is boards[par[j]] after move
// mv[j] (the children of the level before, as the generate kernel lists
// them); the work-group makes each one and counts its moves itself, so the
// level one above the leaf never goes to HBM.  With idx as well, the boards
// made are those listed (j = idx[t]), and with PER their sums go to per[j].
// PLAIN: by leaf_plain.
template <int V, bool PER, bool MOVES = false, bool PLAIN = false>
__device__ __forceinline__ void leaf_tiles(const Pos *__restrict__ boards, const u32 *__restrict__ cnt, u64 n, u64 *acc,
                                           u64 *items, u64 *__restrict__ per, const u8 *__restrict__ state, u64 base,
                                           u32 *err, u32 *ovf, const Tables &t, const u32 *__restrict__ idx = nullptr,
                                           const u32 *__restrict__ par = nullptr, const u16 *__restrict__ mv = nullptr) {
    static_assert(V != SL_BYTE, "the byte-lookup tables leave no LDS for the move window");
    constexpr u32 WAVES = LEAF_WG / 64;
    using Tile = std::conditional_t<PLAIN, PlainTile, LeafTile>;
    __shared__ Tile tiles[WAVES];
    const u32 wave = wave_number();
    Tile &s = tiles[wave];
    const u32 lane = threadIdx.x & 63;
    u64 sum = 0, itemSum = 0;
    n = uniform64(n);
    const u32 T = leaf_tile_boards(n, gridDim.x * WAVES);
    for (u64 tile = blockIdx.x * WAVES + wave; tile * T < n; tile += gridDim.x * WAVES) {
        const u64 t0 = tile * T + lane;
        const bool live = lane < T && t0 < n;
        const u64 i = idx && live ? (u64)idx[t0] : t0;
        bool valid = false, work = live;
        Pos b{};
        if (live) {
            if constexpr (MOVES) {
                b = boards[par[i]];
                make_any(b, mv[i], t);
            } else {
                b = boards[i];
                valid = pos_valid(b);
                work = cnt[i] != 0;  // a board resolved earlier has count 0
            }
        }
        u32 c;
        if constexpr (PLAIN) c = leaf_plain<V>(s, work, b, err, t);
        else c = leaf_expand<V>(s, work, b, err, t);
        itemSum += wave_sum32(c);
        if (live) {
            const u32 p = work ? s.per[lane] : 0;
            if constexpr (PER) {
                if (idx || (state ? state[i] == ST_LIVE : valid)) {
                    const u64 v = base + p;
                    if (v < base) *ovf = 1;
                    per[i] = v;
                }
            } else {
                sum += p;
            }
        }
        wave_sync();
    }
    if ((threadIdx.x & 63) == 0 && items && itemSum) atomicAdd(items, itemSum);
    if (!PER) {
        sum = wave_sum(sum);
        if ((threadIdx.x & 63) == 0 && sum) add_checked(acc, sum, ovf);
    }
}

// three waves per SIMD (see above): at 168 registers no vector register spills;
// 5 to 67 scalar ones are kept in the lanes of vector registers
#define PG_LEAF_BOUNDS __launch_bounds__(LEAF_WG) __attribute__((amdgpu_waves_per_eu(3, 8)))

template <int V, bool PER, bool PLAIN>
__global__ PG_LEAF_BOUNDS void k_leaf_fused(
    const Pos *__restrict__ boards, const u32 *__restrict__ cnt, u64 n, u64 *acc, u64 *items, u64 *__restrict__ per,
    u32 *err, u32 *ovf, Tables t, const u32 *__restrict__ idx) {
    leaf_tiles<V, PER, false, PLAIN>(boards, cnt, n, acc, items, per, nullptr, 0, err, ovf, t, idx);
}

// the leaf over the children of `gp` listed by par/mv (see leaf_tiles, MOVES)
template <int V, bool PLAIN>
__global__ PG_LEAF_BOUNDS void k_leaf_moves(
    const Pos *__restrict__ gp, const u32 *__restrict__ par, const u16 *__restrict__ mv, u64 n, u64 *acc, u64 *items,
    u32 *err, u32 *ovf, Tables t) {
    leaf_tiles<V, false, true, PLAIN>(gp, nullptr, n, acc, items, nullptr, nullptr, 0, err, ovf, t, nullptr, par, mv);
}

// per-child sums over the children of `gp` listed by idx (see leaf_tiles,
// MOVES with idx): perft(2) of each listed child into per[]
template <int V, bool PLAIN>
__global__ PG_LEAF_BOUNDS void k_leaf_moves_per(
    const Pos *__restrict__ gp, const u32 *__restrict__ par, const u16 *__restrict__ mv, const u32 *__restrict__ idx,
    u64 n, u64 *items, u64 *__restrict__ per, u32 *err, u32 *ovf, Tables t) {
    leaf_tiles<V, true, true, PLAIN>(gp, nullptr, n, nullptr, items, per, nullptr, 0, err, ovf, t, idx, par, mv);
}

// ---------------------------------------------------------------- live list
// The boards of a leaf level that have moves, in index order: a level whose
// other boards were resolved from the table or collapsed into an equal board
// (count 0) then fills the fused leaf's tiles with boards that have work.
// Each work-group takes LIVE_CHUNK consecutive boards: k_live_count counts
// its live boards, the counts are scanned, and k_live_write lists them at
// the chunk's offset.  With state given, a live board is one whose state is
// ST_LIVE (a level whose boards were not written, so not counted either).
constexpr int LIVE_WG = 256, LIVE_PER_THREAD = 16, LIVE_CHUNK = LIVE_WG * LIVE_PER_THREAD;

__device__ __forceinline__ bool live_at(const u32 *__restrict__ cnt, const u8 *__restrict__ state, u64 i) {
    return state ? state[i] == ST_LIVE : cnt[i] != 0;
}

static __global__ __launch_bounds__(LIVE_WG) void k_live_count(const u32 *__restrict__ cnt, const u8 *__restrict__ state,
                                                              u64 n, u32 *__restrict__ chunkCount) {
    const u64 base = (u64)blockIdx.x * LIVE_CHUNK;
    u32 c = 0;
#pragma unroll
    for (int k = 0; k < LIVE_PER_THREAD; k++) {
        const u64 i = base + (u64)k * LIVE_WG + threadIdx.x;
        c += i < n && live_at(cnt, state, i);
    }
    u64 total;
    (void)block_excl_scan<LIVE_WG>(c, &total);
    if (threadIdx.x == 0) chunkCount[blockIdx.x] = (u32)total;
}

static __global__ __launch_bounds__(LIVE_WG) void k_live_write(const u32 *__restrict__ cnt, const u8 *__restrict__ state,
                                                              u64 n, const u64 *__restrict__ chunkOff,
                                                              u32 *__restrict__ idx) {
    const u64 base = (u64)blockIdx.x * LIVE_CHUNK;
    u64 at = chunkOff[blockIdx.x];
    for (int k = 0; k < LIVE_PER_THREAD; k++) {
        const u64 i = base + (u64)k * LIVE_WG + threadIdx.x;
        const bool f = i < n && live_at(cnt, state, i);
        u64 total;
        const u64 pos = block_excl_scan<LIVE_WG>(f ? 1 : 0, &total);
        if (f) idx[at + pos] = (u32)i;
        at += total;
    }
}

// ---------------------------------------------------------------- scan
// Exclusive scan of u32 counts into u64 offsets; off[n] receives the total.
// Reduce-then-scan over 2048-item tiles: k_scan_reduce (tile sums),
// k_scan_spine (one work-group scans the tile sums), k_scan_down (each tile
// rescans itself from its base).
__device__ __forceinline__ void load_tile(const u32 *c, u64 n, u64 base, u32 v[SCAN_IPT]) {
    if (base + SCAN_IPT <= n && (reinterpret_cast<uintptr_t>(c + base) & 15) == 0) {
        const uint4 a = *reinterpret_cast<const uint4 *>(c + base);
        const uint4 b = *reinterpret_cast<const uint4 *>(c + base + 4);
        v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
        v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
    } else {
#pragma unroll
        for (int j = 0; j < SCAN_IPT; j++) v[j] = base + j < n ? c[base + j] : 0;
    }
}

static __global__ __launch_bounds__(SCAN_WG) void k_scan_reduce(const u32 *__restrict__ c, u64 n, u64 *__restrict__ tileSum) {
    const u64 base = (u64)blockIdx.x * SCAN_TILE + (u64)threadIdx.x * SCAN_IPT;
    u32 v[SCAN_IPT];
    load_tile(c, n, base, v);
    u64 s = 0;
#pragma unroll
    for (int j = 0; j < SCAN_IPT; j++) s += v[j];
    u64 tot;
    block_excl_scan<SCAN_WG>(s, &tot);
    if (threadIdx.x == 0) tileSum[blockIdx.x] = tot;
}

static __global__ __launch_bounds__(1024) void k_scan_spine(u64 *tileSum, u64 tiles, u64 *total) {
    u64 carry = 0;
    for (u64 s = 0; s < tiles; s += 1024) {
        const u64 i = s + threadIdx.x;
        const u64 v = i < tiles ? tileSum[i] : 0;
        u64 tot;
        const u64 ex = block_excl_scan<1024>(v, &tot);
        if (i < tiles) tileSum[i] = carry + ex;
        carry += tot;
    }
    if (threadIdx.x == 0) *total = carry;
}

static __global__ __launch_bounds__(SCAN_WG) void k_scan_down(const u32 *__restrict__ c, u64 n, const u64 *__restrict__ tileSum,
                                                      u64 *__restrict__ off) {
    const u64 base = (u64)blockIdx.x * SCAN_TILE + (u64)threadIdx.x * SCAN_IPT;
    u32 v[SCAN_IPT];
    load_tile(c, n, base, v);
    u64 s = 0;
#pragma unroll
    for (int j = 0; j < SCAN_IPT; j++) s += v[j];
    u64 tot;
    u64 run = tileSum[blockIdx.x] + block_excl_scan<SCAN_WG>(s, &tot);
#pragma unroll
    for (int j = 0; j < SCAN_IPT; j++) {
        if (base + j < n) off[base + j] = run;
        run += v[j];
    }
}

// ---------------------------------------------------------------- probes

template <int V>
__global__ __launch_bounds__(wg_size<V>()) void k_probe_generate(const Pos *__restrict__ b, u64 n, u16 *__restrict__ moves,
                                                                 u32 *__restrict__ cnt, Tables t) {
    stage_tables<V>(t);
    PG_GRID_LOOP(i, n) cnt[i] = generate_any<V>(b[i], t, moves + i * 256);
}

static __global__ __launch_bounds__(256) void k_probe_make(const Pos *__restrict__ b, const u16 *__restrict__ mv, u64 n,
                                                    Pos *__restrict__ out, Key128 *keys, Tables t) {
    PG_GRID_LOOP(i, n) {
        Pos p = b[i];
        if (keys) {
            Key128 h = keys[i];
            make_any_hash(p, mv[i], h, t);
            keys[i] = h;
        } else {
            make_any(p, mv[i], t);
        }
        out[i] = p;
    }
}

template <int V>
__global__ __launch_bounds__(wg_size<V>()) void k_probe_slider(int rook, const u8 *__restrict__ sq, const u64 *__restrict__ occ,
                                                               u64 n, u64 *__restrict__ out, Tables t) {
    stage_tables<V>(t);
    PG_GRID_LOOP(i, n) out[i] = rook ? Sl<V>::rook(t, sq[i], occ[i]) : Sl<V>::bishop(t, sq[i], occ[i]);
}

}  // namespace pg
