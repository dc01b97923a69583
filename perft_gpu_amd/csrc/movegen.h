// movegen.h -- legal move counting, generation and make-move for gfx950.
//
// Written for 64-lane wavefronts: the leaf count is branch-light so that the
// lanes of a wave (sibling positions) stay converged.  The leaf itself counts
// the replies to a board's moves by difference (Kin, leaf_eval, count_child
// below); what follows holds for the counting of one board by itself.
//  * One "target" mask folds the reference's separate out-of-check path
//    (MoveGeneratorBitboard.h:2825-2994) into the normal one: not in check ->
//    ~own, single check -> checker | squares between, double check -> 0.
//    A pinned piece can never land on a check-resolving square, so the
//    result equals the reference's countMovesOutOfCheck.
//  * Pawns are counted in bulk (one shift + popcount per direction); pinned
//    pawns move only along the king line they sit on, which is applied as a
//    per-direction mask instead of a per-pawn loop.  Knights take one table
//    lookup + popcount each (at most two knights is cheaper than eight
//    direction shifts).
//  * With Kogge-Stone sliders, moves are also counted in bulk: the rays of
//    different sliders in one direction are disjoint (a ray stops at the
//    first occupied square), so popcount(fill_d(all movers) & target) sums
//    the per-piece counts.  Pinned sliders join the fills of the axis their
//    pin lies on.  The magic variants count per piece.
//  * Enemy attacks (with the moving king removed, so sliders see through
//    it), pins and slider checkers follow the reference's method
//    (findAttackedSquares :1254, findPinnedPieces :1213).
// The same source compiles for the host so the library can list moves and
// build workloads without a GPU; perft itself only runs on the device.
#pragma once
#include "pg_types.h"

namespace pg {

enum Slider { SL_KOGGE = 0, SL_PLAIN = 1, SL_FANCY = 2, SL_BYTE = 3, SL_COUNT = 4 };

// Fixed-shift fancy magic entry: factor, base offset into the shared
// 97264-entry table, and (byte-lookup variant) offset into the per-piece list
// of distinct attack sets.  Same fields as the reference's FancyMagicEntry
// (chess.h:343-359).
struct FancyEntry {
    u64 factor;
    int base;
    int offset;
};
static_assert(sizeof(FancyEntry) == 16, "fancy entry is 16 bytes");

// What a king's square determines, one cache line: the squares a rook, bishop
// or knight there would reach on an empty board, the king's own steps, and
// the whole file, rank and diagonals through it.
struct KingRow {
    u64 rook, bishop, knight, king, file, rank, diag, anti;
};
static_assert(sizeof(KingRow) == 64, "a king's row is one line");
// For a king and a slider on one line: the squares strictly between, and the
// square next to the king away from the slider (0: off the board).
struct PinEntry {
    u64 between, behind;
};

constexpr int ROOK_BITS = 12, BISHOP_BITS = 9;
constexpr int FANCY_TABLE_SIZE = 97264, BYTE_ROOK_SIZE = 4900, BYTE_BISHOP_SIZE = 1428;
constexpr int ZOB_WORDS = 782;

// Table pointers (device or host memory; on the device the byte-lookup
// variant repoints some of them at LDS copies).
struct Tables {
    const u64 *knight, *king;            // [64] empty-board attacks
    const KingRow *row;                  // [64]
    const PinEntry *pin;                 // [64*64] king, slider
    const u64 *line;                     // [64*64] full line through two squares
    const u64 *rookMask, *bishopMask;    // [64] relevant occupancy (edges off)
    const u64 *rookMagic, *bishopMagic;  // [64] plain magic factors
    const u64 *rookPlain, *bishopPlain;  // [64*4096], [64*512]
    const FancyEntry *rookFancy, *bishopFancy;  // [64]
    const u64 *fancy;                    // [97264]
    const u8 *byteIdx;                   // [97264]
    const u64 *byteRook, *byteBishop;    // [4900], [1428]
    const u64 *zobLo, *zobHi;            // [782] each
};

PG_HD int popc(u64 x) { return __builtin_popcountll(x); }
// n + popc(x), the two halves through the count instruction's own addend
// (LLVM sums the halves first and adds with further instructions)
PG_HD int popc_add(u64 x, int n) {
#if defined(__HIP_DEVICE_COMPILE__)
    asm("v_bcnt_u32_b32 %0, %1, %0" : "+v"(n) : "v"((u32)x));
    asm("v_bcnt_u32_b32 %0, %1, %0" : "+v"(n) : "v"((u32)(x >> 32)));
    return n;
#else
    return n + __builtin_popcountll(x);
#endif
}
// all ones if c
PG_HD u64 mask_if(bool c) {
    const u32 m = c ? ~0u : 0u;
    return (u64)m << 32 | m;
}
PG_HD int ctz(u64 x) { return __builtin_ctzll(x); }
PG_HD u64 bit(int s) { return 1ULL << s; }
PG_HD bool several(u64 x) { return (x & (x - 1)) != 0; }

// Three-input bitwise function given by its truth table F: bit i of F is the
// result for inputs (a, b, c) = (i >> 2 & 1, i >> 1 & 1, i & 1), so F for an
// expression is that expression evaluated on a = 0xF0, b = 0xCC, c = 0xAA.
// On gfx950 each 32-bit half is one v_bitop3_b32; the compiler does not form
// these from 64-bit and/or chains by itself.
template <u32 F>
PG_HD u64 bop3(u64 a, u64 b, u64 c) {
#if defined(__HIP_DEVICE_COMPILE__)
    const u32 lo = __builtin_amdgcn_bitop3_b32((u32)a, (u32)b, (u32)c, F);
    const u32 hi = __builtin_amdgcn_bitop3_b32((u32)(a >> 32), (u32)(b >> 32), (u32)(c >> 32), F);
    return ((u64)hi << 32) | lo;
#else
    u64 r = 0;
    for (int i = 0; i < 8; i++)
        if ((F >> i) & 1) r |= ((i & 4) ? a : ~a) & ((i & 2) ? b : ~b) & ((i & 1) ? c : ~c);
    return r;
#endif
}
PG_HD u64 or_and(u64 a, u64 b, u64 c) { return bop3<0xF8>(a, b, c); }    // a | (b & c)
PG_HD u64 and3(u64 a, u64 b, u64 c) { return bop3<0x80>(a, b, c); }      // a & b & c
PG_HD u64 or3(u64 a, u64 b, u64 c) { return bop3<0xFE>(a, b, c); }       // a | b | c
PG_HD u64 and_or(u64 a, u64 b, u64 c) { return bop3<0xE0>(a, b, c); }    // a & (b | c)
PG_HD u64 and_nor(u64 a, u64 b, u64 c) { return bop3<0x10>(a, b, c); }   // a & ~b & ~c
PG_HD u64 andn(u64 a, u64 b) { return bop3<0x30>(a, b, b); }             // a & ~b
PG_HD u64 or_xor(u64 a, u64 b, u64 c) { return bop3<0xF6>(a, b, c); }    // a | (b ^ c)
PG_HD u64 xor_and(u64 a, u64 b, u64 c) { return bop3<0x28>(a, b, c); }   // (a ^ b) & c

// A board the generator accepts: one king per side, no white bit on an empty
// square and an en-passant field of 0 (none) or a file 1..8.  (Inputs arriving over the C ABI are checked with this.)
PG_HD bool pos_sane(const Pos &p) {
    const u64 occ = pos_occ(p);
    return popc(p.kings & p.white) == 1 && popc(p.kings & ~p.white) == 1 && (p.white & ~occ) == 0 &&
           pos_ep(p) <= 8;
}

// ---------------------------------------------------------------- fills
// Kogge-Stone occluded fill, returns the squares attacked in one direction
// (first blocker included).  S = shift, M = wrap mask of the target file.
template <int S, u64 M>
PG_HD u64 fill_up(u64 g, u64 e) {
    e &= M;
    g |= (g << S) & e;
    e &= e << S;
    g |= (g << (2 * S)) & e;
    e &= e << (2 * S);
    g |= (g << (4 * S)) & e;
    return (g << S) & M;
}
template <int S, u64 M>
PG_HD u64 fill_dn(u64 g, u64 e) {
    e &= M;
    g |= (g >> S) & e;
    e &= e >> S;
    g |= (g >> (2 * S)) & e;
    e &= e >> (2 * S);
    g |= (g >> (4 * S)) & e;
    return (g >> S) & M;
}
PG_HD u64 att_n(u64 g, u64 e) { return fill_up<8, ~0ULL>(g, e); }
PG_HD u64 att_s(u64 g, u64 e) { return fill_dn<8, ~0ULL>(g, e); }
PG_HD u64 att_e(u64 g, u64 e) { return fill_up<1, ~FILEA>(g, e); }
PG_HD u64 att_w(u64 g, u64 e) { return fill_dn<1, ~FILEH>(g, e); }
PG_HD u64 att_ne(u64 g, u64 e) { return fill_up<9, ~FILEA>(g, e); }
PG_HD u64 att_nw(u64 g, u64 e) { return fill_up<7, ~FILEH>(g, e); }
PG_HD u64 att_se(u64 g, u64 e) { return fill_dn<7, ~FILEA>(g, e); }
PG_HD u64 att_sw(u64 g, u64 e) { return fill_dn<9, ~FILEH>(g, e); }
PG_HD u64 ks_rook(u64 g, u64 e) { return att_n(g, e) | att_s(g, e) | att_e(g, e) | att_w(g, e); }
PG_HD u64 ks_bishop(u64 g, u64 e) { return att_ne(g, e) | att_nw(g, e) | att_se(g, e) | att_sw(g, e); }

PG_HD u64 king_att(u64 k) {
    u64 a = ((k << 1) & ~FILEA) | ((k >> 1) & ~FILEH);
    k |= a;
    return a | (k << 8) | (k >> 8);
}
PG_HD u64 knight_att(u64 n) {
    u64 l1 = (n >> 1) & 0x7f7f7f7f7f7f7f7fULL, l2 = (n >> 2) & 0x3f3f3f3f3f3f3f3fULL;
    u64 r1 = (n << 1) & 0xfefefefefefefefeULL, r2 = (n << 2) & 0xfcfcfcfcfcfcfcfcULL;
    u64 h1 = l1 | r1, h2 = l2 | r2;
    return (h1 << 16) | (h1 >> 16) | (h2 << 8) | (h2 >> 8);
}

PG_HD u64 rev64(u64 x) {
#if defined(__clang__)
    return __builtin_bitreverse64(x);
#else
    x = ((x >> 1) & 0x5555555555555555ULL) | ((x & 0x5555555555555555ULL) << 1);
    x = ((x >> 2) & 0x3333333333333333ULL) | ((x & 0x3333333333333333ULL) << 2);
    x = ((x >> 4) & 0x0F0F0F0F0F0F0F0FULL) | ((x & 0x0F0F0F0F0F0F0F0FULL) << 4);
    return __builtin_bswap64(x);
#endif
}

PG_HD u64 nor2(u64 a, u64 b) { return bop3<0x03>(a, b, b); }  // ~(a | b)

// squares east of each slider in s up to and including its first blocker,
// given eo = ~(occ | FILEH); every slider must be in occ
PG_HD u64 east_sum(u64 s, u64 eo) { return (andn(s, FILEH) << 1) + eo; }

template <int S> PG_HD u64 shift(u64 x) {
#if defined(__HIP_DEVICE_COMPILE__)
    if constexpr (S > 0 && S < 32) {
        u64 r;
        asm("v_lshlrev_b64 %0, %1, %2" : "=v"(r) : "i"(S), "v"(x));
        return r;
    } else if constexpr (S < 0 && S > -32) {
        u64 r;
        asm("v_lshrrev_b64 %0, %1, %2" : "=v"(r) : "i"(-S), "v"(x));
        return r;
    }
#endif
    return S > 0 ? x << S : x >> -S;
}
PG_HD u64 and_mask(u64 x, u64 m) { return m == ~0ULL ? x : x & m; }
template <int N> struct Int {
    static constexpr int value = N;
};
struct Prop3 {
    u64 a, b, c;
};
// propagators of a direction from the empty squares that may be entered
template <int S> PG_HD Prop3 props(u64 a) {
    Prop3 p;
    p.a = a;
    p.b = a & shift<S>(a);
    p.c = p.b & shift<2 * S>(p.b);
    return p;
}
// generators grown through the propagators (the ray squares shifted back
// by one step, still to be shifted by S and wrap-masked)
template <int S> PG_HD u64 grow(u64 g, const Prop3 &p) {
    g = or_and(g, shift<S>(g), p.a);
    g = or_and(g, shift<2 * S>(g), p.b);
    if constexpr (S == 8 || S == -8) {
        // a shift by 32 moves one half into the other: one 32-bit step
        u32 lo = (u32)g, hi = (u32)(g >> 32);
        if (S == 8) hi |= lo & (u32)(p.c >> 32);
        else lo |= hi & (u32)p.c;
        return ((u64)hi << 32) | lo;
    }
    return or_and(g, shift<4 * S>(g), p.c);
}
// the side's part of a piece word (every piece word lies inside occ)
template <int C> PG_HD u64 side_of(u64 b, u64 white) { return C == WHITE ? b & white : andn(b, white); }

// Attacks of the sliders in b (bishop-like) and r (rook-like) through the
// empty squares e, one pass over the eight directions with the propagators
// built once per direction; every slider must be off e.
PG_HD u64 ks_attacks(u64 b, u64 r, u64 e) {
    const Prop3 pn = props<8>(e), ps = props<-8>(e);
    u64 a = shift<8>(grow<8>(r, pn)) | shift<-8>(grow<-8>(r, ps));
    const u64 eA = andn(e, FILEA), eH = andn(e, FILEH);
    a = or_xor(a, eH, east_sum(r, eH));
    a = or_xor(a, eA, rev64(east_sum(rev64(r), rev64(eA))));
    const Prop3 p9 = props<9>(eA), m9 = props<-9>(eH), p7 = props<7>(eH), m7 = props<-7>(eA);
    a = or_and(a, shift<9>(grow<9>(b, p9)), ~FILEA);
    a = or_and(a, shift<-9>(grow<-9>(b, m9)), ~FILEH);
    a = or_and(a, shift<7>(grow<7>(b, p7)), ~FILEH);
    return or_and(a, shift<-7>(grow<-7>(b, m7)), ~FILEA);
}

// Attacks of one slider along one line through its square (the line may
// include the square): (o - s) ^ rev(rev(o) - rev(s)) with o the occupied
// squares of the line other than s (hyperbola quintessence, no tables).
PG_HD u64 line_att(u64 sb, u64 occ, u64 line) {
    const u64 o = bop3<0x40>(occ, line, sb);  // occ & line & ~sb
    return xor_and(o - sb, rev64(rev64(o) - rev64(sb)), line);
}

// pawn geometry per side
template <int C> PG_HD u64 fwd(u64 x) { return C == WHITE ? x << 8 : x >> 8; }
template <int C> PG_HD u64 fwd_west(u64 x) { return C == WHITE ? (x << 7) & ~FILEH : (x >> 9) & ~FILEH; }
template <int C> PG_HD u64 fwd_east(u64 x) { return C == WHITE ? (x << 9) & ~FILEA : (x >> 7) & ~FILEA; }
template <int C> PG_HD u64 pawn_att(u64 x) { return fwd_west<C>(x) | fwd_east<C>(x); }

// lines through a square
PG_HD u64 file_of(int s) { return FILEA << (s & 7); }
PG_HD u64 rank_of(int s) { return RANK1 << (s & 56); }
PG_HD u64 diag_of(int s) {  // a1-h8 direction
    int d = (s & 7) - (s >> 3);
    return d >= 0 ? DIAG_A1H8 >> (8 * d) : DIAG_A1H8 << (-8 * d);
}
PG_HD u64 anti_of(int s) {  // a8-h1 direction
    int d = (s & 7) + (s >> 3) - 7;
    return d >= 0 ? DIAG_A8H1 << (8 * d) : DIAG_A8H1 >> (-8 * d);
}

// ---------------------------------------------------------------- sliders
template <int V> struct Sl;

template <> struct Sl<SL_KOGGE> {
    static constexpr bool kBulk = true;
    PG_HD static u64 rook(const Tables &, int s, u64 occ) {
        const u64 sb = bit(s);
        return line_att(sb, occ, file_of(s)) | line_att(sb, occ, rank_of(s));
    }
    PG_HD static u64 bishop(const Tables &, int s, u64 occ) {
        const u64 sb = bit(s);
        return line_att(sb, occ, diag_of(s)) | line_att(sb, occ, anti_of(s));
    }
};

// high 32 bits of the low 64-bit word of a*b, i.e. (a*b) >> 32 mod 2^32:
// three 32-bit multiplies instead of a full 64x64 product.
PG_HD u32 mul_hi32_lo64(u64 a, u64 b) {
    u32 al = (u32)a, ah = (u32)(a >> 32), bl = (u32)b, bh = (u32)(b >> 32);
    u32 hi = (u32)(((u64)al * bl) >> 32);
    return hi + al * bh + ah * bl;
}

template <> struct Sl<SL_PLAIN> {
    static constexpr bool kBulk = false;
    PG_HD static u64 rook(const Tables &t, int s, u64 occ) {
        u32 i = mul_hi32_lo64(t.rookMagic[s], occ & t.rookMask[s]) >> (32 - ROOK_BITS);
        return t.rookPlain[(s << ROOK_BITS) + i];
    }
    PG_HD static u64 bishop(const Tables &t, int s, u64 occ) {
        u32 i = mul_hi32_lo64(t.bishopMagic[s], occ & t.bishopMask[s]) >> (32 - BISHOP_BITS);
        return t.bishopPlain[(s << BISHOP_BITS) + i];
    }
};

template <> struct Sl<SL_FANCY> {
    static constexpr bool kBulk = false;
    PG_HD static u64 rook(const Tables &t, int s, u64 occ) {
        FancyEntry f = t.rookFancy[s];
        return t.fancy[f.base + (mul_hi32_lo64(f.factor, occ & t.rookMask[s]) >> (32 - ROOK_BITS))];
    }
    PG_HD static u64 bishop(const Tables &t, int s, u64 occ) {
        FancyEntry f = t.bishopFancy[s];
        return t.fancy[f.base + (mul_hi32_lo64(f.factor, occ & t.bishopMask[s]) >> (32 - BISHOP_BITS))];
    }
};

template <> struct Sl<SL_BYTE> {
    static constexpr bool kBulk = false;
    PG_HD static u64 rook(const Tables &t, int s, u64 occ) {
        FancyEntry f = t.rookFancy[s];
        u32 i = mul_hi32_lo64(f.factor, occ & t.rookMask[s]) >> (32 - ROOK_BITS);
        return t.byteRook[t.byteIdx[f.base + i] + f.offset];
    }
    PG_HD static u64 bishop(const Tables &t, int s, u64 occ) {
        FancyEntry f = t.bishopFancy[s];
        u32 i = mul_hi32_lo64(f.factor, occ & t.bishopMask[s]) >> (32 - BISHOP_BITS);
        return t.byteBishop[t.byteIdx[f.base + i] + f.offset];
    }
};

// ---------------------------------------------------------------- context
// A board as the side to move sees it.  Bishops and rooks include the queens.
struct Sides {
    u64 occ, mine, enemy;
    u64 myPawns, myKnights, myBishops, myRooks, myKing;
    u64 ePawns, eKnights, eBishops, eRooks;
    int k, ek;        // king squares, in range even for a board without a king (king_square)
    u32 castle, eCastle;  // castling rights of the side, of the enemy (2 bits each)
    u32 ep;               // en-passant file + 1
};

// The square of a king, or 31 if there is none (it was taken, on a board that
// no game leads to).  ctz(0) is not defined: 31 is what it came to in the
// kernels that hold a board per lane, but in scalar registers it is -1, the
// compiler leaves out a mask after it, and tables were read 4 GB out of place.
PG_HD int king_square(u64 kings) { return kings ? ctz(kings) : 31; }

template <int C> PG_HD Sides sides_of(const Pos &p) {
    Sides s;
    const u64 W = p.white, pawns = pos_pawns(p);
    s.occ = or3(p.kings, pawns, or3(p.knights, p.bishopQueens, p.rookQueens));
    s.mine = C == WHITE ? W : andn(s.occ, W);
    s.enemy = C == WHITE ? andn(s.occ, W) : W;
    s.myPawns = side_of<C>(pawns, W);
    s.myKnights = side_of<C>(p.knights, W);
    s.myBishops = side_of<C>(p.bishopQueens, W);
    s.myRooks = side_of<C>(p.rookQueens, W);
    s.myKing = side_of<C>(p.kings, W);
    s.ePawns = side_of<1 - C>(pawns, W);
    s.eKnights = side_of<1 - C>(p.knights, W);
    s.eBishops = side_of<1 - C>(p.bishopQueens, W);
    s.eRooks = side_of<1 - C>(p.rookQueens, W);
    s.k = king_square(s.myKing);
    s.ek = king_square(side_of<1 - C>(p.kings, W));
    s.castle = (u32)(C == WHITE ? pos_wcastle(p) : pos_bcastle(p));
    s.eCastle = (u32)(C == WHITE ? pos_bcastle(p) : pos_wcastle(p));
    s.ep = (u32)pos_ep(p);
    return s;
}

struct MoveCtx {
    u64 pinned, checkers, threatened, target;
};

// squares the enemy attacks with king, pawns and knights
template <int C> PG_HD u64 leaper_attacks(const Sides &s, const Tables &t) {
    const u64 pw = C == WHITE ? shift<-9>(s.ePawns) : shift<7>(s.ePawns);
    const u64 pe = C == WHITE ? shift<-7>(s.ePawns) : shift<9>(s.ePawns);
    u64 a = or3(t.king[s.ek], andn(pw, FILEH), andn(pe, FILEA));
    const u64 h1 = or_and(andn(shift<-1>(s.eKnights), FILEH), shift<1>(s.eKnights), ~FILEA);
    const u64 h2 = or_and(andn(shift<-2>(s.eKnights), FILEG | FILEH), shift<2>(s.eKnights), ~(FILEA | FILEB));
    a = or3(a, shift<16>(h1), shift<-16>(h1));
    return or3(a, shift<8>(h2), shift<-8>(h2));
}

// squares from which an enemy pawn or knight checks, as found
template <int C> PG_HD u64 leaper_checks(const Sides &s, const Tables &t, u64 chk) {
    const u64 kw = C == WHITE ? shift<7>(s.myKing) : shift<-9>(s.myKing);
    const u64 ke = C == WHITE ? shift<9>(s.myKing) : shift<-7>(s.myKing);
    return or_and(or_and(chk, or_and(andn(kw, FILEH), ke, ~FILEA), s.ePawns), t.row[s.k].knight, s.eKnights);
}

// Pinned pieces, checkers and the squares a move other than the king's must
// end on; returns the squares behind the king on a slider's check line.
// Sliders on a king line: no blocker -> checker, one blocker -> pinned.
template <int C> PG_HD u64 pins_and_checks(const Sides &s, const Tables &t, MoveCtx &x) {
    const KingRow &row = t.row[s.k];
    u64 cand = or_and(row.rook & s.eRooks, row.bishop, s.eBishops);
    u64 pinned = 0, chk = 0, behind = 0;
    for (; cand; cand &= cand - 1) {
        const int q = ctz(cand);
        const PinEntry e = t.pin[(s.k << 6) | q];
        const u64 b = e.between & s.occ;
        // (masks: selects would be runs of v_cndmask on vcc, which issue slowly)
        const u64 none = mask_if(b == 0);
        pinned = or_and(pinned, b, mask_if(!several(b)));
        chk = or_and(chk, bit(q), none);
        behind = or_and(behind, e.behind, none);
    }
    chk = leaper_checks<C>(s, t, chk);
    x.pinned = pinned & s.mine;
    x.checkers = chk;
    u64 tgt = ~s.mine;
    if (chk) tgt &= several(chk) ? 0ULL : (chk | t.pin[(s.k << 6) | ctz(chk)].between);
    x.target = tgt;
    return behind;
}

template <int C, int V>
PG_HD void prologue(const Sides &s, const Tables &t, MoveCtx &x) {
    // squares the enemy attacks, sliders looking through our king
    u64 a = leaper_attacks<C>(s, t);
    if (Sl<V>::kBulk) {
        a |= ks_attacks(s.eBishops, s.eRooks, ~s.occ | s.myKing);
    } else {
        const u64 o = s.occ ^ s.myKing;
        for (u64 b = s.eBishops; b; b &= b - 1) a |= Sl<V>::bishop(t, ctz(b), o);
        for (u64 r = s.eRooks; r; r &= r - 1) a |= Sl<V>::rook(t, ctz(r), o);
    }
    x.threatened = a;

    (void)pins_and_checks<C>(s, t, x);
}

enum { P_PAWN = 1, P_KNIGHT, P_BISHOP, P_ROOK, P_QUEEN, P_KING };
// The piece words that a moving piece belongs to, one bit each; a queen is in
// both slider words.
// M_SPECIAL marks a move that is more than a piece leaving one square for
// another: a promotion, castling, an en-passant capture, or a double push that
// lets the enemy capture en passant.
enum : u32 { M_PAWN = 1, M_KNIGHT = 2, M_BISHOP = 4, M_ROOK = 8, M_QUEEN = 12, M_KING = 16, M_SPECIAL = 128 };
PG_HD int piece_code(u32 m) {
    constexpr u64 code = (u64)P_PAWN << 3 | (u64)P_KNIGHT << 6 | (u64)P_BISHOP << 12 | (u64)P_ROOK << 24 |
                         (u64)P_QUEEN << 36 | (u64)P_KING << 48;
    return (int)(code >> (3 * (m & 31))) & 7;
}

// calls f(square) for every set square of m, low half then high half (a
// 32-bit find-first-set and clear per square instead of the 64-bit ones)
template <class F>
PG_HD void each_square(u64 m, F &&f) {
    for (u32 lo = (u32)m; lo; lo &= lo - 1) f(__builtin_ctz(lo));
    for (u32 hi = (u32)(m >> 32); hi; hi &= hi - 1) f(32 + __builtin_ctz(hi));
}
// Move writers.  squares(m, full, piece, f): one move f(square) per square of
// m, those on `full` to be counted in full (see Gen); add(move, piece): one
// such move; skipped(m): quiet moves.  They are bounded: a writer never
// stores past its cap, but keeps counting so a caller can detect a mismatch
// with the counted size.
struct MoveSink {
    u16 *out;
    u32 cap, n;
    PG_HD void add(u32 m, u32) {
        if (n < cap) out[n] = (u16)m;
        n++;
    }
    template <class F> PG_HD void squares(u64 m, u64, u32 piece, F &&f) {
        each_square(m, [&](int to) { add(f(to), piece); });
    }
    PG_HD void skipped(u64) {}
};
// A window of words, move | owner << 16 | moving piece and kind of move (M_*)
// << 24, so that the child can be made without looking the piece up.  Moves
// past the cap (>= 1) land on its last slot.
struct WordSink {
    u32 *out;
    u32 cap, n, owner;
    PG_HD void add(u32 m, u32 piece) {
        out[n < cap ? n : cap - 1] = m | owner << 16 | piece << 24;
        n++;
    }
    template <class F> PG_HD void squares(u64 m, u64, u32 piece, F &&f) {
        each_square(m, [&](int to) { add(f(to), piece); });
    }
    PG_HD void skipped(u64) {}
};
// The fused leaf's window of `cap` words: calm moves upwards from place
// `calm`, the others downwards from place `full`.  A place out of the window
// (the numbers listed and counted differ) becomes its last.
struct LeafSink {
    u32 *word;
    u32 cap, owner, calm, full;
    PG_HD void put(u32 m, u32 piece, u32 isFull) {
        const u32 at = isFull ? full : calm;
        word[at < cap ? at : cap - 1] = m | owner << 16 | piece << 24;
        full -= isFull;
        calm += isFull ^ 1;
    }
    PG_HD void add(u32 m, u32 piece) { put(m, piece, 1); }
    template <class F> PG_HD void squares(u64 m, u64 on, u32 piece, F &&f) {
        each_square(m, [&](int to) { put(f(to), piece, (u32)(on >> to) & 1); });
    }
    PG_HD void skipped(u64) {}
};
struct NoSink {
    PG_HD void add(u32, u32) {}
};

// en-passant: number of legal captures (MoveGeneratorBitboard.h:3050-3085,
// and :2891-2902 when in check), each handed to the sink.
template <int C, class Sink>
PG_HD int ep_moves(const Sides &s, const Tables &t, const MoveCtx &x, Sink &out) {
    const int f = (int)s.ep;
    if (!f) return 0;
    const u64 dst = C == WHITE ? bit(39 + f) : bit(15 + f);
    const u64 cap = C == WHITE ? dst >> 8 : dst << 8;
    u64 src = (((cap << 1) & ~FILEA) | ((cap >> 1) & ~FILEH)) & s.myPawns;
    int n = 0;
    const int to = ctz(dst);
    if (x.checkers) {
        if (x.checkers != cap) return 0;
        src &= ~x.pinned;
        for (; src; src &= src - 1) {
            out.add((u32)(ctz(src) | (to << 6) | (MF_EP_CAPTURE << 12)), M_PAWN | M_SPECIAL);
            n++;
        }
        return n;
    }
    for (; src; src &= src - 1) {
        const int q = ctz(src);
        bool ok;
        if (x.pinned & bit(q)) {
            ok = (dst & t.line[(q << 6) | s.k]) != 0;
        } else {
            // both pawns leave the rank: no rook or queen may then see the king along it
            const u64 e = ~s.occ | cap | bit(q), eH = andn(e, FILEH), eA = andn(e, FILEA);
            const u64 ray = (eH ^ east_sum(s.eRooks, eH)) | (eA ^ rev64(east_sum(rev64(s.eRooks), rev64(eA))));
            ok = (ray & s.myKing) == 0;
        }
        if (ok) {
            out.add((u32)(q | (to << 6) | (MF_EP_CAPTURE << 12)), M_PAWN | M_SPECIAL);
            n++;
        }
    }
    return n;
}

// Castling moves: bit 0 king side, bit 1 queen side.  The squares lie in one
// byte of the back rank; in it, e is bit 4.
template <int C>
PG_HD u32 castle_bits(u64 occupied, u64 attacked, u32 rights, u64 checkers) {
    const u32 occ = C == WHITE ? (u32)occupied : (u32)(occupied >> 56);
    const u32 att = C == WHITE ? (u32)attacked : (u32)(attacked >> 56);
    const u32 kside = (occ | att) >> 5;                   // f, g neither occupied nor attacked
    const u32 qside = ((occ & 0x0E) | (att & 0x0C)) >> 1; // b, c, d not occupied, c, d not attacked
    const u32 stop = ((kside | kside >> 1) & 1) | ((qside | qside >> 1 | qside >> 2) & 1) << 1;
    return checkers ? 0u : rights & ~stop;
}
template <int C>
PG_HD u32 castle_moves(const Sides &s, const MoveCtx &x) {
    return castle_bits<C>(s.occ, x.threatened, s.castle, x.checkers);
}

// ---------------------------------------------------------------- count
// Knights per piece (pinned knights never move): one table lookup and
// popcount each.
struct KnightLoop {
    PG_HD int operator()(u64 knights, u64 tgt, const Tables &t) const {
        int n = 0;
        for (u64 b = knights; b; b &= b - 1) n += popc(t.knight[ctz(b)] & tgt);
        return n;
    }
};

// n + the pawns' moves but en passant; pf, pw, pe: those that may push, take
// westwards, take eastwards
template <int C>
PG_HD int pawn_moves(u64 pf, u64 pw, u64 pe, u64 empty, u64 enemy, u64 tgt, int n) {
    // pushes on the low or high half only where the rank allows
    const u64 PROMO = C == WHITE ? RANK8 : RANK1;
    const u64 p1 = fwd<C>(pf) & empty;
    const u64 p2 = fwd<C>(p1 & (C == WHITE ? RANK3 : RANK6)) & empty & tgt;
    const u64 t1 = p1 & tgt;
    n = popc_add(t1, popc_add(p2, n));
    const u64 et = enemy & tgt;
    const u64 cw = and3(C == WHITE ? shift<7>(pw) : shift<-9>(pw), ~FILEH, et);
    const u64 ce = and3(C == WHITE ? shift<9>(pe) : shift<-7>(pe), ~FILEA, et);
    n = popc_add(cw, popc_add(ce, n));
    // a move to the last rank is four (one half of each word holds that rank)
    return n + 3 * (popc(t1 & PROMO) + popc(cw & PROMO) + popc(ce & PROMO));
}

template <int C, class Knights> PG_HD u32 count_sides_ks(const Sides &s, const Tables &t, const Knights &knights);

template <int C, int V, class Knights>
PG_HD u32 count_sides(const Sides &s, const Tables &t, const Knights &knights) {
    if constexpr (V == SL_KOGGE) return count_sides_ks<C>(s, t, knights);
    MoveCtx x;
    prologue<C, V>(s, t, x);
    const u64 tgt = x.target, empty = ~s.occ;
    int n = popc(and_nor(t.king[s.k], s.mine, x.threatened));
    if (tgt == 0) return n;  // double check: king moves only

    // movers; a pinned piece moves only along its pin line
    u64 pf = s.myPawns, pw = s.myPawns, pe = s.myPawns, myN = s.myKnights;
    if (x.pinned) {
        const u64 np = ~x.pinned;
        const KingRow &row = t.row[s.k];
        pf = and_or(s.myPawns, np, row.file);
        pw = and_or(s.myPawns, np, C == WHITE ? row.anti : row.diag);
        pe = and_or(s.myPawns, np, C == WHITE ? row.diag : row.anti);
        myN = andn(myN, x.pinned);
    }

    // pawns
    const u64 PROMO = C == WHITE ? RANK8 : RANK1;
    const u64 p1 = fwd<C>(pf) & empty;
    const u64 p2 = fwd<C>(p1 & (C == WHITE ? RANK3 : RANK6)) & empty & tgt;
    const u64 t1 = p1 & tgt;
    n += popc(t1) + 3 * popc(t1 & PROMO) + popc(p2);
    const u64 et = s.enemy & tgt;
    const u64 cw = and3(C == WHITE ? shift<7>(pw) : shift<-9>(pw), ~FILEH, et);
    const u64 ce = and3(C == WHITE ? shift<9>(pe) : shift<-7>(pe), ~FILEA, et);
    n += popc(cw) + 3 * popc(cw & PROMO) + popc(ce) + 3 * popc(ce & PROMO);

    n += knights(myN, tgt, t);

    // sliders, per piece
    for (u64 b = s.myBishops; b; b &= b - 1) {
        const int q = ctz(b);
        u64 m = Sl<V>::bishop(t, q, s.occ) & tgt;
        if (x.pinned & bit(q)) m &= t.line[(q << 6) | s.k];
        n += popc(m);
    }
    for (u64 r = s.myRooks; r; r &= r - 1) {
        const int q = ctz(r);
        u64 m = Sl<V>::rook(t, q, s.occ) & tgt;
        if (x.pinned & bit(q)) m &= t.line[(q << 6) | s.k];
        n += popc(m);
    }
    n += popc((u64)castle_moves<C>(s, x));
    NoSink none;
    n += ep_moves<C>(s, t, x, none);
    return (u32)n;
}

// ---------------------------------------------------------------- count, Kogge-Stone
// The Kogge-Stone count in one pass over the eight directions, written to
// keep the VALU instruction count down:
//  * and/or chains are three-input bitop3 instructions (two per 64-bit word);
//  * each direction's propagator chain (empty, empty & empty<<s, ...) is
//    built once and shared by the enemy-attack fill and the own-move fill;
//  * enemy sliders fill through empty squares only; the one square the
//    moving king must not step to because a slider checks it through the
//    king ("behind" it on the check line) is added explicitly;
//  * east rays of every slider at once by one add: with the h-file as
//    sentinel, o = occ | FILEH and e = ~o, the squares from each slider up
//    to its first blocker are o ^ (o - 2s) = e ^ (e + 2s); west rays the
//    same on the bit-reversed board;
//  * pinned pieces need the king-line masks only when something is pinned.
template <int C, class Knights>
PG_HD u32 count_sides_ks(const Sides &s, const Tables &t, const Knights &knights) {
    MoveCtx x;
    const KingRow &row = t.row[s.k];
    const u64 eB = s.eBishops, eR = s.eRooks;
    const u64 behind = pins_and_checks<C>(s, t, x);
    const u64 tgt = x.target;

    // movers; a pinned piece moves only along its pin line
    const u64 rq = s.myRooks, bq = s.myBishops;
    u64 rf = rq, rr = rq, bd = bq, ba = bq, pf = s.myPawns, pw = s.myPawns, pe = s.myPawns;
    u64 myN = s.myKnights;
    if (x.pinned) {
        const u64 np = ~x.pinned;
        rf = and_or(rq, np, row.file);
        rr = and_or(rq, np, row.rank);
        bd = and_or(bq, np, row.diag);
        ba = and_or(bq, np, row.anti);
        pf = and_or(s.myPawns, np, row.file);
        pw = and_or(s.myPawns, np, C == WHITE ? row.anti : row.diag);
        pe = and_or(s.myPawns, np, C == WHITE ? row.diag : row.anti);
        myN = andn(myN, x.pinned);
    }

    // enemy attacks without sliders: king, pawns, knights
    u64 att = leaper_attacks<C>(s, t) | behind;

    const u64 empty = ~s.occ;
    int n = 0;
    {   // north and south
        const Prop3 pn = props<8>(empty), ps = props<-8>(empty);
        const u64 an = grow<8>(eR, pn), as = grow<-8>(eR, ps);
        att = or3(att, shift<8>(an), shift<-8>(as));
        n = popc_add((grow<8>(rf, pn) << 8) & tgt, n);
        n = popc_add((grow<-8>(rf, ps) >> 8) & tgt, n);
    }
    const u64 eA = nor2(s.occ, FILEA), eH = nor2(s.occ, FILEH);
    {   // east: one add per side
        att = or_xor(att, eH, east_sum(eR, eH));
        n = popc_add(xor_and(eH, east_sum(rr, eH), tgt), n);
    }
    {   // west: east on the bit-reversed board
        const u64 eoR = rev64(eA);
        att = or_xor(att, eA, rev64(east_sum(rev64(eR), eoR)));
        n = popc_add(xor_and(eA, rev64(east_sum(rev64(rr), eoR)), tgt), n);
    }
    {   // north-east and south-west
        const Prop3 pa = props<9>(eA), pb = props<-9>(eH);
        att = or_and(att, shift<9>(grow<9>(eB, pa)), ~FILEA);
        att = or_and(att, shift<-9>(grow<-9>(eB, pb)), ~FILEH);
        n = popc_add(and3(shift<9>(grow<9>(bd, pa)), ~FILEA, tgt), n);
        n = popc_add(and3(shift<-9>(grow<-9>(bd, pb)), ~FILEH, tgt), n);
    }
    {   // north-west and south-east
        const Prop3 pa = props<7>(eH), pb = props<-7>(eA);
        att = or_and(att, shift<7>(grow<7>(eB, pa)), ~FILEH);
        att = or_and(att, shift<-7>(grow<-7>(eB, pb)), ~FILEA);
        n = popc_add(and3(shift<7>(grow<7>(ba, pa)), ~FILEH, tgt), n);
        n = popc_add(and3(shift<-7>(grow<-7>(ba, pb)), ~FILEA, tgt), n);
    }
    x.threatened = att;
    n = popc_add(and_nor(row.king, s.mine, att), n);

    n = pawn_moves<C>(pf, pw, pe, empty, s.enemy, tgt, n);
    n += knights(myN, tgt, t);
    n += popc((u64)castle_moves<C>(s, x));
    NoSink none;
    n += ep_moves<C>(s, t, x, none);
    return (u32)n;
}

template <int C, int V>
PG_HD u32 count_moves(const Pos &p, const Tables &t) {
    return count_sides<C, V>(sides_of<C>(p), t, KnightLoop());
}

// ---------------------------------------------------------------- generate
PG_HD u32 mk_move(int from, int to, int flags) { return (u32)(from | (to << 6) | (flags << 12)); }

// What the moves of a side follow from.  A move between two squares of the
// quiet set of its piece (qP, qN, qB, qR; a queen's is qB & qR) is left out;
// one between two squares of its calm set (zP, ...) is calm (see quiet
// moves).  king, kingFull: the king's moves that are not quiet, not calm.
struct Gen {
    u64 pinned, checkers, target, king, kingFull;
    u64 qP, qN, qB, qR, zP, zN, zB, zR;
    u32 castle;
};

template <int C, int V>
PG_HD Gen gen_all(const Sides &s, const Tables &t) {
    MoveCtx x;
    prologue<C, V>(s, t, x);
    return Gen{x.pinned, x.checkers, x.target, and_nor(t.row[s.k].king, s.mine, x.threatened), 0, 0, 0, 0, 0, 0, 0, 0, 0,
               castle_moves<C>(s, x)};
}

// Hands the legal moves of s that are not left out to the sink (at most 218 in
// a game; boards set up with 26 queens have 278).
// Pawn captures carry the capture flag; other captures do not, as on the
// reference's device path (MoveGeneratorBitboard.h:2525-2529).
// First the king's and the pawns' moves and castling; false if the king alone
// may move.
template <int C, class Sink>
PG_HD bool king_pawn_moves(const Sides &s, const Gen &g, const Tables &t, Sink &o) {
    const u64 tgt = g.target, empty = ~s.occ;
    o.squares(g.king, g.kingFull, M_KING, [&](int to) { return mk_move(s.k, to, MF_QUIET); });
    if (tgt == 0) return false;

    // a pinned pawn moves only along its pin line
    u64 pf = s.myPawns, pw = s.myPawns, pe = s.myPawns;
    if (g.pinned) {
        const u64 np = ~g.pinned;
        const KingRow &row = t.row[s.k];
        pf = and_or(s.myPawns, np, row.file);
        pw = and_or(s.myPawns, np, C == WHITE ? row.anti : row.diag);
        pe = and_or(s.myPawns, np, C == WHITE ? row.diag : row.anti);
    }
    const int up = C == WHITE ? 8 : -8;
    const u64 PROMO = C == WHITE ? RANK8 : RANK1;
    auto promos = [&](u64 m, int back, int cap) {
        each_square(m, [&](int to) {
            o.add(mk_move(to - back, to, MF_PROMO | cap | 0), M_PAWN | M_SPECIAL);
            o.add(mk_move(to - back, to, MF_PROMO | cap | 1), M_PAWN | M_SPECIAL);
            o.add(mk_move(to - back, to, MF_PROMO | cap | 3), M_PAWN | M_SPECIAL);
            o.add(mk_move(to - back, to, MF_PROMO | cap | 2), M_PAWN | M_SPECIAL);
        });
    };
    // pushes
    const u64 p1 = fwd<C>(pf) & empty;
    const u64 p2 = fwd<C>(p1 & (C == WHITE ? RANK3 : RANK6)) & empty & tgt;
    const u64 t1 = p1 & tgt;
    const u64 beside = (andn(s.ePawns, FILEH) << 1) | (andn(s.ePawns, FILEA) >> 1);
    const u64 q1 = and3(andn(t1, PROMO), g.qP, fwd<C>(g.qP)), q2 = andn(and3(p2, g.qP, fwd<C>(fwd<C>(g.qP))), beside);
    o.skipped(q1);
    o.skipped(q2);
    o.squares(and_nor(t1, PROMO, q1), ~(g.zP & fwd<C>(g.zP)), M_PAWN, [&](int to) { return mk_move(to - up, to, MF_QUIET); });
    promos(t1 & PROMO, up, 0);
    o.squares(and_nor(p2, q2, beside), ~(g.zP & fwd<C>(fwd<C>(g.zP))), M_PAWN,
              [&](int to) { return mk_move(to - 2 * up, to, MF_DOUBLE_PUSH); });
    o.squares(p2 & beside, ~0ULL, M_PAWN | M_SPECIAL, [&](int to) { return mk_move(to - 2 * up, to, MF_DOUBLE_PUSH); });
    // captures
    const u64 et = s.enemy & tgt;
    const u64 cw = and3(C == WHITE ? shift<7>(pw) : shift<-9>(pw), ~FILEH, et);
    const u64 ce = and3(C == WHITE ? shift<9>(pe) : shift<-7>(pe), ~FILEA, et);
    constexpr int dw = C == WHITE ? 7 : -9, de = C == WHITE ? 9 : -7;
    o.squares(andn(cw, PROMO), ~(g.zP & shift<dw>(g.zP)), M_PAWN, [&](int to) { return mk_move(to - dw, to, MF_CAPTURE); });
    o.squares(andn(ce, PROMO), ~(g.zP & shift<de>(g.zP)), M_PAWN, [&](int to) { return mk_move(to - de, to, MF_CAPTURE); });
    promos(cw & PROMO, dw, MF_CAPTURE);
    promos(ce & PROMO, de, MF_CAPTURE);
    MoveCtx x;
    x.pinned = g.pinned;
    x.checkers = g.checkers;
    ep_moves<C>(s, t, x, o);
    // castling
    constexpr int e = C == WHITE ? 4 : 60;
    if (g.castle & 1) o.add(mk_move(e, e + 2, MF_KING_CASTLE), M_KING | M_SPECIAL);
    if (g.castle & 2) o.add(mk_move(e, e - 2, MF_QUEEN_CASTLE), M_KING | M_SPECIAL);
    return true;
}

template <int C, int V, class Sink>
PG_HD void generate_sides(const Sides &s, const Gen &g, const Tables &t, Sink &o) {
    if (!king_pawn_moves<C>(s, g, t, o)) return;
    const u64 tgt = g.target;
    // a piece on q with moves m, its quiet and calm sets
    auto moves = [&](int q, u64 m, u64 quiet, u64 calm, u32 piece) {
        const u64 left = and3(m, quiet, mask_if((quiet >> q) & 1));
        o.skipped(left);
        o.squares(andn(m, left), ~(calm & mask_if((calm >> q) & 1)), piece, [&](int to) { return mk_move(q, to, MF_QUIET); });
    };
    // knights (pinned knights never move)
    for (u64 b = andn(s.myKnights, g.pinned); b; b &= b - 1) {
        const int q = ctz(b);
        moves(q, t.knight[q] & tgt, g.qN, g.zN, M_KNIGHT);
    }
    // sliders
    for (u64 b = s.myBishops; b; b &= b - 1) {
        const int q = ctz(b);
        u64 m = Sl<V>::bishop(t, q, s.occ) & tgt;
        if (g.pinned & bit(q)) m &= t.line[(q << 6) | s.k];
        const bool queen = s.myRooks & bit(q);
        moves(q, m, queen ? g.qB & g.qR : g.qB, queen ? g.zB & g.zR : g.zB, queen ? M_QUEEN : M_BISHOP);
    }
    for (u64 r = s.myRooks; r; r &= r - 1) {
        const int q = ctz(r);
        u64 m = Sl<V>::rook(t, q, s.occ) & tgt;
        if (g.pinned & bit(q)) m &= t.line[(q << 6) | s.k];
        const bool queen = s.myBishops & bit(q);
        moves(q, m, queen ? g.qB & g.qR : g.qR, queen ? g.zB & g.zR : g.zR, queen ? M_QUEEN : M_ROOK);
    }
}

// Writes the legal moves of p to out (at most cap of them); returns the
// number of legal moves.
template <int C, int V>
PG_HD u32 generate_moves(const Pos &p, const Tables &t, u16 *out, u32 cap) {
    MoveSink o{out, cap, 0};
    const Sides s = sides_of<C>(p);
    generate_sides<C, V>(s, gen_all<C, V>(s, t), t, o);
    return o.n;
}

// ---------------------------------------------------------------- kin
// A board as its children see it: the fused leaf keeps its boards in this
// form in LDS.  Most of a child is its parent unchanged, so what would be
// worked out for every child is worked out once: the piece words by side, the
// kings' squares, and the attack sets of the first two knights of the side
// that will reply.  A child then takes one xor or and-not per word instead of
// a make-move on the combined words and the split by side after it.
struct Kin {
    u64 bP, bN, bB, bR;  // the replying side
    u64 aP, aN, aB, aR;  // the side to move
    u64 occ, mine;       // all men, the replying side's
    u64 n0, n1;          // attacks of the first two of bN
    u64 pinned;          // the replying side's pinned men if the other passes
    u32 info;            // see KIN_*
    u32 knights;         // squares of the first two of bN: 6 bits each; KIN_MORE: there are others; king and
                         // castling moves if the other side passes << KIN_STAY
};
static_assert(sizeof(Kin) == 104 + 8, "a tile of 64 boards is 7 KB of its wave's LDS");
// info: king squares (replying side, side to move), castling rights (replying
// side, side to move), en-passant file + 1, side to move
enum { KIN_EK = 6, KIN_CASTLE = 12, KIN_MYCASTLE = 14, KIN_EP = 16, KIN_SIDE = 20 };
constexpr u32 KIN_MORE = 1u << 12;
constexpr int KIN_STAY = 13;

template <int A> PG_HD Kin kin_of(const Sides &s, const Tables &t) {
    Kin k;
    k.bP = s.ePawns;
    k.bN = s.eKnights;
    k.bB = s.eBishops;
    k.bR = s.eRooks;
    k.aP = s.myPawns;
    k.aN = s.myKnights;
    k.aB = s.myBishops;
    k.aR = s.myRooks;
    k.occ = s.occ;
    k.mine = s.enemy;
    k.n0 = k.n1 = k.pinned = 0;
    k.knights = 0;
    u64 n = k.bN;
    if (n) {
        const int q = ctz(n);
        k.n0 = t.knight[q];
        k.knights = (u32)q;
        n &= n - 1;
        if (n) {
            const int r = ctz(n);
            k.n1 = t.knight[r];
            k.knights |= (u32)r << 6 | (several(n) ? KIN_MORE : 0u);
        }
    }
    k.info = (u32)s.ek | (u32)s.k << KIN_EK | s.eCastle << KIN_CASTLE | s.castle << KIN_MYCASTLE | s.ep << KIN_EP |
             (u32)A << KIN_SIDE;
    return k;
}

// the board itself again, as the side to move sees it
PG_HD Sides sides_of_kin(const Kin &k) {
    Sides s;
    s.occ = k.occ;
    s.mine = andn(k.occ, k.mine);
    s.enemy = k.mine;
    s.myPawns = k.aP;
    s.myKnights = k.aN;
    s.myBishops = k.aB;
    s.myRooks = k.aR;
    s.ePawns = k.bP;
    s.eKnights = k.bN;
    s.eBishops = k.bB;
    s.eRooks = k.bR;
    s.ek = (int)(k.info & 63);
    s.k = (int)(k.info >> KIN_EK & 63);
    s.myKing = bit(s.k);
    s.castle = k.info >> KIN_MYCASTLE & 3;
    s.eCastle = k.info >> KIN_CASTLE & 3;
    s.ep = k.info >> KIN_EP & 15;
    return s;
}

// popcount of the knights' moves with the parent's attack sets of the first
// two: a knight that was captured or is pinned is not in `knights`
struct KinKnights {
    const Kin &k;
    PG_HD int operator()(u64 knights, u64 tgt, const Tables &t) const {
        const int q = (int)(k.knights & 63), r = (int)(k.knights >> 6 & 63);
        const u32 m0 = (u32)((int)((u32)(knights >> q) << 31) >> 31), m1 = (u32)((int)((u32)(knights >> r) << 31) >> 31);
        int n = popc_add(and3(k.n0, tgt, (u64)m0 << 32 | m0), popc_add(and3(k.n1, tgt, (u64)m1 << 32 | m1), 0));
        if (k.knights & KIN_MORE) n += KnightLoop()(and_nor(knights, bit(q), bit(r)), tgt, t);
        return n;
    }
};

// Number of legal replies (by side B) after the move of window word `w`, not
// a special one, from the board k.
template <int B, int V>
PG_HD u32 count_child(const Kin &k, u32 w, const Tables &t) {
    const int to = (int)(w >> 6 & 63);
    const u64 src = bit((int)(w & 63)), dst = bit(to), both = src | dst;
    // the moving piece's words change on both squares, its enemy's lose the target
    const auto moved = [&](u64 x, int i) {
        const u32 m = (u32)((int)(w << (7 - i)) >> 31);
        return bop3<0x78>(x, both, (u64)m << 32 | m);  // x ^ (both & m)
    };
    Sides s;
    s.ePawns = moved(k.aP, 0);
    s.eKnights = moved(k.aN, 1);
    s.eBishops = moved(k.aB, 2);
    s.eRooks = moved(k.aR, 3);
    s.myPawns = andn(k.bP, dst);
    s.myKnights = andn(k.bN, dst);
    s.myBishops = andn(k.bB, dst);
    s.myRooks = andn(k.bR, dst);
    s.occ = bop3<0xBA>(k.occ, src, dst);  // (occ & ~src) | dst
    s.mine = andn(k.mine, dst);
    s.enemy = andn(s.occ, s.mine);
    s.k = (int)(k.info & 63);
    s.myKing = bit(s.k);
    s.ek = w >> 28 & 1 ? to : (int)(k.info >> KIN_EK & 63);
    // a move to a corner takes that side's right, as make_move
    const u32 edge = B == WHITE ? (u32)dst : (u32)(dst >> 56);
    s.castle = k.info >> KIN_CASTLE & 3 & ~((edge >> 7 & 1) | (edge & 1) << 1);
    s.eCastle = 0;
    s.ep = 0;
    return count_sides<B, V>(s, t, KinKnights{k});
}

// the board itself again (clock 0)
PG_HD Pos pos_of_kin(const Kin &k) {
    const u32 side = k.info >> KIN_SIDE & 1, mine = k.info >> KIN_MYCASTLE & 3, theirs = k.info >> KIN_CASTLE & 3;
    Pos p;
    p.white = side ? k.mine : andn(k.occ, k.mine);
    p.pawns = k.aP | k.bP | (u64)(side ? theirs | mine << 2 : mine | theirs << 2) | (u64)side << 63;
    p.knights = k.aN | k.bN;
    p.bishopQueens = k.aB | k.bB;
    p.rookQueens = k.aR | k.bR;
    p.kings = bit((int)(k.info & 63)) | bit((int)(k.info >> KIN_EK & 63));
    return p;
}

// ---------------------------------------------------------------- quiet moves
// Most moves change little of what the other side could do.  Let side A be to
// move, B not in check, and let the zone be B's king, the squares it could step
// to, and those it would cross castling.
//
// A move of A from s to t that is not special (M_SPECIAL) is calm when neither
// s nor t is
//  * on an open line between a slider of A and a zone square, first blockers
//    included, or on a line between a slider of A and B's king, whatever
//    stands on it: then no other slider's view of the zone changes, nor a pin
//    on a man of B;
//  * one from which the moved piece itself reaches the zone: a pawn's, knight's
//    or king's step from it; for a slider an open line, or the line of B's
//    king (a pin);
//  * between king and rook where B may still castle, or that rook's corner, or
//    a man of B next to its king.
// After it B is not in check, its pins are those it would have if A passed,
// and so are its king's and castling moves: only its sliders, pawns and
// knights need counting (count_calm).
//
// A calm move to an empty square is quiet when moreover neither s nor t is on
// a ray of a slider of B (up to and including its first blocker), in front of
// a pawn of B within its push, or on a square it attacks: then every man of B
// has the moves it would have if A passed (a knight's do not depend on s and
// t), so the replies to the quiet moves are their number times that count, and
// the moves are not even listed.
//
// Of the moves of all positions four plies into the game 74% are quiet and 21%
// calm; in random games 59 and 29% up to ply 19, 38 and 36% to ply 39, 30 and
// 35% to ply 59, 25 to 30 and 15 to 31% later.
struct LeafEval {
    Gen g;
    u32 calm, full, quiet;  // numbers of moves
    u32 c0;                 // replies to each quiet move
};

// keeps the compiler from carrying what it loaded from LDS in registers past
// this point (it is loaded again)
PG_HD void reload() {
#if defined(__HIP_DEVICE_COMPILE__)
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#endif
}

// k: the board (kin_of); its pins and staying moves are filled in.
template <int A>
PG_HD LeafEval leaf_eval(Kin &k, const Tables &t) {
    constexpr int B = 1 - A, sh = B == WHITE ? 0 : 56;
    Sides s = sides_of_kin(k);
    const KingRow &ra = t.row[s.k], &rb = t.row[s.ek];
    const u64 e = ~s.occ, kb = bit(s.ek), aB = s.myBishops, aR = s.myRooks, bB = s.eBishops, bR = s.eRooks;
    LeafEval r;
    Gen &g = r.g;
    MoveCtx x;
    const u64 behind = pins_and_checks<A>(s, t, x);
    const u64 tgtA = x.target, tgtB = ~s.enemy;

    // B's pins and checks, the zone, and the squares that are not calm for any
    // piece: on lines between B's king and sliders of A, ...
    u64 zone = andn(rb.king, s.enemy) | kb, tied = rb.king & s.enemy, pinB = 0, chkB = 0;
    if (s.eCastle & 1) {
        zone |= 0x60ULL << sh;
        tied |= 0xE0ULL << sh;
    }
    if (s.eCastle & 2) {
        zone |= 0x0CULL << sh;
        tied |= 0x0FULL << sh;
    }
    for (u64 c = or_and(rb.rook & aR, rb.bishop, aB); c; c &= c - 1) {
        const int q = ctz(c);
        const u64 btw = t.pin[(s.ek << 6) | q].between, on = btw & s.occ;
        pinB = or_and(pinB, on, mask_if(!several(on)));
        tied = or3(tied, btw, bit(q));
        chkB = or_and(chkB, bit(q), mask_if(on == 0));
    }
    pinB &= s.enemy;
    chkB = or_and(or_and(chkB, rb.knight, s.myKnights), pawn_att<B>(kb), s.myPawns);

    // one pass over the directions, B's sliders, A's and the zone's view
    // through the same propagators: the two sides' slider moves, the squares
    // each attacks, the open lines between A and the zone, and where a slider
    // of A would reach the zone from
    const u64 pB = pawn_att<B>(s.ePawns);
    u64 attA = or3(t.king[s.k], pawn_att<A>(s.myPawns), knight_att(s.myKnights));
    u64 raysB = 0, zR = rb.rook, zB = rb.bishop;
    int nA = 0, nB = 0;
    const auto pair = [&](auto dir, const Prop3 &pu, const Prop3 &pd, u64 mu, u64 md, u64 a, u64 b, u64 &z) {
        constexpr int S = decltype(dir)::value;
        const u64 au = and_mask(shift<S>(grow<S>(a, pu)), mu), ad = and_mask(shift<-S>(grow<-S>(a, pd)), md);
        const u64 zu = and_mask(shift<S>(grow<S>(zone, pu)), mu), zd = and_mask(shift<-S>(grow<-S>(zone, pd)), md);
        const u64 bu = and_mask(shift<S>(grow<S>(b, pu)), mu), bd = and_mask(shift<-S>(grow<-S>(b, pd)), md);
        nA = popc_add(au & tgtA, popc_add(ad & tgtA, nA));
        nB = popc_add(bu & tgtB, popc_add(bd & tgtB, nB));
        tied = or_and(or_and(tied, au, zd), ad, zu);
        attA = or3(attA, au, ad);
        raysB = or3(raysB, bu, bd);
        z = or3(z, zu, zd);
    };
    const u64 eA = andn(e, FILEA), eH = andn(e, FILEH);
    pair(Int<8>(), props<8>(e), props<-8>(e), ~0ULL, ~0ULL, aR, bR, zR);
    pair(Int<1>(), props<1>(eA), props<-1>(eH), ~FILEA, ~FILEH, aR, bR, zR);
    pair(Int<9>(), props<9>(eA), props<-9>(eH), ~FILEA, ~FILEH, aB, bB, zB);
    pair(Int<7>(), props<7>(eH), props<-7>(eA), ~FILEH, ~FILEA, aB, bB, zB);
    // pinned sliders were counted as if they could leave their line
    const auto bound = [&](u64 pins, u64 bishops, u64 rooks, u64 tgt, int king) {
        int n = 0;
        for (u64 c = and_or(pins, bishops, rooks); c; c &= c - 1) {
            const int q = ctz(c);
            const u64 off = andn(tgt, t.line[(q << 6) | king]);
            n = popc_add(and3(Sl<SL_KOGGE>::bishop(t, q, s.occ), off, mask_if((bishops >> q) & 1)), n);
            n = popc_add(and3(Sl<SL_KOGGE>::rook(t, q, s.occ), off, mask_if((rooks >> q) & 1)), n);
        }
        return n;
    };
    if (x.pinned) nA -= bound(x.pinned, aB, aR, tgtA, s.k);
    if (pinB) nB -= bound(pinB, bB, bR, tgtB, s.ek);

    // B's moves if A passed
    const u32 stay = (u32)popc(and_nor(rb.king, s.enemy, attA)) +
                     (u32)popc((u64)castle_bits<B>(s.occ, attA, s.eCastle, 0));
    {
        u64 pf = s.ePawns, pw = pf, pe = pf;
        if (pinB) {
            const u64 np = ~pinB;
            pf = and_or(pf, np, rb.file);
            pw = and_or(pw, np, B == WHITE ? rb.anti : rb.diag);
            pe = and_or(pe, np, B == WHITE ? rb.diag : rb.anti);
        }
        nB = pawn_moves<B>(pf, pw, pe, e, s.mine, tgtB, nB);
    }
    nB += KinKnights{k}(andn(s.eKnights, pinB), tgtB, t);
    r.c0 = (u32)nB + stay;
    k.pinned = pinB;
    k.knights = (k.knights & (2 * KIN_MORE - 1)) | stay << KIN_STAY;
    reload();
    s = sides_of_kin(k);

    // the calm and quiet sets
    const u64 calm = andn(mask_if(chkB == 0), tied);
    const u64 pawnHome = B == WHITE ? RANK1 << 8 : RANK8 >> 8;
    const u64 push = fwd<B>(s.ePawns) | fwd<B>(fwd<B>(s.ePawns & pawnHome));
    const u64 still = andn(~or3(raysB, push, pB), s.enemy);
    g.zP = andn(calm, pawn_att<B>(zone));
    g.zN = andn(calm, knight_att(zone));
    g.zB = andn(calm, zB);
    g.zR = andn(calm, zR);
    g.qP = g.zP & still;
    g.qN = g.zN & still;
    g.qB = g.zB & still;
    g.qR = g.zR & still;
    const u64 zK = andn(calm, king_att(zone)), zKm = zK & mask_if((zK >> s.k) & 1);

    // A's moves by kind
    g.pinned = x.pinned;
    g.checkers = x.checkers;
    g.target = tgtA;
    const u64 attB = or3(t.king[s.ek], pB, or3(knight_att(s.eKnights), behind, raysB));
    const u64 kings = and_nor(ra.king, s.mine, attB);
    const u64 kq = and3(kings, zKm, still & mask_if((still >> s.k) & 1));
    g.king = andn(kings, kq);
    g.kingFull = andn(kings, zKm);
    g.castle = castle_bits<A>(s.occ, attB, s.castle, x.checkers);
    int all = nA + popc(kings) + popc((u64)g.castle), quiet = popc(kq), notFull = popc(kings & zKm);  // notFull: calm or quiet
    if (tgtA) {
        u64 pf = s.myPawns, pw = pf, pe = pf;
        if (x.pinned) {
            const u64 np = ~x.pinned;
            pf = and_or(pf, np, ra.file);
            pw = and_or(pw, np, A == WHITE ? ra.anti : ra.diag);
            pe = and_or(pe, np, A == WHITE ? ra.diag : ra.anti);
        }
        const u64 PROMO = A == WHITE ? RANK8 : RANK1;
        const u64 beside = (andn(s.ePawns, FILEH) << 1) | (andn(s.ePawns, FILEA) >> 1);
        const u64 p1 = fwd<A>(pf) & e, p2 = fwd<A>(p1 & (A == WHITE ? RANK3 : RANK6)) & e & tgtA;
        const u64 t1 = p1 & tgtA, s1 = andn(t1, PROMO), s2 = andn(p2, beside);
        const u64 et = s.enemy & tgtA;
        constexpr int dw = A == WHITE ? 7 : -9, de = A == WHITE ? 9 : -7;
        const u64 cw = and3(shift<dw>(pw), ~FILEH, et), ce = and3(shift<de>(pe), ~FILEA, et);
        all = popc_add(t1, popc_add(p2, popc_add(cw, popc_add(ce, all))));
        all += 3 * (popc(t1 & PROMO) + popc(cw & PROMO) + popc(ce & PROMO));
        const u64 z1 = fwd<A>(g.zP), z2 = fwd<A>(z1), q1 = fwd<A>(g.qP), q2 = fwd<A>(q1);
        notFull = popc_add(and3(s1, g.zP, z1), popc_add(and3(s2, g.zP, z2), notFull));
        quiet = popc_add(and3(s1, g.qP, q1), popc_add(and3(s2, g.qP, q2), quiet));
        notFull = popc_add(and3(andn(cw, PROMO), g.zP, shift<dw>(g.zP)), notFull);
        notFull = popc_add(and3(andn(ce, PROMO), g.zP, shift<de>(g.zP)), notFull);
        NoSink none;
        all += ep_moves<A>(s, t, x, none);
        const auto kinds = [&](int q, u64 m, u64 zs, u64 qs) {
            notFull = popc_add(and3(m, zs, mask_if((zs >> q) & 1)), notFull);
            quiet = popc_add(and3(m, qs, mask_if((qs >> q) & 1)), quiet);
        };
        for (u64 b = andn(s.myKnights, x.pinned); b; b &= b - 1) {
            const int q = ctz(b);
            const u64 m = t.knight[q] & tgtA;
            all = popc_add(m, all);
            kinds(q, m, g.zN, g.qN);
        }
        const u64 queens = aB & aR;
        for (u64 b = and_or(aB & g.zB, ~queens, g.zR); b; b &= b - 1) {
            const int q = ctz(b);
            const u64 nq = mask_if(!((queens >> q) & 1));
            u64 m = Sl<SL_KOGGE>::bishop(t, q, s.occ) & tgtA;
            if (x.pinned & bit(q)) m &= t.line[(q << 6) | s.k];
            kinds(q, m, and_or(g.zB, nq, g.zR), and_or(g.qB, nq, g.qR));
        }
        for (u64 b = and_or(aR & g.zR, ~queens, g.zB); b; b &= b - 1) {
            const int q = ctz(b);
            const u64 nq = mask_if(!((queens >> q) & 1));
            u64 m = Sl<SL_KOGGE>::rook(t, q, s.occ) & tgtA;
            if (x.pinned & bit(q)) m &= t.line[(q << 6) | s.k];
            kinds(q, m, and_or(g.zR, nq, g.zB), and_or(g.qR, nq, g.qB));
        }
    }
    r.quiet = (u32)quiet;
    r.calm = (u32)(notFull - quiet);
    r.full = (u32)(all - notFull);
    return r;
}

// Number of replies (by side B) after the calm move of window word `w`.
template <int B>
PG_HD u32 count_calm(const Kin &k, u32 w, const Tables &t) {
    const u64 src = bit((int)(w & 63)), dst = bit((int)(w >> 6 & 63));
    const u64 occ = bop3<0xBA>(k.occ, src, dst), mine = andn(k.mine, dst);  // (occ & ~src) | dst
    const u64 tgt = ~mine, empty = ~occ;
    const u64 bq = andn(k.bB, dst), rq = andn(k.bR, dst);
    u64 rf = rq, rr = rq, bd = bq, ba = bq, pf = andn(k.bP, dst), pw = pf, pe = pf, kn = andn(k.bN, dst);
    if (k.pinned) {
        const KingRow &row = t.row[k.info & 63];
        const u64 np = ~k.pinned;
        rf = and_or(rq, np, row.file);
        rr = and_or(rq, np, row.rank);
        bd = and_or(bq, np, row.diag);
        ba = and_or(bq, np, row.anti);
        pw = and_or(pf, np, B == WHITE ? row.anti : row.diag);
        pe = and_or(pf, np, B == WHITE ? row.diag : row.anti);
        pf = and_or(pf, np, row.file);
        kn &= np;
    }
    int n = (int)(k.knights >> KIN_STAY);
    n = popc_add((grow<8>(rf, props<8>(empty)) << 8) & tgt, n);
    n = popc_add((grow<-8>(rf, props<-8>(empty)) >> 8) & tgt, n);
    const u64 eA = nor2(occ, FILEA), eH = nor2(occ, FILEH);
    n = popc_add(xor_and(eH, east_sum(rr, eH), tgt), n);
    n = popc_add(xor_and(eA, rev64(east_sum(rev64(rr), rev64(eA))), tgt), n);
    n = popc_add(and3(shift<9>(grow<9>(bd, props<9>(eA))), ~FILEA, tgt), n);
    n = popc_add(and3(shift<-9>(grow<-9>(bd, props<-9>(eH))), ~FILEH, tgt), n);
    n = popc_add(and3(shift<7>(grow<7>(ba, props<7>(eH))), ~FILEH, tgt), n);
    n = popc_add(and3(shift<-7>(grow<-7>(ba, props<-7>(eA))), ~FILEA, tgt), n);
    n = pawn_moves<B>(pf, pw, pe, empty, andn(occ, mine), tgt, n);
    return (u32)(n + KinKnights{k}(kn, tgt, t));
}

// ---------------------------------------------------------------- make move
// Zobrist word offsets in the 782-word key set (chess.h:326-333)
PG_HD int zob_piece(int color, int piece /*1..6*/, int sq) { return color * 384 + (piece - 1) * 64 + sq; }
constexpr int ZOB_CASTLE = 768, ZOB_EP = 772, ZOB_SIDE = 780;

PG_HD void zob_xor(Key128 &h, const Tables &t, int w) {
    h.lo ^= t.zobLo[w];
    h.hi ^= t.zobHi[w];
}
PG_HD void zob_state(Key128 &h, const Tables &t, const Pos &p) {
    const int w = pos_wcastle(p), b = pos_bcastle(p), e = pos_ep(p);
    if (w & 1) zob_xor(h, t, ZOB_CASTLE + 0);
    if (w & 2) zob_xor(h, t, ZOB_CASTLE + 1);
    if (b & 1) zob_xor(h, t, ZOB_CASTLE + 2);
    if (b & 2) zob_xor(h, t, ZOB_CASTLE + 3);
    if (e) zob_xor(h, t, ZOB_EP + e - 1);
}

PG_HD int piece_on(const Pos &p, u64 b) {
    if (p.kings & b) return P_KING;
    if (p.knights & b) return P_KNIGHT;
    if (pos_pawns(p) & b) return P_PAWN;
    if (p.bishopQueens & p.rookQueens & b) return P_QUEEN;
    if (p.bishopQueens & b) return P_BISHOP;
    if (p.rookQueens & b) return P_ROOK;
    return 0;
}

// Applies a legal move (MoveGeneratorBitboard.h:3575-3836): the en-passant
// file is recorded only when an enemy pawn can take, and castling rights are
// cleared by king moves, rook moves from a corner and captures on a corner.
// With HASH the 128-bit key is updated incrementally.
// make_move_as takes the moving piece from the caller (the generator records
// it); make_move looks it up.
template <int C, bool HASH>
PG_HD void make_move_as(Pos &p, u16 mv, int piece, Key128 *h, const Tables &t) {
    const int from = mv & 63, to = (mv >> 6) & 63, fl = mv >> 12;
    const u64 src = bit(from), dst = bit(to);
    if (HASH) {
        zob_xor(*h, t, zob_piece(C, piece, from));
        const int cap = piece_on(p, dst);
        if (cap) zob_xor(*h, t, zob_piece(1 - C, cap, to));
        zob_xor(*h, t, ZOB_SIDE);
        zob_state(*h, t, p);
    }
    const bool movedRook = piece == P_ROOK;
    if (fl & MF_PROMO) {
        const int pr = fl & 3;  // N, B, R, Q
        piece = pr == 0 ? P_KNIGHT : pr == 1 ? P_BISHOP : pr == 2 ? P_ROOK : P_QUEEN;
    }
    if (HASH) zob_xor(*h, t, zob_piece(C, piece, to));
    const u64 clr = ~(src | dst);
    p.bishopQueens &= clr;
    p.rookQueens &= clr;
    p.kings &= clr;
    p.knights &= clr;
    p.pawns &= ~((src | dst) & RANKS2TO7);
    if (piece == P_KING) p.kings |= dst;
    if (piece == P_KNIGHT) p.knights |= dst;
    if (piece == P_PAWN) p.pawns |= dst;
    if (piece == P_BISHOP || piece == P_QUEEN) p.bishopQueens |= dst;
    if (piece == P_ROOK || piece == P_QUEEN) p.rookQueens |= dst;
    if (C == WHITE) p.white = (p.white ^ src) | dst;
    else p.white &= ~dst;

    if (fl == MF_EP_CAPTURE) {
        const u64 cap = C == WHITE ? dst >> 8 : dst << 8;
        p.pawns &= ~cap;
        if (C == BLACK) p.white &= ~cap;
        if (HASH) zob_xor(*h, t, zob_piece(1 - C, P_PAWN, ctz(cap)));
    }
    if (fl == MF_KING_CASTLE || fl == MF_QUEEN_CASTLE) {
        const int sh = C == WHITE ? 0 : 56;
        const int rf = (fl == MF_KING_CASTLE ? 7 : 0) + sh, rt = (fl == MF_KING_CASTLE ? 5 : 3) + sh;
        p.rookQueens = (p.rookQueens ^ bit(rf)) | bit(rt);
        if (C == WHITE) p.white = (p.white ^ bit(rf)) | bit(rt);
        if (HASH) {
            zob_xor(*h, t, zob_piece(C, P_ROOK, rf));
            zob_xor(*h, t, zob_piece(C, P_ROOK, rt));
        }
    }

    // game state: side, en passant, castling
    u64 st = p.pawns & ~(0xFFULL | (1ULL << 63));
    int wc = pos_wcastle(p), bc = pos_bcastle(p);
    if (piece == P_KING) { if (C == WHITE) wc = 0; else bc = 0; }
    // a capture on the enemy's corner (updateCastleFlag, :1311)
    if (C == WHITE) {
        if (dst & bit(63)) bc &= ~1;
        else if (dst & bit(56)) bc &= ~2;
    } else {
        if (dst & bit(7)) wc &= ~1;
        else if (dst & bit(0)) wc &= ~2;
    }
    if (movedRook && piece == P_ROOK) {
        if (C == WHITE) {
            if (src & bit(7)) wc &= ~1;
            else if (src & bit(0)) wc &= ~2;
        } else {
            if (src & bit(63)) bc &= ~1;
            else if (src & bit(56)) bc &= ~2;
        }
    }
    int epf = 0;
    if (fl == MF_DOUBLE_PUSH) {
        const u64 ePawns = (C == WHITE) ? (p.pawns & RANKS2TO7 & ~p.white) : (p.pawns & RANKS2TO7 & p.white);
        if ((((dst << 1) & ~FILEA) | ((dst >> 1) & ~FILEH)) & ePawns) epf = (from & 7) + 1;
    }
    p.pawns = st | (u64)wc | ((u64)bc << 2) | ((u64)epf << 4) | ((u64)(1 - C) << 63);
    if (HASH) zob_state(*h, t, p);
}

template <int C, bool HASH>
PG_HD void make_move(Pos &p, u16 mv, Key128 *h, const Tables &t) {
    int piece = piece_on(p, bit(mv & 63));
    if (!piece) piece = P_PAWN;  // only for a move that is not legal here; keeps key indices in range
    make_move_as<C, HASH>(p, mv, piece, h, t);
}

// Full 128-bit key (MoveGeneratorBitboard.h:3914-3980); the side key is
// present when white is to move.
PG_HD Key128 zobrist128(const Pos &p, const Tables &t) {
    Key128 h = {0, 0};
    if (pos_side(p) == WHITE) zob_xor(h, t, ZOB_SIDE);
    zob_state(h, t, p);
    for (u64 all = pos_occ(p); all; all &= all - 1) {
        const int s = ctz(all);
        const int color = (p.white >> s) & 1 ? WHITE : BLACK;
        zob_xor(h, t, zob_piece(color, piece_on(p, bit(s)), s));
    }
    return h;
}

// The men nearest to square k either way on a line through it.
PG_HD u64 nearest(int k, u64 line, u64 occ) {
    const u64 below = bit(k) - 1, up = line & occ & ~below & ~bit(k), down = line & occ & below;
    return (up & (0 - up)) | (down & bit(63 - __builtin_clzll(down | 1)));
}
// Whether a board that pos_sane accepts is one that a game can be in, as far as
// the moves go: one man per square, castling rights only where king and rook
// stand at home, an en-passant field only behind an enemy pawn, and the side
// not to move not in check.  Legal moves lead from such a board to such boards.
// On others a king can be taken or a rook castle with no king, and the quiet
// and calm moves are not what they are taken for: leaf_plain counts those.
// (Straight through and without tables, for both sides: kd_begin asks it of
// every root, and a batch waits for that.)
PG_HD bool pos_regular(const Pos &p) {
    const u64 occ = pos_occ(p), pawns = pos_pawns(p), sliders = p.bishopQueens | p.rookQueens;
    const u64 twice = (pawns & (p.knights | sliders | p.kings)) | (p.knights & (sliders | p.kings)) | (sliders & p.kings);
    // men that a castling right needs, and that are not there
    const u64 rights = p.pawns & 15, wk = rights & 1, wq = rights >> 1 & 1, bk = rights >> 2 & 1, bq = rights >> 3;
    const u64 rooks = p.rookQueens & ~p.bishopQueens;
    const u64 away = ((wk | wq) << 4 & ~(p.kings & p.white)) | ((wk << 7 | wq) & ~(rooks & p.white)) |
                     ((bk | bq) << 60 & ~(p.kings & ~p.white)) | ((bk << 63 | bq << 56) & ~(rooks & ~p.white));
    const bool black = pos_side(p);
    const u64 mine = black ? occ & ~p.white : p.white, king = p.kings & ~mine;
    const int k = king_square(king);
    const u64 checks = ((p.knights & knight_att(king)) | (p.kings & king_att(king)) |
                        (pawns & (black ? pawn_att<WHITE>(king) : pawn_att<BLACK>(king))) |
                        (p.rookQueens & (nearest(k, file_of(k), occ) | nearest(k, rank_of(k), occ))) |
                        (p.bishopQueens & (nearest(k, diag_of(k), occ) | nearest(k, anti_of(k), occ)))) & mine;
    u64 ep = 0;
    if (const int f = pos_ep(p)) {
        const u64 dst = black ? bit(15 + f) : bit(39 + f), pawn = black ? dst << 8 : dst >> 8;
        ep = (occ & dst) | (pawn & ~(pawns & ~mine));
        // a pawn that did not come by a double push may stand between a bishop
        // and the king of the side that takes it
        const int q = king_square(p.kings & mine);
        const u64 seen = nearest(q, diag_of(q), occ & ~pawn) | nearest(q, anti_of(q), occ & ~pawn);
        ep |= p.bishopQueens & ~mine & seen & ~(nearest(q, diag_of(q), occ) | nearest(q, anti_of(q), occ));
    }
    return (twice | away | checks | ep) == 0;
}

// side dispatch helpers
template <int V>
PG_HD u32 count_any(const Pos &p, const Tables &t) {
    return pos_side(p) ? count_moves<BLACK, V>(p, t) : count_moves<WHITE, V>(p, t);
}
template <int V>
PG_HD u32 generate_any(const Pos &p, const Tables &t, u16 *out, u32 cap = 256) {
    return pos_side(p) ? generate_moves<BLACK, V>(p, t, out, cap) : generate_moves<WHITE, V>(p, t, out, cap);
}
// the same into window words (WordSink)
template <int V>
PG_HD u32 generate_words(const Pos &p, const Tables &t, u32 *out, u32 cap, u32 owner) {
    WordSink o{out, cap, 0, owner};
    if (pos_side(p)) {
        const Sides s = sides_of<BLACK>(p);
        generate_sides<BLACK, V>(s, gen_all<BLACK, V>(s, t), t, o);
    } else {
        const Sides s = sides_of<WHITE>(p);
        generate_sides<WHITE, V>(s, gen_all<WHITE, V>(s, t), t, o);
    }
    return o.n;
}
// the moves of k that are not quiet
template <int V>
PG_HD void generate_leaf(const Kin &k, const Gen &g, const Tables &t, LeafSink &o) {
    const Sides s = sides_of_kin(k);
    if (k.info >> KIN_SIDE & 1) generate_sides<BLACK, V>(s, g, t, o);
    else generate_sides<WHITE, V>(s, g, t, o);
}
template <int V>
PG_HD u32 count_child_any(const Kin &k, u32 w, const Tables &t) {
    return k.info >> KIN_SIDE & 1 ? count_child<WHITE, V>(k, w, t) : count_child<BLACK, V>(k, w, t);
}
// the same for any move, by making it
template <int V>
PG_HD u32 count_made(const Kin &k, u32 w, const Tables &t) {
    Pos p = pos_of_kin(k);
    const int piece = piece_code(w >> 24);
    if (pos_side(p)) {
        make_move_as<BLACK, false>(p, (u16)w, piece, nullptr, t);
        return count_moves<WHITE, V>(p, t);
    }
    make_move_as<WHITE, false>(p, (u16)w, piece, nullptr, t);
    return count_moves<BLACK, V>(p, t);
}
PG_HD u32 count_calm_any(const Kin &k, u32 w, const Tables &t) {
    return k.info >> KIN_SIDE & 1 ? count_calm<WHITE>(k, w, t) : count_calm<BLACK>(k, w, t);
}
PG_HD Kin kin_any(const Pos &p, const Tables &t) {
    return pos_side(p) ? kin_of<BLACK>(sides_of<BLACK>(p), t) : kin_of<WHITE>(sides_of<WHITE>(p), t);
}
PG_HD LeafEval leaf_any(Kin &k, const Tables &t) {
    return k.info >> KIN_SIDE & 1 ? leaf_eval<BLACK>(k, t) : leaf_eval<WHITE>(k, t);
}
PG_HD void make_any(Pos &p, u16 mv, const Tables &t) {
    if (pos_side(p)) make_move<BLACK, false>(p, mv, nullptr, t);
    else make_move<WHITE, false>(p, mv, nullptr, t);
}
PG_HD void make_any_hash(Pos &p, u16 mv, Key128 &h, const Tables &t) {
    if (pos_side(p)) make_move<BLACK, true>(p, mv, &h, t);
    else make_move<WHITE, true>(p, mv, &h, t);
}

}  // namespace pg
