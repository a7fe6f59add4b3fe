// leaf.h -- perft 2 of a position without making most of its children, for
// host and device.
//
// The leaf level of every perft run sums, over the legal moves of a position,
// the number of legal replies.  Making each child and counting its moves
// costs some 840 vector instructions a child, 27,000 for a position of 32
// moves; the sums below cost 4,900 for the position, 870 for each of the 4
// children still made, 240 for each of the 3 whose king's replies are counted
// and 700 to list both: 9,800 in all.  Both are bound by the vector ALUs.  The leaf level
// of 256 positions at perft 5 (8.16 million parents, 2.65e8 children): 4.79 ms
// move by move, 1.95 ms by sets.  Most moves change only a few
// of the replies, and by an amount that the position itself tells: so the
// replies are counted once, as if the opponent were to move in the position
// (`base`), and a quiet move or capture from f to t changes that number by
//     + P(f) - P(t)                          t empty
//     + P(f) - P(t) + cap_offset             t an opponent's piece
// where P is one number per square, the same for every move:
//   f (ours)    replies that an empty f would add: what the opponent's sliders
//               that stop at f see beyond it, pawn pushes onto or over f;
//               less the pawn captures on f;
//   t (empty)   replies lost if one of our pieces stood there: what sliders
//               crossing t see beyond it, pawn pushes onto or over it; less
//               the pawn captures it would offer;
//   t (theirs)  the captured piece's own replies, less the captures of our
//               piece on t by its defenders.
// P is kept bit-sliced, one 64-bit word per binary digit, so it is built for
// all squares at once with Kogge-Stone runs and adders, and the sum of P over
// a set of target squares is five popcounts.
//
// That is exact for a move that
//   - gives no check, moves no pinner or discoverer, does not enter or leave a
//     pin line of the opponent's king: pins and checks stay as they are;
//   - leaves every square around the opponent's king (and the squares its
//     castling crosses) attacked or not as it was;
//   - does not run along the line on which an opponent's slider sees f (pawn
//     pushes may: what they gain there is added apart), nor, but for pawns,
//     between the two squares in front of an opponent's pawn;
//   - is no castling, promotion or en passant, no capture next to the
//     opponent's king or of a pawn about to promote.
// Those moves are summed here, set by set: 78% of the moves of positions after
// 11 to 43 random plies, 92% after 4 to 12.  All others are handed out, piece
// by piece, to be made and counted one by one (12.5% and 5.5%) -- but a move
// that fails only the second condition (9% and 3%) changes nothing but the
// replies of the opponent's king: it is summed without them and handed out as
// a record of its own kind, for which only the king's moves and castling are
// counted (leaf_king_replies).
// A position in which the opponent is in check already, a side has not
// exactly one king, or two pieces share a square (a castle with a right whose
// rook is not at home may have put one on another piece) hands out every move.
#pragma once
#include "movegen.h"

namespace pf {

// Moves handed out: one record per moving piece (or set of pawn moves).
//   piece: from square s, targets `to`; pawn set: targets `to`, from = t - s.
// meta: s | kind << 6.
enum : u32 { kLeafPiece = 0, kLeafPawn = 1u << 6, kLeafDouble = 2u << 6, kLeafOO = 3u << 6, kLeafOOO = 4u << 6, kLeafEP = 5u << 6 };
constexpr u32 kLeafMetaBits = 9;
// The moves of a record one by one; k is 0 but for the second to fourth
// promotion of a pawn move.
struct LeafRecIter {
    u64 to;
    u32 meta, k;
    PF_HD bool done() const { return !to; }
    PF_HD u32 next() {
        const u32 d = (u32)ctz(to), s = meta & 63, kind = (meta >> 6) & 7;
        const bool pawn = kind - 1 < 2;
        const u32 from = pawn ? d - s : s;
        u32 fl = (0x532100u >> (4 * kind)) & 15;  // the move flag of each kind
        if (pawn && d >= 56) {
            fl = kFlPromoN + k;
            k = (k + 1) & 3;
        }
        if (!k) to &= to - 1;
        return mk_move((int)from, (int)d, (int)fl);
    }
};
PF_HD u32 leaf_rec_moves(u64 to, u32 meta) {
    const u32 n = (u32)popc(to);
    return ((meta >> 6) & 7) == 1 ? n + mul24((u32)popc(to & kRank8), 3) : n;
}

// P, bit-sliced in five digits.  On empty squares and on ours it is at most
// 28: a line holds at most two of the opponent's rays through a square, which
// see at most six squares beyond it, and pawns count at most four.  Captured
// pieces can reach more; their squares are noted in `over`.  Few of ours reach
// 16; their moves are handed out.
struct LeafPlanes {
    u64 p[5], over;
    // t0 + 2 t1 + 4 t2 + 8 t3 on the squares of m, and 1 for every square of c
    PF_HD void add(u64 t0, u64 t1, u64 t2, u64 m, u64 c) {
        fa(0, t0 & m, c);
        fa(1, t1 & m, c);
        fa(2, t2 & m, c);
        ha(3, c);
        ha(4, c);
        over |= c;
    }
    PF_HD void add4(u64 t0, u64 t1, u64 t2, u64 t3, u64 c) {
        fa(0, t0, c);
        fa(1, t1, c);
        fa(2, t2, c);
        fa(3, t3, c);
        ha(4, c);
        over |= c;
    }
    PF_HD void add2(u64 x, u64 y) {  // 1 for every square of x and 1 for every square of y
        fa(0, x, y);
#pragma unroll
        for (int i = 1; i < 5; i++) ha(i, y);
        over |= y;
    }
    PF_HD void fa(int i, u64 t, u64& c) {
        const u64 n = bitop3<0x96>(p[i], t, c);  // sum
        c = bitop3<0xE8>(p[i], t, c);            // carry
        p[i] = n;
    }
    PF_HD void ha(int i, u64& c) {
        const u64 n = p[i] ^ c;
        c &= p[i];
        p[i] = n;
    }
    PF_HD u32 sum(u64 s) const { return sum_from(s, popc_add(s & p[4], 0)); }  // of P over the squares of s
    PF_HD u32 sum_from(u64 s, u32 n = 0) const {  // the same where no square of s reaches 16
#pragma unroll
        for (int i = 3; i >= 0; i--) n = popc_add(s & p[i], n + n);
        return n;
    }
    PF_HD void stage_end() {
#pragma unroll
        for (int i = 0; i < 5; i++) pin(p[i]);
        pin(over);
    }
};

// Adds, on the squares of m, the number of squares of v that a slider there
// would see in direction D (its run through empty squares and the first
// piece, if that is in v), and 1 on the squares of c.
template <int D>
PF_HD void leaf_add_reach(LeafPlanes& pl, u64 v, u64 empty, u64 m, u64 c) {
    const u64 wrap = step_mask<-D>();
    const u64 c1 = step<-D>(v) & wrap, m1 = step<-D>(empty) & wrap;
    const u64 b = step<-D>(c1);  // one, two squares ahead
    const u64 l0 = xor_and(c1, b, m1), l1 = and3(c1, b, m1);
    const u64 x1 = m1 & step<-D>(m1);
    const u64 g0 = step<-2 * D>(l0), g1 = step<-2 * D>(l1) & x1;  // up to four
    const u64 s0 = xor_and(l0, g0, x1), k0 = and3(l0, g0, x1);
    const u64 s1 = bitop3<0x96>(l1, g1, k0), s2 = bitop3<0xE8>(l1, g1, k0);
    const u64 x3 = x1 & step<-2 * D>(x1);
    const u64 h0 = step<-4 * D>(s0), h1 = step<-4 * D>(s1) & x3, h2 = step<-4 * D>(s2) & x3;  // up to seven
    const u64 t0 = xor_and(s0, h0, x3), q0 = and3(s0, h0, x3);
    const u64 t1 = bitop3<0x96>(s1, h1, q0), q1 = bitop3<0xE8>(s1, h1, q0);
    pl.add(t0, t1, bitop3<0x96>(s2, h2, q1), m, c);
}

struct LeafYes { static constexpr bool value = true; };
struct LeafNo { static constexpr bool value = false; };

// The sides of a board.
struct LeafSides {
    u64 pawns, occ, us, them, K, eK;
    PF_HD explicit LeafSides(const Board& b) {
        pawns = b.pawns & kRanks2to7;
        occ = or3(or3(pawns, b.knights, b.bishops), b.rooks, b.kings);
        us = b.us;
        them = occ & ~us;
        K = b.kings & us;
        eK = b.kings & them;
    }
    PF_HD u64 uR(const Board& b) const { return b.rooks & us; }
    PF_HD u64 uB(const Board& b) const { return b.bishops & us; }
    PF_HD u64 tR(const Board& b) const { return b.rooks & them; }
    PF_HD u64 tB(const Board& b) const { return b.bishops & them; }
};

PF_HD u64 pawn_from(u64 z) { return ((z >> 7) & kNotA) | ((z >> 9) & kNotH); }  // our pawns there attack z
PF_HD u64 pawn_hits(u64 p) { return ((p << 7) & kNotH) | ((p << 9) & kNotA); }  // what our pawns attack

// First pass over one axis (directions D and -D): what decides pins and the
// squares each side's sliders attack.
struct LeafScan {
    u64 att;       // squares our sliders see
    u64 thr;       // squares the opponent's sliders see
    u64 pinned;    // the opponent's pinned pieces
    u64 from, to;  // squares that must not be left / entered: pins and what would become one
};
// Returns the squares seen from the opponent's king and past the first piece
// of its own: a slider of ours landing there checks or pins.
template <int D>
PF_HD u64 leaf_scan_axis(LeafScan& o, u64 empty, u64 us, u64 them, u64 mine, u64 theirs, u64 eK, u64 line) {
    const RayChain cp = ray_chain<D>(empty), cm = ray_chain<-D>(empty);
    const u64 up = ray_fill<D>(mine, cp), um = ray_fill<-D>(mine, cm);
    o.att = or3(o.att, up, um);
    o.thr = or3(o.thr, ray_fill<D>(theirs, cp), ray_fill<-D>(theirs, cm));
    const u64 kp = ray_fill<D>(eK, cp), km = ray_fill<-D>(eK, cm);
    // A piece of theirs on the king's line that a slider of ours sees from
    // the far side is pinned, or would be if our piece before it left: the
    // line's squares up to the first piece, and our sliders on it, stay put.
    const u64 above = line & (0 - (eK << 1)), below = line & (eK - 1);  // D > 0 moves up the board
    const u64 hp = and3(um, them, above), hm = and3(up, them, below);
    o.pinned = or_and(or_and(o.pinned, hp, kp), hm, km);
    const u64 fp = hp ? ~0ULL : 0ULL, fm = hm ? ~0ULL : 0ULL;
    o.from = or_and(or_and(o.from, or_and(kp, above, mine), fp), or_and(km, below, mine), fm);
    o.to = or_and(or_and(o.to, kp, fp), km, fm);
    // What stands between a slider of ours and such a square would uncover a
    // check or a pin; an empty square there lies on a pin line.
    const u64 rp = kp | ray_fill<D>(kp & them, cp), rm = km | ray_fill<-D>(km & them, cm);
    const u64 open = or_and(up & rm, um, rp);
    o.from = or_and(o.from, open, us);
    o.to = or_and(o.to, open, empty);
    return rp | rm;
}

// Second pass over one axis: the opponent's replies and P, and the paths to
// the squares that matter around its king.
struct LeafAxis {
    u64 line;            // squares the opponent's movers see along the axis
    u64 zatt;            // squares seen from the zone squares we attack
    u64 zray;            // squares seen from those we do not
    u64 keep;            // squares between our sliders and zone squares they attack
    u64 open;            // pieces between our sliders and the other zone squares
    u64 north;           // squares seen upwards (vertical axis)
};
template <int D>
PF_HD LeafAxis leaf_axis(LeafPlanes& pl, u32& base, u64 empty, u64 them, u64 gain, u64 mine, u64 theirs, u64 za, u64 zf) {
    const u64 v = ~them;  // and `gain`: the squares of v whose P takes what is seen beyond them
    const RayChain cp = ray_chain<D>(empty), cm = ray_chain<-D>(empty);
    const u64 tp = ray_fill<D>(theirs, cp), tm = ray_fill<-D>(theirs, cm);
    base = popc_add(tm & v, popc_add(tp & v, base));
    leaf_add_reach<D>(pl, v, empty, and_or(tp, gain, theirs), them & ~tp);
    leaf_add_reach<-D>(pl, v, empty, and_or(tm, gain, theirs), them & ~tm);
    const u64 up = ray_fill<D>(mine, cp), um = ray_fill<-D>(mine, cm);
    LeafAxis o;
    o.line = tp | tm;
    o.north = tp;
    {
        const u64 p = ray_fill<D>(za, cp), m = ray_fill<-D>(za, cm);
        o.zatt = p | m;
        o.keep = or_and(up & m, um, p);
    }
    {
        const u64 p = ray_fill<D>(zf, cp), m = ray_fill<-D>(zf, cm);
        o.zray = p | m;
        o.open = or_and(up & m, um, p);
    }
    return o;
}

// The opponent's king moves and castling after our move m, which gives no
// check, captures nothing next to that king and is no promotion, castling or
// en passant.
PF_HD u32 leaf_king_replies(const Board& b, u32 m) {
    const int from = m & 63, to = (m >> 6) & 63;
    const u64 src = bit(from), dst = bit(to), mv = src | dst;
    const u64 pawns = b.pawns & kRanks2to7;
    u64 occ = or3(or3(pawns, b.knights, b.bishops), b.rooks, b.kings);
    const u64 them = occ & ~b.us, eK = b.kings & them, empty = ~bitop3<0xBA>(occ, src, dst);  // (occ & ~src) | dst
    auto moved = [&](u64 x) { return xor_and(x & b.us, mv, 0 - ((x >> from) & 1)); };
    const u64 R = moved(b.rooks), B = moved(b.bishops);
    u64 att = knight_fill(moved(b.knights)) | king_fill(moved(b.kings)) | pawn_hits(moved(pawns));
    u64 a, h;
    {
        const RayChain s = ray_chain<-8>(empty), n = north_chain(s);
        att = or3(att, step<8>(ray_reach<8>(R, n)), step<-8>(ray_reach<-8>(R, s)));
    }
    a = step<1>(ray_reach<1>(R, ray_chain<1>(empty)));
    h = step<-1>(ray_reach<-1>(R, ray_chain<-1>(empty)));
    a = or3(a, step<9>(ray_reach<9>(B, ray_chain<9>(empty))), step<-7>(ray_reach<-7>(B, ray_chain<-7>(empty))));
    h = or3(h, step<-9>(ray_reach<-9>(B, ray_chain<-9>(empty))), step<7>(ray_reach<7>(B, ray_chain<7>(empty))));
    att = or_and(or_and(att, a, kNotA), h, kNotH);
    u32 n = popc_add(andn2(king_fill(eK), them, att), 0);
    const u32 hi = (u32)(att >> 32), oc = (u32)(occ >> 32), rights = (u32)b.pawns;
    constexpr u32 F8G8 = 0x60000000u, C8D8 = 0x0C000000u, B8D8 = 0x0E000000u;
    n += ((rights & 4) && !(oc & F8G8) && !(hi & F8G8)) ? 1 : 0;
    n += ((rights & 8) && !(oc & B8D8) && !(hi & C8D8)) ? 1 : 0;
    return n;
}

// The sum, over the legal moves of `b` dealt with set by set, of the
// opponent's replies; emit(king, full, meta) receives the others: records of
// which only the replies of the opponent's king are missing, and of which all
// are (either set may be empty).  On the GPU all lanes of a wave call it and
// emit together; a lane without a position passes an empty board.  `summed`
// (when not null) receives the number of moves not handed out in full.
template <class SL, class Emit>
PF_HD u32 leaf_sum(const Board& b, const SL& sl, Emit& emit, u32* summed = nullptr) {
    // stage 1: pins of the opponent, squares each side attacks
    u64 pinT, thr, hardFrom, hardTo, za, zf, kR, kB, cast = 0;
    u32 base, kings, generic;  // replies but the king's; the king's
    {
        const LeafSides p(b);
        const u64 eK = p.eK, occ = p.occ;
        const int ek = eK ? ctz(eK) : 0;
        LeafScan sc = {};
        kR = leaf_scan_axis<8>(sc, ~occ, p.us, p.them, p.uR(b), p.tR(b), eK, file_of(ek));
        kR |= leaf_scan_axis<1>(sc, ~occ, p.us, p.them, p.uR(b), p.tR(b), eK, rank_of(ek));
        kB = leaf_scan_axis<9>(sc, ~occ, p.us, p.them, p.uB(b), p.tB(b), eK, diag_of(ek));
        kB |= leaf_scan_axis<7>(sc, ~occ, p.us, p.them, p.uB(b), p.tB(b), eK, anti_of(ek));
        pinT = sc.pinned;
        thr = sc.thr;
        const u64 K = p.K;
        const u64 ours = or3(sc.att, knight_fill(b.knights & p.us), king_fill(K)) | pawn_hits(p.pawns & p.us);
        const u64 pk = p.pawns | b.kings, sliders = b.bishops | b.rooks;
        const u64 shared = or_and(or_and(p.pawns & b.kings, b.knights, sliders | pk), sliders, pk);
        generic = !eK || (eK & (eK - 1)) || !K || (K & (K - 1)) || (ours & eK) || shared;
        // the opponent's king: moves, castling, and the squares both depend on
        u64 zone = king_fill(eK) & ~p.them;
        kings = popc_add(zone & ~ours, 0);
        const u64 F8G8 = kF1G1 << 56, C8D8 = kC1D1 << 56, B8D8 = kB1D1 << 56;
        const int rights = st_rights(b);
        if (rights & 4) {
            cast |= F8G8 | bit(60) | bit(63);
            if (!(occ & F8G8)) { zone |= F8G8; kings += !(ours & F8G8); }
        }
        if (rights & 8) {
            cast |= B8D8 | bit(60) | bit(56);
            if (!(occ & B8D8)) { zone |= C8D8; kings += !(ours & C8D8); }
        }
        za = zone & ours;
        zf = zone & ~ours;
        hardFrom = sc.from | cast;
        hardTo = sc.to | cast;
        base = 0;
    }
    stage_end(pinT, thr, hardFrom, hardTo, za, zf, kR, kB, base, kings, generic);

    // stage 2: the opponent's sliders and P, axis by axis; what its king and
    // the squares around it see
    LeafPlanes pl = {};
    u64 line[4], north, zoneFrom, zoneTo, zR, zB;
#define PF_LEAF_AXIS(D, GAIN, LINE_OF, UX, TX)                                                        \
    const LeafSides p(b);                                                                             \
    const LeafAxis o = leaf_axis<D>(pl, base, ~p.occ, p.them, GAIN, p.UX(b),                          \
                                    either_and(~pinT, LINE_OF(p.eK ? ctz(p.eK) : 0), p.TX(b)), za, zf);
    {
        // pinned sliders keep to their line; our pawns' pushes, which run along
        // this axis, add what they gain on it themselves
        PF_LEAF_AXIS(8, andn2(~0ULL, p.them, p.pawns & p.us), file_of, uR, tR)
        line[0] = o.line; north = o.north; zR = o.zray; zoneTo = o.keep; zoneFrom = or_and(o.open, o.zatt, p.uR(b));
    }
    pl.stage_end();
    stage_end(base, line[0], north, zR, zoneFrom, zoneTo);
    {
        PF_LEAF_AXIS(1, ~p.them, rank_of, uR, tR)
        line[1] = o.line; zR |= o.zray; zoneTo |= o.keep; zoneFrom |= or_and(o.open, o.zatt, p.uR(b));
    }
    pl.stage_end();
    stage_end(base, line[1], zR, zoneFrom, zoneTo);
    {
        PF_LEAF_AXIS(9, ~p.them, diag_of, uB, tB)
        line[2] = o.line; zB = o.zray; zoneTo |= o.keep; zoneFrom |= or_and(o.open, o.zatt, p.uB(b));
    }
    pl.stage_end();
    stage_end(base, line[2], zB, zoneFrom, zoneTo);
    {
        PF_LEAF_AXIS(7, ~p.them, anti_of, uB, tB)
        line[3] = o.line; zB |= o.zray; zoneTo |= o.keep; zoneFrom |= or_and(o.open, o.zatt, p.uB(b));
    }
#undef PF_LEAF_AXIS
    pl.stage_end();
    stage_end(base, line[3], zB, zoneFrom, zoneTo);

    // stage 3: the opponent's knights and pawns
    u32 beside;   // double pushes on our fourth rank: files with a pawn of theirs to the left, to the right,
                  // and those whose en passant capture is not settled here (one byte each)
    u32 cap = 8;  // its rays, and below its knights, that do not reach a captured piece count 1 in P
    u64 cSE, cSW, before7;
    {
        const LeafSides p(b);
        const u64 us = p.us, them = p.them, empty = ~p.occ, eK = p.eK, freeT = ~pinT;
        const int ek = eK ? ctz(eK) : 0;
        for (u64 n = b.knights & them & freeT; n; n &= n - 1) {  // pinned ones never move
            const u64 sb = n & (0 - n), f = knight_fill(sb);
            const u32 c = popc_add(f & ~them, 0);
            base += c;
            cap++;
            pl.add4((c & 1) ? sb : 0, (c & 2) ? sb : 0, (c & 4) ? sb : 0, (c & 8) ? sb : 0, them & ~f);
        }
        // pawns: pushes (onto empties; ours in their way), captures
        const u64 tP = p.pawns & them, pp = tP & freeT, pm = tP & pinT;
        const u64 push = or_and(pp, pm, file_of(ek));
        cSE = or_and(pp, pm, anti_of(ek));
        cSW = or_and(pp, pm, diag_of(ek));
        const u64 f1 = push >> 8, p1 = f1 & empty, d1 = (p1 & kRank6) >> 8, p2 = d1 & empty;
        const u64 aSE = (cSE >> 7) & kNotA, aSW = (cSW >> 9) & kNotH, hSE = aSE & us, hSW = aSW & us;
        base = popc_add(hSE, popc_add(hSW, popc_add(p1 | p2, base)));  // the two kinds of push never share a target
        base += mul24(popc_add32((u32)(p1 & kRank1), popc_add32((u32)(hSE & kRank1), popc_add32((u32)(hSW & kRank1), 0))), 3);
        pl.add2(or3(p1 | p2, f1 & us, p1 << 8), or3(p2 << 8, d1 & us, p2 << 16) | and3(f1 & kRank6, us, empty << 8));
        pl.add2(~aSE, ~aSW);
        pl.add2(hSE << 7, hSW << 9);
        before7 = ((push & kRank7) >> 8) | ((push & kRank7) >> 16);  // the squares a double push crosses
        {
            const u32 r4 = (u32)(pp >> 24) & 0xFF, n4 = (u32)(pm >> 24) & 0xFF;
            const u32 lft = (r4 << 1) & 0xFF, rgt = r4 >> 1;
            u32 no = (n4 << 1) | (n4 >> 1);
            if ((eK >> 24 & 0xFF) && ((b.rooks & us) >> 24 & 0xFF)) no |= lft | rgt;  // may uncover the king
            beside = lft | (rgt << 8) | ((no & 0xFF) << 16);
        }
        const u64 edge = kRank1 & or3(f1, aSE, aSW);  // replies that promote
        zoneFrom = or3(zoneFrom, b.knights & knight_fill(za), p.pawns & pawn_from(za)) | (p.K & king_fill(za));
        hardFrom = or3(hardFrom, edge, pl.p[4]);
        if (generic) hardFrom = ~0ULL;
        hardTo = or3(hardTo, edge, pl.over) | (them & (king_fill(eK) | (tP & 0xFF00ULL)));
    }
    pl.stage_end();
    stage_end(base, cap, beside, cSE, cSW, before7, zoneFrom, hardFrom, hardTo);

    // stage 4: our moves
    PosInfo pi;
    u64 beyond = 0;
    pins_checks(b, pi, &beyond);
    const u64 occ = pi.occ, us = pi.us, them = pi.them, empty = ~occ, K = pi.K, eK = b.kings & them;
    const u64 uN = b.knights & us, uP = pi.pawns & us, tP = pi.pawns & them;
    const u64 att = or3(leaper_threats(b, pi), thr, beyond);  // where our king may not go
    const int rights = st_rights(b), ksq = pi.ksq;
    const u64 own = us & ~hardFrom;
    u32 total = 0, nOk = 0, nS = 0, nCap = 0;  // moves summed here; of those with `kings`, of captures
    // The moves of `t` (meta as in a record) of which those in `ok` need only
    // conditions on the opponent's king, and those in `s` none; the P of the
    // from squares of `ok` sum to fsum.
    auto take = [&](u64 t, u64 ok, u64 s, u32 fsum, u32 meta) {
        nOk = popc_add(ok, nOk);
        nS = popc_add(s, nS);
        nCap = popc_add(ok & them, nCap);
        total += fsum - pl.sum(ok);
        emit(ok & ~s, t & ~ok, meta);
    };
    const bool check = pi.checkers != 0, dbl = (pi.checkers & (pi.checkers - 1)) != 0;
    {
        const u64 t = andn2(king_fill(K), us, att);
        // a pawn ahead would push or capture onto the king's square
        u64 ok = (K & own) ? t & ~hardTo : 0;
        ok &= ~(((K << 8) & tP) | (((K << 9) & kNotA) & cSW) | (((K << 7) & kNotH) & cSE));
        if (K & before7) ok &= ~(before7 & ((K << 8) | (K >> 8)));
        if (K & (or3(line[0], line[1], line[2]) | line[3])) ok = 0;
        const u64 s = (K & zoneFrom) ? 0 : ok & ~zoneTo & ~king_fill(zf);
        take(t, ok, s, mul24(popc_add(ok, 0), pl.sum_from(K)), (u32)ksq);
    }
    const u64 tgt = dbl ? 0 : check ? (pi.checkers | pi.block) : ~us;
    const u64 free = ~pi.pinned;
    {
        const u64 hard = hardTo | knight_fill(eK), zone = zoneTo | knight_fill(zf);
        for (u64 n = dbl ? 0 : uN & free; any_lane(n); n &= n - 1) {
            const u64 sb = n & (0 - n), t = knight_fill(sb) & tgt;
            const int sq = ctz(n);
            const u64 ok = (sb & own) ? t & ~hard : 0, s = (sb & zoneFrom) ? 0 : ok & ~zone;
            take(t, ok, s, mul24(popc_add(ok, 0), pl.sum_from(sb)), (u32)sq);
        }
    }
    // sliders, by kind; none of a line is `ok` if an opponent's slider sees the
    // piece along it
    auto sliders = [&](u64 n, auto orth, auto diag) {
        const u64 hard = hardTo | (orth.value ? kR : 0) | (diag.value ? kB : 0);
        const u64 zone = zoneTo | (orth.value ? zR : 0) | (diag.value ? zB : 0);
        for (; any_lane(n); n &= n - 1) {
            const u64 sb = n & (0 - n);
            const int sq = n ? ctz(n) : 0;
            u64 t = 0, bad = hard;
            if (diag.value) {
                t |= sl.bishop(sq, occ);
                bad |= (sb & line[2]) ? diag_of(sq) : 0;
                bad |= (sb & line[3]) ? anti_of(sq) : 0;
            }
            if (orth.value) {
                t |= sl.rook(sq, occ);
                bad |= (sb & line[0]) ? file_of(sq) : 0;
                bad |= (sb & line[1]) ? rank_of(sq) : 0;
                bad |= ((sb & before7) ? before7 & ((sb << 8) | (sb >> 8)) : 0) | (((sb << 8) | (sb << 16)) & tP);
            }
            t &= n ? tgt : 0;
            if (pi.pinned & sb) {
                const u64 kf = file_of(ksq), kr = rank_of(ksq), kd = diag_of(ksq);
                t &= (kf & sb) ? kf : (kr & sb) ? kr : (kd & sb) ? kd : anti_of(ksq);
            }
            const u64 ok = (sb & own) ? t & ~bad : 0, s = (sb & zoneFrom) ? 0 : ok & ~zone;
            u32 f = mul24(popc_add(ok, 0), pl.sum_from(sb));
            if (diag.value)  // a captured pawn's capture of ours is not lost twice
                f = popc_add(ok & ((((sb << 9) & kNotA) & cSW) | (((sb << 7) & kNotH) & cSE)), f);
            take(t, ok, s, f, (u32)sq);
        }
    };
    {
        const u64 may = dbl ? 0 : check ? us & free : us, uR = b.rooks & may, uB = b.bishops & may;
        sliders(uB & ~uR, LeafNo{}, LeafYes{});
        sliders(uR & ~uB, LeafYes{}, LeafNo{});
        sliders(uR & uB, LeafYes{}, LeafYes{});
    }
    {
        const u64 Pf = uP & free, pin = check ? 0 : uP & pi.pinned;
        const u64 hard = hardTo | pawn_from(eK) | kRank8, zone = zoneTo | pawn_from(zf);
        const u64 calm = own & ~zoneFrom;
        const u64 q1 = (or_and(Pf, pin, file_of(ksq)) << 8) & empty;
        {
            // a rook behind the pawn gains one square; a pawn of theirs two ranks
            // ahead loses its push and gains no double one
            const u64 t = q1 & tgt, ok = t & (own << 8) & ~hard;
            const u32 f = popc_add(ok & (north << 8), pl.sum_from(ok >> 8)) - popc_add(and3(ok, before7, before7 << 8), 0);
            take(t, ok, ok & (calm << 8) & ~zone, f, 8u | kLeafPawn);
        }
        {
            const u64 t = (((check ? (q1 & ~tgt) : q1) & kRank3) << 8) & empty & tgt;
            const u64 ok = t & (own << 16) & ~(hard | ((u64)(beside >> 16) << 24));
            const u32 o4 = (u32)(ok >> 24), ep = popc_add32(o4 & beside, popc_add32(o4 & (beside >> 8), 0));
            const u32 f = 2 * popc_add(ok & (north << 16), 0) + ep + pl.sum_from(ok >> 16);
            take(t, ok, ok & (calm << 16) & ~zone, f, 16u | kLeafDouble);
        }
        // a captured pawn's capture of ours is not lost twice
        {
            const u64 t = ((or_and(Pf, pin, diag_of(ksq)) << 9) & kNotA) & them & tgt;
            const u64 ok = t & ((own & ~(line[2] | line[0])) << 9) & ~hard;
            take(t, ok, ok & (calm << 9) & ~zone, popc_add(ok & cSW, pl.sum_from(ok >> 9)), 9u | kLeafPawn);
        }
        {
            const u64 t = ((or_and(Pf, pin, anti_of(ksq)) << 7) & kNotH) & them & tgt;
            const u64 ok = t & ((own & ~(line[3] | line[0])) << 7) & ~hard;
            take(t, ok, ok & (calm << 7) & ~zone, popc_add(ok & cSE, pl.sum_from(ok >> 7)), 7u | kLeafPawn);
        }
    }
    {
        const bool oo = !check && (rights & 1) && !(occ & kF1G1) && !(att & kF1G1);
        const bool ooo = !check && (rights & 2) && !(occ & kB1D1) && !(att & kC1D1);
        if (any_lane(oo || ooo)) {
            emit(0, oo ? bit(6) : 0, 4u | kLeafOO);
            emit(0, ooo ? bit(2) : 0, 4u | kLeafOOO);
        }
    }
    const int ep = dbl ? 0 : st_ep(b);
    if (any_lane((u64)ep)) {
        const u64 T = ep ? bit(40 + ep - 1) : 0, C = T >> 8;
        const u64 src = (((C << 1) & kNotA) | ((C >> 1) & kNotH)) & uP;
        for (int side = 0; side < 2; side++) {  // the capturing pawn left, then right of the captured one
            const u64 s = src & (side ? (C << 1) & kNotA : (C >> 1) & kNotH);
            bool ok = s != 0;
            if (check) {
                ok = ok && (C == pi.checkers) && !(s & pi.pinned);
            } else if (s & pi.pinned) {
                const u64 kf = file_of(ksq), kd = diag_of(ksq), ka = anti_of(ksq);
                ok = (T & ((kd & s) ? kd : (ka & s) ? ka : (kf & s) ? kf : rank_of(ksq))) != 0;
            } else if (s) {
                const u64 pro = empty | C | s;
                ok = !((att_e(b.rooks & them, pro) | att_w(b.rooks & them, pro)) & K & kRank5);
            }
            emit(0, ok ? T : 0, (u32)(s ? ctz(s) : 0) | kLeafEP);
        }
    }
    if (summed) *summed = nOk;
    return total + nOk * base + nS * kings + nCap * cap;
}

}  // namespace pf
