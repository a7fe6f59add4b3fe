// board.h -- position layouts and 64-bit bit primitives shared by host and
// device code (compiled by hipcc for both).
//
// Two layouts:
//  * pf_pos48 (include/perft_gpu_amd.h): the reference HexaBitBoardPosition
//    layout (chess.h:208-230), used only at the C-ABI boundary.
//  * Board: the engine's "side-to-move-is-us" layout.  The position is
//    mirrored vertically whenever black is to move, so every frontier node is
//    generated by the same white-to-move code: no colour templates, no
//    divergence between waves holding positions of different colours.
//    Perft counts are invariant under this colour flip.
#pragma once
#include <stdint.h>

#include <hip/hip_runtime.h>

#define PF_HD __host__ __device__ __forceinline__

namespace pf {

typedef uint64_t u64;
typedef uint32_t u32;
typedef uint16_t u16;
typedef uint8_t u8;

constexpr u64 kRanks2to7 = 0x00FFFFFFFFFFFF00ULL;
constexpr u64 kRank1 = 0x00000000000000FFULL;
constexpr u64 kRank3 = 0x0000000000FF0000ULL;
constexpr u64 kRank5 = 0x000000FF00000000ULL;
constexpr u64 kRank6 = 0x0000FF0000000000ULL;
constexpr u64 kRank7 = 0x00FF000000000000ULL;
constexpr u64 kRank8 = 0xFF00000000000000ULL;
constexpr u64 kFileA = 0x0101010101010101ULL;
constexpr u64 kFileH = 0x8080808080808080ULL;
constexpr u64 kNotA = ~kFileA;
constexpr u64 kNotH = ~kFileH;
constexpr u64 kF1G1 = 0x60ULL;
constexpr u64 kC1D1 = 0x0CULL;
constexpr u64 kB1D1 = 0x0EULL;

// Board: six bitboards, 48 bytes, same field order as the reference layout.
//   us      pieces of the side to move
//   pawns   pawns on ranks 2-7; byte 0 = state, byte 7 = legal-move count
//   knights, bishops (B|Q), rooks (R|Q), kings  -- both colours
// State byte (pawns bits 0-7): bit0 our O-O, bit1 our O-O-O, bit2 their O-O,
// bit3 their O-O-O, bits4-7 en-passant file+1 (target square on rank 6).
// Count byte (pawns bits 56-63): number of legal moves of this node, filled
// in by whoever created the node (0..218 fits).
struct alignas(16) Board {
    u64 us, pawns, knights, bishops, rooks, kings;
};
static_assert(sizeof(Board) == 48, "Board must be 48 bytes");

PF_HD int popc(u64 x) { return __builtin_popcountll(x); }
// n + popcount(x): on the GPU two accumulating v_bcnt_u32_b32.  The empty asm
// statements keep the compiler from regrouping a run of these sums into
// separate popcounts joined by three-input adds, which issue at the
// popcount's own (single) rate on gfx950.
PF_HD u32 popc_add(u64 x, u32 n) {
#if defined(__HIP_DEVICE_COMPILE__)
    n = (u32)__builtin_popcount((u32)x) + n;
    asm("" : "+v"(n));
    n = (u32)__builtin_popcount((u32)(x >> 32)) + n;
    asm("" : "+v"(n));
    return n;
#else
    return n + (u32)__builtin_popcountll(x);
#endif
}
PF_HD u32 popc_add32(u32 x, u32 n) {
    n = (u32)__builtin_popcount(x) + n;
#if defined(__HIP_DEVICE_COMPILE__)
    asm("" : "+v"(n));
#endif
    return n;
}
// Product of two numbers below 2^24: one full-rate instruction.
PF_HD u32 mul24(u32 a, u32 b) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __umul24(a, b);
#else
    return a * b;
#endif
}
// (of 0, which only a side without a king asks for: 31, as the GPU's minimum of
// the halves' find-first-bit results comes out)
PF_HD int ctz(u64 x) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_ctzll(x);
#else
    return x ? __builtin_ctzll(x) : 31;
#endif
}
PF_HD u64 bit(int s) { return 1ULL << s; }
PF_HD u64 flip(u64 x) { return __builtin_bswap64(x); }  // vertical mirror

PF_HD int st_rights(const Board& b) { return (int)(b.pawns & 15); }
PF_HD int st_ep(const Board& b) { return (int)((b.pawns >> 4) & 15); }
PF_HD int meta_count(const Board& b) { return (int)(b.pawns >> 56); }
PF_HD u64 occupancy(const Board& b) {
    return (b.pawns & kRanks2to7) | b.knights | b.bishops | b.rooks | b.kings;
}

// Three-input logic on 64-bit words.  On gfx950 each 32-bit half is one
// v_bitop3_b32, which issues at the rate of a plain and/or; the compiler
// otherwise emits two two-input operations (or the half-rate and_or / or3).
// IMM is the function's truth table: bit (a << 2 | b << 1 | c) of IMM is the
// result for input bits a, b, c, i.e. the function applied to 0xF0, 0xCC and
// 0xAA.  The host form evaluates the same table, so host-built tests check
// every immediate.
template <u32 IMM>
PF_HD u64 bitop3(u64 a, u64 b, u64 c) {
#if defined(__HIP_DEVICE_COMPILE__)
    const u32 lo = __builtin_amdgcn_bitop3_b32((u32)a, (u32)b, (u32)c, IMM);
    const u32 hi = __builtin_amdgcn_bitop3_b32((u32)(a >> 32), (u32)(b >> 32), (u32)(c >> 32), IMM);
    return ((u64)hi << 32) | lo;
#else
    u64 r = 0;
    for (int k = 0; k < 8; k++)
        if ((IMM >> k) & 1) r |= ((k & 4) ? a : ~a) & ((k & 2) ? b : ~b) & ((k & 1) ? c : ~c);
    return r;
#endif
}
template <u32 IMM>
PF_HD u32 bitop3_32(u32 a, u32 b, u32 c) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_bitop3_b32(a, b, c, IMM);
#else
    return (u32)bitop3<IMM>(a, b, c);
#endif
}
PF_HD u64 or_and(u64 a, u64 b, u64 c) { return bitop3<0xF8>(a, b, c); }   // a | (b & c)
PF_HD u64 or3(u64 a, u64 b, u64 c) { return bitop3<0xFE>(a, b, c); }      // a | b | c
PF_HD u64 and3(u64 a, u64 b, u64 c) { return bitop3<0x80>(a, b, c); }     // a & b & c
PF_HD u64 and_or(u64 a, u64 b, u64 c) { return bitop3<0xEA>(a, b, c); }   // (a & b) | c
PF_HD u64 either_and(u64 a, u64 b, u64 c) { return bitop3<0xA8>(a, b, c); }  // (a | b) & c
PF_HD u64 and_andn(u64 a, u64 b, u64 c) { return bitop3<0x40>(a, b, c); }  // a & b & ~c
PF_HD u64 andn2(u64 a, u64 b, u64 c) { return bitop3<0x10>(a, b, c); }     // a & ~b & ~c
PF_HD u64 xor_and(u64 a, u64 b, u64 c) { return bitop3<0x78>(a, b, c); }   // a ^ (b & c)
PF_HD u64 xor_or(u64 a, u64 b, u64 c) { return bitop3<0xBE>(a, b, c); }    // (a ^ b) | c

// 64-bit shifts by a constant that stay one v_lshlrev_b64 / v_lshrrev_b64
// on the GPU (register-only inline asm; a shift whose halves feed 32-bit
// logic is otherwise split into a 32-bit shift plus an alignbit, two issue
// slots instead of one).  A shift by 32 is a register move either way.
template <int S>
PF_HD u64 shl(u64 x) {
#if defined(__HIP_DEVICE_COMPILE__)
    if constexpr (S != 32) {
        u64 r;
        asm("v_lshlrev_b64 %0, %1, %2" : "=v"(r) : "i"(S), "v"(x));
        return r;
    }
#endif
    return x << S;
}
template <int S>
PF_HD u64 shr(u64 x) {
#if defined(__HIP_DEVICE_COMPILE__)
    if constexpr (S != 32) {
        u64 r;
        asm("v_lshrrev_b64 %0, %1, %2" : "=v"(r) : "i"(S), "v"(x));
        return r;
    }
#endif
    return x >> S;
}

// Ends a stage of a long computation on the GPU: the values named are
// computed before it, others are computed (or read from memory) again after
// it rather than kept in registers.
PF_HD void pin(u64& x) {
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+v"(x));
#endif
}
PF_HD void pin(u32& x) {
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+v"(x));
#endif
}
// Whether x is not 0 in any lane of the wave (on the host: of this call).
PF_HD bool any_lane(u64 x) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __ballot(x != 0) != 0;
#else
    return x != 0;
#endif
}
template <class... T>
PF_HD void stage_end(T&... x) {
    (pin(x), ...);
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
#endif
}

// Kogge-Stone occluded fills: `g` generators, `p` propagator (empty squares).
// Each returns the attack set in one direction, including the first blocker.
PF_HD u64 att_n(u64 g, u64 p) {
    g = or_and(g, shl<8>(g), p); p &= shl<8>(p); g = or_and(g, shl<16>(g), p); p &= shl<16>(p);
    g = or_and(g, shl<32>(g), p);
    return shl<8>(g);
}
PF_HD u64 att_s(u64 g, u64 p) {
    g = or_and(g, shr<8>(g), p); p &= shr<8>(p); g = or_and(g, shr<16>(g), p); p &= shr<16>(p);
    g = or_and(g, shr<32>(g), p);
    return shr<8>(g);
}
PF_HD u64 att_e(u64 g, u64 p) {
    p &= kNotA;
    g = or_and(g, shl<1>(g), p); p &= shl<1>(p); g = or_and(g, shl<2>(g), p); p &= shl<2>(p);
    g = or_and(g, shl<4>(g), p);
    return shl<1>(g) & kNotA;
}
PF_HD u64 att_w(u64 g, u64 p) {
    p &= kNotH;
    g = or_and(g, shr<1>(g), p); p &= shr<1>(p); g = or_and(g, shr<2>(g), p); p &= shr<2>(p);
    g = or_and(g, shr<4>(g), p);
    return shr<1>(g) & kNotH;
}
PF_HD u64 att_ne(u64 g, u64 p) {
    p &= kNotA;
    g = or_and(g, shl<9>(g), p); p &= shl<9>(p); g = or_and(g, shl<18>(g), p); p &= shl<18>(p);
    g = or_and(g, shl<36>(g), p);
    return shl<9>(g) & kNotA;
}
PF_HD u64 att_nw(u64 g, u64 p) {
    p &= kNotH;
    g = or_and(g, shl<7>(g), p); p &= shl<7>(p); g = or_and(g, shl<14>(g), p); p &= shl<14>(p);
    g = or_and(g, shl<28>(g), p);
    return shl<7>(g) & kNotH;
}
PF_HD u64 att_se(u64 g, u64 p) {
    p &= kNotA;
    g = or_and(g, shr<7>(g), p); p &= shr<7>(p); g = or_and(g, shr<14>(g), p); p &= shr<14>(p);
    g = or_and(g, shr<28>(g), p);
    return shr<7>(g) & kNotA;
}
PF_HD u64 att_sw(u64 g, u64 p) {
    p &= kNotH;
    g = or_and(g, shr<9>(g), p); p &= shr<9>(p); g = or_and(g, shr<18>(g), p); p &= shr<18>(p);
    g = or_and(g, shr<36>(g), p);
    return shr<9>(g) & kNotH;
}
// The same fills split in two, for several generator sets over one
// occupancy: a direction's propagator chain (the empty squares a step may
// land on, then those that two and four steps may cross) is built once and
// shared.  D is the square delta of one step: 8 N, -8 S, 1 E, -1 W, 9 NE,
// 7 NW, -7 SE, -9 SW.
template <int D>
PF_HD u64 step(u64 x) {
    if constexpr (D > 0) return shl<D>(x);
    else return shr<-D>(x);
}
template <int D>
constexpr u64 step_mask() {  // squares a step in direction D can land on
    return (D == 1 || D == 9 || D == -7) ? kNotA : (D == -1 || D == 7 || D == -9) ? kNotH : ~0ULL;
}
struct RayChain {
    u64 p0, p1, p2;
};
template <int D>
PF_HD RayChain ray_chain(u64 empty) {
    RayChain c;
    c.p0 = empty & step_mask<D>();
    c.p1 = c.p0 & step<D>(c.p0);
    c.p2 = c.p1 & step<2 * D>(c.p1);
    return c;
}
// The north chain is the south chain moved up: a square and the 1 (3)
// squares below it are empty exactly when the square 1 (3) ranks down and
// the squares above it are.
PF_HD RayChain north_chain(const RayChain& south) {
    return RayChain{south.p0, shl<8>(south.p1), shl<24>(south.p2)};
}
// Generators plus every square they reach in direction D through empty
// squares, before the final step: ray_fill = step<D>(ray_reach) & step_mask.
template <int D>
PF_HD u64 ray_reach(u64 g, const RayChain& c) {
    g = or_and(g, step<D>(g), c.p0);
    g = or_and(g, step<2 * D>(g), c.p1);
    return or_and(g, step<4 * D>(g), c.p2);
}
template <int D>
PF_HD u64 ray_fill(u64 g, const RayChain& c) {  // == att_<D>(g, empty)
    return step<D>(ray_reach<D>(g, c)) & step_mask<D>();
}

PF_HD u64 rook_fill(u64 r, u64 empty) {
    return att_n(r, empty) | att_s(r, empty) | att_e(r, empty) | att_w(r, empty);
}
PF_HD u64 bishop_fill(u64 b, u64 empty) {
    return att_ne(b, empty) | att_nw(b, empty) | att_se(b, empty) | att_sw(b, empty);
}
PF_HD u64 knight_fill(u64 n) {
    u64 l1 = (n >> 1) & 0x7f7f7f7f7f7f7f7fULL, l2 = (n >> 2) & 0x3f3f3f3f3f3f3f3fULL;
    u64 r1 = (n << 1) & 0xfefefefefefefefeULL, r2 = (n << 2) & 0xfcfcfcfcfcfcfcfcULL;
    u64 h1 = l1 | r1, h2 = l2 | r2;
    return or3(h1 << 16, h1 >> 16, h2 << 8) | (h2 >> 8);
}
PF_HD u64 king_fill(u64 k) {
    u64 a = ((k << 1) & kNotA) | ((k >> 1) & kNotH);
    k |= a;
    return or3(a, k << 8, k >> 8);
}

// Lines through a square (used to restrict pinned pieces to their pin axis).
PF_HD u64 file_of(int s) { return kFileA << (s & 7); }
PF_HD u64 rank_of(int s) { return kRank1 << (s & 56); }
// The diagonals through s: the long diagonal moved up (d8 > 0) or down by
// d8 = 8 x its rank offset, written as two shifts of which one is by zero, so
// that the result has no branch and repeated uses of it are one computation.
PF_HD u64 shift_rows(u64 m, int d8) {
    const int up = d8 & ~(d8 >> 31);  // max(d8, 0)
    return (m << up) >> (up - d8);
}
PF_HD u64 diag_of(int s) {  // a1-h8 direction
    return shift_rows(0x8040201008040201ULL, (s & 56) - ((s & 7) << 3));
}
PF_HD u64 anti_of(int s) {  // a8-h1 direction
    return shift_rows(0x0102040810204080ULL, (s & 56) + ((s & 7) << 3) - 56);
}

// Attacks along one line mask `m` (through s) of a slider on s: both rays by
// obstruction difference, (o - 2s) ^ o for the squares above s and the same
// on the bit-reversed board for those below.  `rocc` = reverse(occ).
PF_HD u64 reverse(u64 x) { return __builtin_bitreverse64(x); }
PF_HD u64 line_attack(u64 m, u64 occ, u64 rocc, u64 sb, u64 rsb) {
    const u64 up = (occ & m) - (sb << 1), dn = (rocc & reverse(m)) - (rsb << 1);
    return bitop3<0x28>(up, reverse(dn), m);  // (up ^ down) & m
}

}  // namespace pf
