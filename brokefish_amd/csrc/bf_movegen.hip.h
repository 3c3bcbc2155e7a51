// Move generation by rows of sixteen lanes, for the kernel of its own (bf_movegen.hip) and the one that expands what it generates
// (bf_expand.hip): see bf_movegen.hip.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace bf {
namespace moves {

typedef unsigned long long u64;

constexpr unsigned CAPTURED = 0x800u, COLOR = 0x400u, SPECIAL = 0x200u;
enum { PAWN, KNIGHT, BISHOP, ROOK, QUEEN, KING };

struct Enemy {          // the side NOT to move, after the move under test
    u64 pawns, knights, diag, orth, king;
    int behind;         // from a square to the rank its pawns attack it from: +8 for black ones, -8 for white ones
};

__device__ __forceinline__ u64 bit(int sq) { return 1ull << sq; }

constexpr u64 FILE_A = 0x0101010101010101ull, FILE_H = 0x8080808080808080ull;
constexpr u64 NOT_A = ~FILE_A, NOT_H = ~FILE_H, NOT_AB = ~(FILE_A | FILE_A << 1), NOT_GH = ~(FILE_H | FILE_H >> 1);

// Any function of three words in one instruction per half: the truth table over A, B, C.  It issues at the rate of a single
// AND or XOR, which the compiler's three-operand forms (or3, and_or, bfi) do not: 2.5 clocks against 4.2, a pair of two-operand
// ones 4.1.
constexpr unsigned A = 0xF0, B = 0xCC, C = 0xAA;
template <unsigned TABLE>
__device__ __forceinline__ u64 logic(u64 a, u64 b, u64 c) {
    const unsigned lo = __builtin_amdgcn_bitop3_b32((unsigned)a, (unsigned)b, (unsigned)c, TABLE);
    const unsigned hi = __builtin_amdgcn_bitop3_b32((unsigned)(a >> 32), (unsigned)(b >> 32), (unsigned)(c >> 32), TABLE);
    return ((u64)hi << 32) | lo;
}

// The squares a slider on s (one bit) reaches along the line `m` (a rank, file or diagonal through
// s, s excluded) on occupancy occ, blockers included: o - s borrows upwards through the empty
// squares to the first blocker, so o ^ (o - s) is the ray towards the higher bits; the same on the
// bit-reversed board is the ray towards the lower ones.  No loop, no branch.  `less` and `less_rev` are -s and minus the
// reversed s: a 64-bit sum is one instruction, a difference two of the same cost.
__device__ __forceinline__ u64 line_attacks(u64 occ, u64 m, u64 less, u64 less_rev) {
    const u64 o = occ & m;
    const u64 up = o + less;
    const u64 down = __brevll(__brevll(o) + less_rev);
    return logic<(A ^ B) & C>(up, down, m);
}
__device__ __forceinline__ u64 knight_pattern(u64 s) {
    const u64 near = ((s >> 1) & NOT_H) | ((s << 1) & NOT_A), far = ((s >> 2) & NOT_GH) | ((s << 2) & NOT_AB);
    return near << 16 | near >> 16 | far << 8 | far >> 8;
}
__device__ __forceinline__ u64 king_pattern(u64 s) {
    const u64 row = s | ((s << 1) & NOT_A) | ((s >> 1) & NOT_H);
    return (row | row << 8 | row >> 8) ^ s;
}
__device__ __forceinline__ u64 diagonal(int sq) {   // a1-h8 direction: 0x8040201008040201 shifted by whole ranks
    const int d = (sq >> 3) - (sq & 7);
    return (d >= 0 ? 0x8040201008040201ull << (8 * d) : 0x8040201008040201ull >> (8 * -d)) ^ bit(sq);
}
__device__ __forceinline__ u64 antidiagonal(int sq) {   // a8-h1 direction
    const int e = (sq >> 3) + (sq & 7) - 7;
    return (e >= 0 ? 0x0102040810204080ull << (8 * e) : 0x0102040810204080ull >> (8 * -e)) ^ bit(sq);
}

// What a square decides: its lines (the square itself excluded), the knight's and the king's steps from it.
struct Square { u64 diag, anti, knight, king, rank, file, s, less, less_rev; int sq; };
// The first four are looked up: a table of 2 KiB in LDS that the workgroup fills at its start, a field by
// each of its four wavefronts (a field is 10 to 25 instructions, and a lane asks for three squares).
__device__ __forceinline__ Square square(int sq, const ulonglong2 (*table)[2]) {
    Square q;
    q.sq = sq;
    q.s = bit(sq);
    q.less = ~0ull << sq;             // -s
    q.less_rev = ~0ull << (63 - sq);
    q.rank = (0xFFull << (sq & 56)) ^ q.s;
    q.file = (FILE_A << (sq & 7)) ^ q.s;
    const ulonglong2 a = table[sq][0], b = table[sq][1];
    q.diag = a.x; q.anti = a.y; q.knight = b.x; q.king = b.y;
    return q;
}
// the rank that square sq is on; off the board, some other one, which no king's step from beside it reaches
__device__ __forceinline__ u64 rank_of(int sq) { return 0xFFull << (sq & 56); }

__device__ __forceinline__ u64 line_attacks(u64 occ, u64 m, const Square& q) { return line_attacks(occ, m, q.less, q.less_rev); }

// The pieces of `e` that attack square q, given occupancy occ.  Looked at from the square: a rook placed
// there sees the enemy's orthogonal sliders exactly when they see it, and so for the other kinds.
__device__ __forceinline__ u64 attackers(const Enemy& e, u64 occ, const Square& q) {
    // a white pawn on (r-1, c+-1) attacks (r, c); a black one from (r+1, c+-1): the king's steps on the rank behind, the
    // one straight behind left out by its file
    const u64 sliders = logic<(A | B) & C>(line_attacks(occ, q.rank, q), line_attacks(occ, q.file, q), e.orth) |
                        logic<(A | B) & C>(line_attacks(occ, q.diag, q), line_attacks(occ, q.anti, q), e.diag);
    const u64 pawn_from = logic<A & B & (0xFF ^ C)>(q.king, rank_of(q.sq + e.behind), q.file);
    return logic<A | (B & C)>(logic<A | (B & C)>(logic<A | (B & C)>(sliders, pawn_from, e.pawns), q.knight, e.knights), q.king, e.king);
}

// the squares strictly between q and x (one bit) if they share a line, else none
__device__ __forceinline__ u64 between(const Square& q, u64 x) {
    const u64 line = (q.rank & x) ? q.rank : (q.file & x) ? q.file : (q.diag & x) ? q.diag : (q.anti & x) ? q.anti : 0;
    const u64 hi = x > q.s ? x : q.s, lo = x > q.s ? q.s : x;
    return logic<A & (0xFF ^ (B | C))>(line & (hi + ~0ull), lo, lo + ~0ull);
}

// OR over the sixteen lanes of a row, in every lane
template <int CTRL>
__device__ __forceinline__ unsigned or_ror(unsigned v) {
    return v | (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, true);
}
__device__ __forceinline__ u64 row_or(u64 v) {
    unsigned lo = (unsigned)v, hi = (unsigned)(v >> 32);
    lo = or_ror<0x128>(lo); hi = or_ror<0x128>(hi);    // row_ror:8, 4, 2, 1
    lo = or_ror<0x124>(lo); hi = or_ror<0x124>(hi);
    lo = or_ror<0x122>(lo); hi = or_ror<0x122>(hi);
    lo = or_ror<0x121>(lo); hi = or_ror<0x121>(hi);
    return ((u64)hi << 32) | lo;
}

typedef ulonglong2 Table[64][2];   // of a workgroup, in LDS: a square's diagonals, knight's and king's steps

__device__ __forceinline__ void fill(Table& table) {   // 256 lanes: a wavefront a field
    const int sq = threadIdx.x & 63, field = threadIdx.x >> 6;
    reinterpret_cast<u64*>(table[sq])[field] = field == 0 ? diagonal(sq) : field == 1 ? antidiagonal(sq) : field == 2 ? knight_pattern(bit(sq)) : king_pattern(bit(sq));
    __syncthreads();
}

// A row's position: where the piece in slot `lane % 16` of the side to move may go, 0 without a piece of that side.  `attacked`
// is told whether the king is once that piece has left its square: for slot 15, the king, whether it stands in check.  (Told, and
// not returned: two registers through the rest would cost a wavefront of six per SIMD.)
template <typename F>
__device__ __forceinline__ u64 of_row(const uint16_t* bw, bool black, int lane, const Table& table, F&& attacked) {
    const int slot = lane & 15;
    const unsigned w = bw[(black ? 16 : 0) + slot], v = bw[(black ? 0 : 16) + slot];
    const unsigned kw = bw[black ? 31 : 15], ke = bw[black ? 15 : 31];

    // bitboards, the same in every lane of the row
    const bool mine = !(w & CAPTURED) && ((w >> 10) & 1) == (unsigned)black;
    const bool theirs = !(v & CAPTURED) && ((v >> 10) & 1) != (unsigned)black;
    const int sq = w & 63, t = (w >> 6) & 7, te = (v >> 6) & 7;
    const u64 fb = bit(sq), vb = theirs ? bit(v & 63) : 0;
    const u64 own = row_or(mine ? fb : 0);
    Enemy e;
    const int ahead8 = black ? -8 : 8;                  // one rank ahead for the side to move
    e.behind = ahead8;
    e.pawns = row_or(te == PAWN ? vb : 0);
    const u64 ep_pawns = row_or(te == PAWN && (v & SPECIAL) ? vb : 0);
    e.knights = row_or(te == KNIGHT ? vb : 0);
    e.diag = row_or(te == BISHOP || te == QUEEN ? vb : 0);
    e.orth = row_or(te == ROOK || te == QUEEN ? vb : 0);
    e.king = (ke & CAPTURED) ? 0 : bit(ke & 63);
    const u64 opp = logic<A | B | C>(logic<A | B | C>(e.pawns, e.knights, e.diag), e.orth, e.king);
    const u64 occ = own | opp;
    const int ksq = kw & 63;
    // an unmoved own rook on its corner
    const int rowbits = lane & 48;
    const unsigned home = black ? 56u : 0u, rookw = (black ? COLOR : 0u) | (ROOK << 6);
    const bool rook_short = (__ballot(w == (rookw | (home + 7))) >> rowbits) & 0xffff;
    const bool rook_long = (__ballot(w == (rookw | home)) >> rowbits) & 0xffff;

    // ---- what attacks the king once this lane's piece has left its square (the king's own lane: the check) ----
    const Square king = square(ksq, table);
    const u64 att = attackers(e, occ & ~fb, king);
    u64 allowed = ~0ull;
    if (att) allowed = (att & (att - 1)) ? 0 : att | between(king, att);
    attacked(att != 0);

    // ---- this lane's king step or castling square ----
    const u64 kb = king.s;
    unsigned safe;
    {
        const int k9 = slot + (slot >= 4), dr = k9 / 3 - 1, dc = k9 % 3 - 1;
        const bool step = slot < 8;
        const int r = (ksq >> 3) + dr, c = (ksq & 7) + dc;
        const bool kingside = slot < 11;
        const bool unmoved = !(kw & (CAPTURED | SPECIAL));
        int at = step ? r * 8 + c : kingside ? ksq + (slot - 8) : ksq - (slot - 11);
        const bool way_free = kingside ? rook_short && !(occ & (0x60ull << home)) : slot < 14 && rook_long && !(occ & (0x0Eull << home));
        bool may = step ? (unsigned)r < 8u && (unsigned)c < 8u : unmoved && way_free;
        at &= 63;
        const u64 tb = bit(step ? at : (int)home + (kingside ? 6 : 2));
        if (step) may = may && !(own & tb);
        // castling moves the rook too: where it may, its square is taken and the one it goes to free
        const u64 rook = (u64)(step ? 0u : kingside ? 0xA0u : 0x09u) << home;
        const u64 occ2 = logic<(A & (0xFF ^ B)) | C>(occ, kb, tb) ^ rook;
        const bool ok = may && (attackers(e, occ2, square(at, table)) & ~tb) == 0;   // what the step takes attacks no more
        safe = (unsigned)(__ballot(ok) >> rowbits) & 0xffffu;
    }

    // ---- the squares this lane's piece reaches ----
    u64 legal = 0, ep = 0;
    const Square from = square(sq, table);
    if (mine) {
        if (t == PAWN) {
            const int r = sq >> 3;
            const int up = black ? 0 : 8, down = 8 - up;
            const u64 at = (fb << up) >> down;
            const u64 one = at & ~occ, two = r == (black ? 6 : 1) ? ((one << up) >> down) & ~occ : 0;
            // the two squares ahead to either side, and the enemy pawns beside us that just double-pushed
            const u64 sides = logic<A & B & (0xFF ^ C)>(from.king, rank_of(sq + ahead8), at);
            legal = logic<A | (B & C)>(one | two, sides, opp) & allowed;
            if (r == (black ? 3 : 4)) {
                const u64 beside = logic<A & B & C>(from.king, from.rank, ep_pawns);
                ep = ((beside << up) >> down) & ~opp;
            }
        } else if (t == KNIGHT) {
            legal = logic<A & (0xFF ^ B) & C>(from.knight, own, allowed);
        } else if (t == KING) {
            const u64 around = (safe & 7u) | ((safe & 8u) << 5) | ((safe & 16u) << 6) | ((u64)(safe & 0xE0u) << 11);
            legal = ksq >= 9 ? around << (ksq - 9) : around >> (9 - ksq);
            if (((safe >> 8) & 7u) == 7u) legal |= bit(home + 6);
            if (((safe >> 11) & 7u) == 7u) legal |= bit(home + 2);
        } else if (t == BISHOP || t == ROOK || t == QUEEN) {
            u64 reach = 0;
            if (t != BISHOP) reach = line_attacks(occ, from.rank, from) | line_attacks(occ, from.file, from);
            if (t != ROOK) reach = logic<A | B | C>(reach, line_attacks(occ, from.diag, from), line_attacks(occ, from.anti, from));
            legal = logic<A & (0xFF ^ B) & C>(reach, own, allowed);
        }
    }
    while (__any(ep != 0)) {   // en passant: replayed, the victim is behind the target
        const u64 tb = ep & (0 - ep), victim = black ? tb << 8 : tb >> 8;
        if (ep && (attackers(e, ((occ & ~fb) | tb) & ~victim, king) & ~(tb | victim)) == 0) legal |= tb;
        ep &= ep - 1;
    }
    return legal;
}

}  // namespace moves
}  // namespace bf
