// cantor.hpp -- the arithmetic and the index maps of the Cantor transform
// (fft.hip), written once for device and host: the kernels and the CPU
// emulation of the tests run the same functions.
//
// Field elements inside the transform are kept in a tower basis of
// GF(2^64) over GF(2^8):  u3 = b[8], u4 = b[16], u5 = b[32] of the Cantor
// basis, u_k^2 = u_k + c_k with c3 = b[7], c4 = b[15], c5 = b[31], and
// bytes in the basis b[0..7].  span(b[0..2^k-1]) is the subfield
// GF(2^(2^k)), so the twiddle of a butterfly whose index t has at most 7,
// 15 or 31 bits lies in GF(2^8), GF(2^16) or GF(2^32), and its product
// with an element acts byte-wise: a product with a constant of GF(2^8) is
// three byte permutes per four bytes (the 3 + 3 + 2 bits of a byte each
// select from an eight-entry table).  Per 32-bit word that is 5
// operations to split the bits, 3 permutes and 2 three-input XORs; a
// GF(2^64) product from 32 x 32 integer multiplies takes 144.
//
// Two elements form a unit of four words, so that each word holds the
// same tower coordinate of both: word p (bits of p: u3, u4) holds bytes
// (E u5^0, E u5^1, F u5^0, F u5^1) of elements E = 2i and F = 2i + 1.
#pragma once
#include "gf2t_arith.hpp"

struct alignas(16) U4 {
    u32 w[4];
};
// A twiddle W = Wa + Wb u4 (Wa, Wb in GF(2^16)) as the bytes its product
// needs: p for the product with Wa, q with c4 Wb, r with Wa + Wb, each as
// the three byte factors of a Karatsuba product over GF(2^8), v0, c3 v1 and
// v0 + v1.  Every byte is linear in W.  Two to a word, each times 16, the
// byte offset of its entry in the first multiply table (a quarter of it in
// the second).
struct alignas(16) TwEnt {
    u32 p02, r02;   // bytes 0 (low half) and 2 of p, r: an element v of
                    // GF(2^8) added to W adds v to all four
    u32 p1r1, q01, q2;
    u32 pad[3];
};
GF2T_HD u32 tw_lo(u32 w) { return w & 0xFF0u; }
GF2T_HD u32 tw_hi(u32 w) { return w >> 16; }
GF2T_HD u32 tw_byte(u32 v) { return (v << 4) | (v << 20); }
GF2T_HD TwEnt tw_xor(const TwEnt &a, const TwEnt &b) {
    return TwEnt{a.p02 ^ b.p02, a.r02 ^ b.r02, a.p1r1 ^ b.p1r1, a.q01 ^ b.q01, a.q2 ^ b.q2, {}};
}
// multiply-by-v tables: a = images of the byte's bits 0..2 (8 bytes), b of
// bits 3..5, c of bits 6, 7 (4 bytes)
struct Mul8 {
    u32 a0, a1, b0, b1, c;
};
struct alignas(16) FftTables {
    // the first two runs are copied to LDS as they stand
    u32 mulA[256][4];   // a0, a1, b0, b1 of the product with v
    u32 mulB[256];      // c (apart: rows of 16 bytes spread over all LDS
                        // banks; with rows of 32, the low pass of a 2^23-
                        // point product took 360 us instead of 267)
    u32 d32[4][256];    // GF(2^32): tower byte p -> basis of powers of rho
    u32 d5[4][256];     // the same times c5
    u32 b32[4][256];    // back: byte k -> the four tower bytes
    u64 emb[8][256];    // polynomial-basis byte k -> tower halfwords
    u64 une[8][256];    // tower byte k -> polynomial basis
    TwEnt tw[4][256];   // W(t) for byte k of t: sum of b[8k + j + 1] over its bits j
};

// rho: a root of x^32 + x^7 + x^3 + x^2 + 1 in GF(2^64)
constexpr u64 FFT_RHO = 0x0b8b4dab63c1ea4bULL;

// ------------------------------------------------------------ byte maps
struct Bits8 {   // the 3 + 3 + 2 bits of four bytes
    u32 l, m, h;
};
GF2T_HD Bits8 split8(u32 x) {
    return Bits8{x & 0x07070707u, (x >> 3) & 0x07070707u, (x >> 6) & 0x03030303u};
}
GF2T_HD Bits8 xor8(const Bits8 &x, const Bits8 &y) {
    return Bits8{x.l ^ y.l, x.m ^ y.m, x.h ^ y.h};
}
GF2T_HD u32 map8(const Mul8 &t, const Bits8 &s) {
    return xor3_32(perm8(t.a1, t.a0, s.l), perm8(t.b1, t.b0, s.m), perm8(t.c, t.c, s.h));
}
// The factor tables of one twiddle, by the subfield it lies in: CLS 8 one
// table, 16 three, 32 nine; tab(off) reads the entry at byte offset off.
// All of them but those of bytes 0 and 2 of p and r stay the same when an
// element of GF(2^8) is added to W, so a stage fetches those once per
// level.
template <int CLS>
struct TwTab {
    Mul8 p0, p1, p2, q0, q1, q2, r0, r1, r2;
    template <class Tab>
    GF2T_HDM void fixed(const TwEnt &w, const Tab &tab) {
        if (CLS >= 16) p1 = tab(tw_lo(w.p1r1));
        if (CLS >= 32) {
            r1 = tab(tw_hi(w.p1r1));
            q0 = tab(tw_lo(w.q01));
            q1 = tab(tw_hi(w.q01));
            q2 = tab(w.q2);
        }
    }
    template <class Tab>   // for W + v, v in GF(2^8)
    GF2T_HDM void add(const TwEnt &w, u32 v, const Tab &tab) {
        const u32 p = w.p02 ^ tw_byte(v), r = w.r02 ^ tw_byte(v);
        p0 = tab(tw_lo(p));
        if (CLS >= 16) p2 = tab(tw_hi(p));
        if (CLS >= 32) {
            r0 = tab(tw_lo(r));
            r2 = tab(tw_hi(r));
        }
    }
};

struct UnitBits {   // the bits of a unit's words
    Bits8 b[4];
};
GF2T_HD UnitBits unit_bits(const U4 &x) {
    return UnitBits{{split8(x.w[0]), split8(x.w[1]), split8(x.w[2]), split8(x.w[3])}};
}
// y += W x on units, x by its bits
template <int CLS>
GF2T_HD void unit_madd(U4 &y, const UnitBits &x, const TwTab<CLS> &t) {
    if (CLS == 8) {
#pragma unroll
        for (int k = 0; k < 4; k++) y.w[k] ^= map8(t.p0, x.b[k]);
    } else if (CLS == 16) {
#pragma unroll
        for (int k = 0; k < 4; k += 2) {
            const Bits8 &s0 = x.b[k], &s1 = x.b[k + 1];
            const u32 P = map8(t.p0, s0);
            y.w[k] = xor3_32(y.w[k], P, map8(t.p1, s1));
            y.w[k + 1] = xor3_32(y.w[k + 1], P, map8(t.p2, xor8(s0, s1)));
        }
    } else {
        const Bits8 &a0 = x.b[0], &a1 = x.b[1], &b0 = x.b[2], &b1 = x.b[3];
        const Bits8 c0 = xor8(a0, b0), c1 = xor8(a1, b1);
        const u32 P0 = map8(t.p0, a0);
        const u32 A = P0 ^ map8(t.p1, a1);             // Wa Xa, low and high
        const u32 B = P0 ^ map8(t.p2, xor8(a0, a1));
        const u32 Q0 = map8(t.q0, b0);
        y.w[0] = xor3_32(y.w[0], A, Q0) ^ map8(t.q1, b1);
        y.w[1] = xor3_32(y.w[1], B, Q0) ^ map8(t.q2, xor8(b0, b1));
        const u32 R0 = map8(t.r0, c0);
        y.w[2] = xor3_32(y.w[2], A, R0) ^ map8(t.r1, c1);
        y.w[3] = xor3_32(y.w[3], B, R0) ^ map8(t.r2, xor8(c0, c1));
    }
}
GF2T_HD void unit_xor(U4 &y, const U4 &x) {
    for (int k = 0; k < 4; k++) y.w[k] ^= x.w[k];
}

// A thread of the butterflies holds 2^RB units and takes RB levels between
// exchanges.  RB = 2 keeps the kernels at 58-78 registers (six to eight
// waves per SIMD) and the code of a stage at four unrolled products; 16
// units (RB = 4) took 100-210 registers, and a straight-line stage of 32
// products ran at the speed its instructions were fetched: the fused low
// pass of a 2^23-point product took 657 us with RB = 4, 282 with 3, 257
// with 2 (and a 2^20-point transform pair 325, 256, 227 us).
constexpr int RB = 2;

// Up to RB butterfly levels on 2^RB units in registers: row bit rb of the
// unit index is a level, active when bit rb of act is set; W[rb] is the
// twiddle of the rows whose bits above rb are clear, and the rows whose
// bits above rb spell `up` add sum of b[j + 1] over the bits j of up, the
// byte up << 1.  zero: the W[.] are all 0 (the topmost levels), so the rows
// with up = 0 have no product.
template <int rb, int CLS, bool INV, class Tab>
GF2T_HD void fft_level(U4 *x, const TwEnt &W, bool zero, const Tab &tab) {
    TwTab<CLS> t;
    t.fixed(W, tab);
#pragma unroll
    for (int up = 0; up < ((1 << (RB - 1)) >> rb); up++) {
        const bool mul = up || !zero;
        if (mul) t.add(W, (u32)up << 1, tab);
#pragma unroll
        for (int lo = 0; lo < (1 << rb); lo++) {
            const int r0 = (up << (rb + 1)) | lo, r1 = r0 | (1 << rb);
            if (INV) {
                unit_xor(x[r1], x[r0]);
                if (mul) unit_madd<CLS>(x[r0], unit_bits(x[r1]), t);
            } else {
                if (mul) unit_madd<CLS>(x[r0], unit_bits(x[r1]), t);
                unit_xor(x[r1], x[r0]);
            }
        }
    }
}
template <int CLS, bool INV, class Tab>
GF2T_HD void fft_stage(U4 *x, int act, const TwEnt *W, bool zero, const Tab &tab) {
    static_assert(RB == 2, "two levels");
    if (INV) {
        if (act & 1) fft_level<0, CLS, true>(x, W[0], zero, tab);
        if (act & 2) fft_level<1, CLS, true>(x, W[1], zero, tab);
    } else {
        if (act & 2) fft_level<1, CLS, false>(x, W[1], zero, tab);
        if (act & 1) fft_level<0, CLS, false>(x, W[0], zero, tab);
    }
}
// Level 0, inside the units: rows r and r + 1 (r even) are taken together,
// E of both in one word and F of both in another; W is the twiddle of row
// 0, row r adds the byte r << 1.
template <int CLS, bool INV, class Tab>
GF2T_HD void fft_level0(U4 *x, const TwEnt &W, const Tab &tab) {
    const u32 LO = 0x05040100u, HI = 0x07060302u, TOP = 0xFFFF0000u;
    const Mul8 b1 = tab(2 << 4);
    TwTab<CLS> t;
    t.fixed(W, tab);
#pragma unroll
    for (int r = 0; r < (1 << RB); r += 2) {
        t.add(W, (u32)r << 1, tab);
        U4 e, f;
#pragma unroll
        for (int p = 0; p < 4; p++) {
            e.w[p] = perm8(x[r + 1].w[p], x[r].w[p], LO);
            f.w[p] = perm8(x[r + 1].w[p], x[r].w[p], HI);
        }
        if (INV) unit_xor(f, e);
        const UnitBits s = unit_bits(f);
        unit_madd<CLS>(e, s, t);
#pragma unroll
        for (int p = 0; p < 4; p++)   // row r + 1: W + b[1]
            e.w[p] ^= map8(b1, Bits8{s.b[p].l & TOP, s.b[p].m & TOP, s.b[p].h & TOP});
        if (!INV) unit_xor(f, e);
#pragma unroll
        for (int p = 0; p < 4; p++) {
            x[r].w[p] = perm8(f.w[p], e.w[p], LO);
            x[r + 1].w[p] = perm8(f.w[p], e.w[p], HI);
        }
    }
}

// W(t) from the byte tables
template <class TwT>
GF2T_HD TwEnt tw_of(const TwT &tw, u32 t) {
    return tw_xor(tw_xor(tw[0][t & 255], tw[1][(t >> 8) & 255]),
                  tw_xor(tw[2][(t >> 16) & 255], tw[3][t >> 24]));
}
// W + v for v in GF(2^8)
GF2T_HD TwEnt tw_add8(TwEnt w, u32 v) {
    const u32 b = tw_byte(v);
    w.p02 ^= b;
    w.r02 ^= b;
    return w;
}

// --------------------------------------------------- basis conversions
GF2T_HD U4 unit_from(u64 e, u64 f) {
    const u32 e0 = (u32)e, e1 = (u32)(e >> 32), f0 = (u32)f, f1 = (u32)(f >> 32);
    U4 u;
    u.w[0] = perm8(f0, e0, 0x05040100u);
    u.w[1] = perm8(f0, e0, 0x07060302u);
    u.w[2] = perm8(f1, e1, 0x05040100u);
    u.w[3] = perm8(f1, e1, 0x07060302u);
    return u;
}
template <class E>   // 32-bit chunks
GF2T_HD U4 unit_embed32(u32 e, u32 f, const E &emb) {
    u64 a = 0, b = 0;
    for (int k = 0; k < 4; k++) {
        a ^= emb[k][(e >> (8 * k)) & 255];
        b ^= emb[k][(f >> (8 * k)) & 255];
    }
    return unit_from(a, b);
}
template <class E>   // whole elements
GF2T_HD U4 unit_embed64(u64 e, u64 f, const E &emb) {
    u64 a = 0, b = 0;
    for (int k = 0; k < 8; k++) {
        a ^= emb[k][(e >> (8 * k)) & 255];
        b ^= emb[k][(f >> (8 * k)) & 255];
    }
    return unit_from(a, b);
}
template <class E>
GF2T_HD void unit_unembed(const U4 &u, const E &une, u64 &e, u64 &f) {
    e = f = 0;
    for (int p = 0; p < 4; p++) {
        const u32 w = u.w[p];
        e = xor3(e, une[2 * p][w & 255], une[2 * p + 1][(w >> 8) & 255]);
        f = xor3(f, une[2 * p][(w >> 16) & 255], une[2 * p + 1][w >> 24]);
    }
}

// ------------------------------------------------------ products of units
// GF(2^64) = GF(2^32)[u5]: both halves to the polynomial basis of
// GF(2^32), three 32 x 32 products, two reductions, and back.
GF2T_HD u32 red32(u64 v) {
    const u32 lo = (u32)v, h = (u32)(v >> 32);
    const u64 t = (u64)lo ^ (u64)h ^ ((u64)h << 2) ^ ((u64)h << 3) ^ ((u64)h << 7);
    const u32 o = (u32)(t >> 32);
    return (u32)t ^ o ^ (o << 2) ^ (o << 3) ^ (o << 7);
}
struct Half32 {   // (E u5^0, E u5^1, F u5^0, F u5^1), powers of rho
    u32 v[4];
};
template <class D>
GF2T_HD Half32 unit_to32(const U4 &u, const D &d) {
    Half32 h;
    for (int k = 0; k < 4; k++)
        h.v[k] = xor3_32(d[0][(u.w[0] >> (8 * k)) & 255], d[1][(u.w[1] >> (8 * k)) & 255],
                         d[2][(u.w[2] >> (8 * k)) & 255]) ^
                 d[3][(u.w[3] >> (8 * k)) & 255];
    return h;
}
// c5 times the u5^1 halves (v[1], v[3]; the others unused)
template <class D>
GF2T_HD Half32 unit_c5(const U4 &u, const D &d5) {
    Half32 h;
    h.v[0] = h.v[2] = 0;
    for (int k = 1; k < 4; k += 2)
        h.v[k] = xor3_32(d5[0][(u.w[0] >> (8 * k)) & 255], d5[1][(u.w[1] >> (8 * k)) & 255],
                         d5[2][(u.w[2] >> (8 * k)) & 255]) ^
                 d5[3][(u.w[3] >> (8 * k)) & 255];
    return h;
}
struct Acc64 {   // unreduced low and high halves of a sum of products
    u64 lo, hi;
};
GF2T_HD void acc_mul(Acc64 &s, u32 a0, u32 a1, u32 b0, u32 b1, u32 b1c5) {
    const u64 P = clmul32(a0, b0);
    s.lo = xor3(s.lo, P, clmul32(a1, b1c5));
    s.hi = xor3(s.hi, P, clmul32(a0 ^ a1, b0 ^ b1));
}
template <class B>
GF2T_HD U4 unit_back(const Acc64 &E, const Acc64 &F, const B &b32) {
    const u32 v[4] = {red32(E.lo), red32(E.hi), red32(F.lo), red32(F.hi)};
    u32 t[4];
    for (int k = 0; k < 4; k++)
        t[k] = xor3_32(b32[0][v[k] & 255], b32[1][(v[k] >> 8) & 255], b32[2][(v[k] >> 16) & 255]) ^
               b32[3][v[k] >> 24];
    // t[k] holds byte k of the words 0..3: transpose
    const u32 a = perm8(t[1], t[0], 0x05010400u), b = perm8(t[1], t[0], 0x07030602u);
    const u32 c = perm8(t[3], t[2], 0x05010400u), d = perm8(t[3], t[2], 0x07030602u);
    U4 u;
    u.w[0] = perm8(c, a, 0x05040100u);
    u.w[1] = perm8(c, a, 0x07060302u);
    u.w[2] = perm8(d, b, 0x05040100u);
    u.w[3] = perm8(d, b, 0x07060302u);
    return u;
}
template <class T>
GF2T_HD U4 unit_mul(const U4 &x, const U4 &y, const T &d32, const T &d5, const T &b32) {
    const Half32 a = unit_to32(x, d32), b = unit_to32(y, d32), c = unit_c5(y, d5);
    Acc64 E{0, 0}, F{0, 0};
    acc_mul(E, a.v[0], a.v[1], b.v[0], b.v[1], c.v[1]);
    acc_mul(F, a.v[2], a.v[3], b.v[2], b.v[3], c.v[3]);
    return unit_back(E, F, b32);
}

// ------------------------------------------------------- index maps
// A butterfly pass over the element bits [a, a + w) (w <= 8) of a 2^m-point
// transform, in tiles of 2^tb units: local bits [0, lc) are the unit bits
// [0, lc) of memory, local bits [lc, tb) are the window; tile `blk` holds
// the rest.  A thread has 2^RB units; in stage s they are the local bits
// [tb - RB (s + 1), tb - RB s), and the thread number is the others.
struct BfPass {
    int m, a, w, tb;
};
struct BfTile {
    u32 base;     // unit index of local index 0
    u32 hi;       // element index bits above the window
};
GF2T_HD BfTile bf_tile(const BfPass &P, u32 blk) {
    const int lc = P.tb - P.w, nlo = P.a - 1 - lc;
    const u32 lo = blk & ((1u << nlo) - 1), up = blk >> nlo;
    return BfTile{(lo << lc) | (up << (P.a - 1 + P.w)), up << (P.a + P.w)};
}
GF2T_HD u32 bf_unit(const BfPass &P, const BfTile &T, u32 local) {
    const int lc = P.tb - P.w;
    return T.base + (local & ((1u << lc) - 1)) + ((local >> lc) << (P.a - 1));
}
// index with the low k bits of t low, r above them, the rest of t on top
GF2T_HD u32 spread_rows(u32 t, int r, int k, int bits) {
    return (t & ((1u << k) - 1)) | ((u32)r << k) | ((t >> k) << (k + bits));
}
GF2T_HD u32 bf_local(const BfPass &P, int s, u32 tid, int r) {
    return spread_rows(tid, r, P.tb - RB * (s + 1), RB);
}
GF2T_HD int bf_stages(const BfPass &P) { return (P.w + RB - 1) / RB; }
// row bit j of stage s is element bit a + w - RB (s + 1) + j, a level when
// that is a or more; the thread's bits above the rows are the element bits
// from there up to a + w, at most seven above a level
GF2T_HD int bf_active(const BfPass &P, int s) {
    const int out = RB * (s + 1) - P.w;   // row bits below the window
    return out > 0 ? ((1 << RB) - 1) & ~((1 << out) - 1) : (1 << RB) - 1;
}
template <class TwT>
GF2T_HD void bf_twiddles(const BfPass &P, const BfTile &T, int s, u32 tid, const TwT &tw,
                         TwEnt *W) {
    const u32 up = tid >> (P.tb - RB * (s + 1));
#pragma unroll
    for (int j = 0; j < RB; j++) {
        const int L = P.a + P.w - RB * (s + 1) + j;
        W[j] = tw_add8(tw_of(tw, L >= P.a ? T.hi >> (L + 1) : 0), (up << (RB - j)) & 255);
    }
}

// the twiddles of the stage's row 0 are all 0: the top of the transform
GF2T_HD bool bf_zero(const BfPass &P, const BfTile &T, int s) { return s == 0 && T.hi == 0; }

// The last (lowest) levels 7..0: a wave's 64 lanes hold 64 << RB
// consecutive units, in stage s the rows being the unit bits from
// lo_pos(s) up: levels lo_pos + 1 + j on row bits j, level 0 inside the
// units after the last stage: unit bits 6 and 5, 4 and 3, 2 and 1, 1 and 0
// (only bit 0 a level there).
GF2T_HD constexpr int lo_pos(int s) { return 7 - RB * (s + 1) > 0 ? 7 - RB * (s + 1) : 0; }
GF2T_HD constexpr int lo_stages() { return (7 + RB - 1) / RB; }
GF2T_HD u32 lo_unit(int s, u32 lane, int r) { return spread_rows(lane, r, lo_pos(s), RB); }
GF2T_HD int lo_active(int m, int s) {
    int act = 0;
    for (int j = 0; j < RB; j++) {
        const int bit = lo_pos(s) + j;   // unit bit, level bit + 1
        if (bit < 7 - RB * s && bit + 1 < m) act |= 1 << j;
    }
    return act;
}
// twiddle of row 0 at level L, wave's first unit ubase: t_lane are the lane
// bits above the rows; those below 2^7 are the byte t << 1, the two bits
// above go through the table hi
template <class TwC, class TwG>
GF2T_HD TwEnt lo_twiddle(u32 ubase, int L, u32 tlane, bool high, const TwC &tw, const TwG &hi) {
    TwEnt w = tw_add8(tw_of(tw, (ubase << 1) >> (L + 1)), (tlane << 1) & 255);
    if (high) w = tw_xor(w, hi[(tlane >> 7) & 3]);
    return w;
}
template <int S, class TwC, class TwG>
GF2T_HD void lo_twiddles(u32 ubase, u32 lane, const TwC &tw, const TwG &hi, TwEnt *W, TwEnt &W0) {
    constexpr int pos = lo_pos(S);
#pragma unroll
    for (int j = 0; j < RB; j++)
        W[j] = lo_twiddle(ubase, pos + 1 + j, (lane >> pos) << (RB - 1 - j),
                          6 - pos + RB - 1 - j > 7, tw, hi);
    if (S == lo_stages() - 1) W0 = lo_twiddle(ubase, 0, lane << RB, true, tw, hi);
}

// ------------------------------------------------- conversion of the basis
// From powers of X to the basis X_i = prod s_k(X)^(bit k of i), s_k the
// vanishing polynomial of span(b[0..k-1]), and back.  s_h(X) = X^(2^h) + X
// for h = 1, 2, 4, 8, 16, and s_(j+k) = s_j(s_k), so a polynomial of
// 2^k coefficients is expanded in powers of s_h (h the largest of those
// below k) and both index parts are converted by themselves.  One step of
// that expansion, X^(2^(h+e)) = s_h^(2^e) + X^(2^e), on blocks of
// 2^(h+e+1) coefficients with halves f0, f1 of 2^(h+e):
//   f1[p] += f1[2^(h+e) - 2^e + p] for p < 2^e;  f0[p + 2^e] += f1[p].
// Only XORs of whole coefficients, so forward it runs on the 32-bit input
// chunks, before they become field elements.
// T_h at register bit POS of N coefficients in registers
template <int H, int POS, int N, bool INV, class T>
GF2T_HD void conv_regs(T *x) {
    constexpr int U = 1 << POS, L = U << H;
#pragma unroll
    for (int b = 0; b < N; b += 2 * L) {
        T *f0 = x + b, *f1 = x + b + L;
        if (!INV) {
#pragma unroll
            for (int p = 0; p < U; p++) f1[p] ^= f1[L - U + p];
        }
#pragma unroll
        for (int p = 0; p + U < L; p++) f0[p + U] ^= f1[p];
        if (INV) {
#pragma unroll
            for (int p = 0; p < U; p++) f1[p] ^= f1[L - U + p];
        }
    }
}
// the four register bits from POS on
template <int POS, int N, bool INV, class T>
GF2T_HD void conv_nibble(T *x) {
    if (!INV) {
        conv_regs<2, POS + 1, N, false>(x);
        conv_regs<2, POS, N, false>(x);
        conv_regs<1, POS + 2, N, false>(x);
        conv_regs<1, POS, N, false>(x);
    } else {
        conv_regs<1, POS, N, true>(x);
        conv_regs<1, POS + 2, N, true>(x);
        conv_regs<2, POS, N, true>(x);
        conv_regs<2, POS + 1, N, true>(x);
    }
}
// Steps e0 + K - 1 .. e0 of the expansion in powers of s_h, with unit =
// 2^e0 (times 2^off inside a higher index part): 2^K rows of 2^hb
// coefficients, hb = h + e0 + off, each step adding row k (bit e set) to
// row k - 2^e, 2^e units further on.  In columns skewed by row, i = c -
// (2^K - 1 - k) unit, the rows add in place; the first and last columns,
// where a shift leaves its row, are a problem of the same form with rows
// of 2^K units (the middle of each row left out), done apart.
struct ConvStep {
    int K, hb, ub;   // rows 2^K of 2^hb coefficients, unit 2^ub
};
GF2T_HD u32 conv_full(const ConvStep &s) { return (1u << s.hb) - (1u << (s.ub + s.K)); }
// skewed column number t < conv_full: coefficient of row k, within its row
GF2T_HD u32 conv_col(const ConvStep &s, u32 t, int k) {
    return (1u << s.ub) + t + ((u32)((1 << s.K) - 1 - k) << s.ub);
}
// coefficient of row k, boundary unit q < 2^K, at rho < unit, in its row
GF2T_HD u32 conv_edge(const ConvStep &s, int k, u32 q, u32 rho) {
    const u32 n = 1u << s.K;
    return q < n - (u32)k ? (q << s.ub) + rho : (1u << s.hb) - ((n - q) << s.ub) + rho;
}
// step e on the 2^K x 2^K coefficients of an edge, x(row * 2^K + q): pair
// number idx of half of them
template <class X>
GF2T_HD void conv_edge_pair(X &&x, int K, int e, bool inv, u32 idx) {
    const u32 L = 1u << (K + e), U = 1u << e;
    const u32 p = idx & (L - 1), f0 = idx + (idx & ~(L - 1)), f1 = f0 + L;
    auto v = x(f1);
    if (!inv && p < U) {
        v ^= x(f1 + L - U);
        x(f1) = v;
    }
    if (p + U < L) x(f0 + U) ^= v;
    if (inv && p < U) x(f1) = v ^ x(f1 + L - U);
}
// Inside a tile the steps run on local index bits, 16 coefficients per
// thread in registers between two passes through LDS; x(i) is local
// coefficient i, q the thread of 2^(T-4).
// One step (K = 1): eight pairs, T_h of s at local bit s.ub
template <bool INV, class E, class X>
GF2T_HD void conv_tile1(X &&x, u32 q, u32 threads, const ConvStep &s) {
    const u32 L = 1u << s.hb, U = 1u << s.ub;
    E v[8];
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const u32 idx = q + (u32)i * threads, p = idx & (L - 1), f1 = idx + (idx & ~(L - 1)) + L;
        v[i] = x(f1);
        if (!INV && p < U) {
            v[i] ^= x(f1 + L - U);
            x(f1) = v[i];
        }
    }
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const u32 idx = q + (u32)i * threads, p = idx & (L - 1), f0 = idx + (idx & ~(L - 1));
        if (p + U < L) x(f0 + U) ^= v[i];
        if (INV && p < U) x(f0 + L) = v[i] ^ x(f0 + L + L - U);
    }
}
// Two steps (K = 2): four skewed columns of four rows, or the 16
// coefficients of an edge.  A block of four rows of 2^hb has 2^hb / 4
// threads: (2^hb - 4 unit) / 4 for the columns, unit for the edges.
template <bool INV, class E, class X>
GF2T_HD void conv_tile2(X &&x, u32 q, const ConvStep &s) {
    const u32 per = 1u << (s.hb - 2), cols = per - (1u << s.ub);
    const u32 t = q & (per - 1), base = (q >> (s.hb - 2)) << (s.hb + 2);
    E v[16];
    if (t < cols) {
#pragma unroll
        for (int c = 0; c < 4; c++)
#pragma unroll
            for (int k = 0; k < 4; k++)
                v[4 * c + k] = x(base + ((u32)k << s.hb) + conv_col(s, t + (u32)c * cols, k));
#pragma unroll
        for (int c = 0; c < 4; c++) {
            E *y = v + 4 * c;
            if (!INV) { y[0] ^= y[2]; y[1] ^= y[3]; }
            y[0] ^= y[1];
            y[2] ^= y[3];
            if (INV) { y[0] ^= y[2]; y[1] ^= y[3]; }
        }
#pragma unroll
        for (int c = 0; c < 4; c++)
#pragma unroll
            for (int k = 0; k < 3; k++)   // row 3 keeps its value
                x(base + ((u32)k << s.hb) + conv_col(s, t + (u32)c * cols, k)) = v[4 * c + k];
    } else {
        const u32 rho = t - cols;
#pragma unroll
        for (int i = 0; i < 16; i++)
            v[i] = x(base + ((u32)(i >> 2) << s.hb) + conv_edge(s, i >> 2, (u32)(i & 3), rho));
        if (!INV) { conv_regs<2, 1, 16, INV>(v); conv_regs<2, 0, 16, INV>(v); }
        else { conv_regs<2, 0, 16, INV>(v); conv_regs<2, 1, 16, INV>(v); }
#pragma unroll
        for (int i = 0; i < 16; i++)
            x(base + ((u32)(i >> 2) << s.hb) + conv_edge(s, i >> 2, (u32)(i & 3), rho)) = v[i];
    }
}
// all of the conversion of nb bits (2, 3 or 4) whose top is local bit
// pos + 3, the registers being the local bits pos .. pos + 3
template <bool INV, class E, class X>
GF2T_HD void conv_tile_nibble(X &&x, u32 q, int pos, int nb) {
    const u32 base = spread_rows(q, 0, pos, 4);
    E v[16];
#pragma unroll
    for (int r = 0; r < 16; r++) v[r] = x(base + ((u32)r << pos));
    if (nb == 4) {
        conv_nibble<0, 16, INV>(v);
    } else if (nb == 3) {
        if (!INV) { conv_regs<2, 1, 16, INV>(v); conv_regs<1, 1, 16, INV>(v); }
        else { conv_regs<1, 1, 16, INV>(v); conv_regs<2, 1, 16, INV>(v); }
    } else {
        conv_regs<1, 2, 16, INV>(v);
    }
#pragma unroll
    for (int r = 0; r < 16; r++) x(base + ((u32)r << pos)) = v[r];
}
// a stage of a tile: K = 1, 2 steps s, or K = 0: nibble at s.ub, s.hb bits
template <bool INV, class E, class X>
GF2T_HD void conv_tile_stage(X &&x, u32 q, u32 threads, const ConvStep &s) {
    if (s.K == 2) conv_tile2<INV, E>(x, q, s);
    else if (s.K == 1) conv_tile1<INV, E>(x, q, threads, s);
    else conv_tile_nibble<INV, E>(x, q, s.ub, s.hb);
}
// a tile: the local bits [0, c) are memory's, [c, c + w) the index bits
// [a, a + w)
constexpr int CONV_MAX_STAGES = 12;
struct ConvTile {
    int c, a, w, n;
    ConvStep st[CONV_MAX_STAGES];   // forward order
};
GF2T_HD u64 tile_base(const ConvTile &t, u32 blk) {
    const int nlo = t.a - t.c;
    return ((u64)(blk & ((1u << nlo) - 1)) << t.c) | ((u64)(blk >> nlo) << (t.a + t.w));
}
GF2T_HD u64 tile_mem(const ConvTile &t, u32 l) {
    return (l & ((1u << t.c) - 1)) + ((u64)(l >> t.c) << t.a);
}

// ------------------------------------------------------------- host side
#include <vector>
namespace cantor_host {
// the plan of a basis conversion of 2^k coefficients, in forward order
struct ConvPlan {
    std::vector<ConvStep> steps;    // before the tiles
    std::vector<ConvTile> tiles;
    bool empty() const { return steps.empty() && tiles.empty(); }
    size_t launches() const { return steps.size() + tiles.size(); }
};
// steps e = n - 1 .. 0 of the expansion in powers of s_h, at index bit off,
// at most `most` to a group, the groups counted from the bottom
template <class F>
inline void conv_steps(int off, int h, int n, int most, F &&put) {
    for (int lo = (n - 1) / most * most; lo >= 0; lo -= most)
        put(ConvStep{n - lo < most ? n - lo : most, h + lo + off, lo + off});
}
// stages of the bits [pos, pos + k), k <= 8, of a tile of 2^T: the top one
// of a k that is no multiple of four has the tile's top bits
inline void tile_group(ConvTile &t, int pos, int k) {
    auto put = [&](const ConvStep &s) { t.st[t.n++] = s; };
    if (k <= 1) return;
    if (k <= 4) {
        put(ConvStep{0, k, pos + k - 4 < 0 ? 0 : pos + k - 4});
        return;
    }
    conv_steps(pos, 4, k - 4, 2, put);
    tile_group(t, pos + 4, k - 4);
    tile_group(t, pos, 4);
}
// one_tile: the largest k converted in a single tile; tile_bits: of the
// others' tiles.  Tiles have at least 16 coefficients (k < 4: zeros above).
inline ConvPlan conv_plan(int k, int one_tile, int tile_bits) {
    ConvPlan P;
    if (k <= 1) return P;
    auto step = [&](const ConvStep &s) { P.steps.push_back(s); };
    if (k <= one_tile) {
        ConvTile t{k < 4 ? 4 : k, k < 4 ? 4 : k, 0, 0, {}};
        auto put = [&](const ConvStep &s) { t.st[t.n++] = s; };
        if (k > 8) {
            conv_steps(0, 8, k - 8, 2, put);
            tile_group(t, 8, k - 8);
        }
        tile_group(t, 0, k > 8 ? 8 : k < 4 ? 4 : k);
        P.tiles.push_back(t);
        return P;
    }
    const int low = k < 16 ? k : 16;
    if (k > 16) {
        conv_steps(0, 16, k - 16, 4, step);
        if (k > 24) conv_steps(16, 8, k - 24, 4, step);
    }
    // the low part's expansion in powers of s_8: its steps 3..0 run in the
    // contiguous tiles
    const int n8 = low - 8;
    if (n8 > 4) P.steps.push_back(ConvStep{n8 - 4, 12, 4});
    ConvTile lo{12, 12, 0, 0, {}};
    conv_steps(0, 8, n8 < 4 ? n8 : 4, 2, [&](const ConvStep &s) { lo.st[lo.n++] = s; });
    tile_group(lo, 0, 8);
    P.tiles.push_back(lo);
    for (int off = 8; off < k; off += 8) {
        const int w = k - off < 8 ? k - off : 8;
        if (w < 2) break;
        int c = tile_bits - w;
        if (c > off) c = off;
        ConvTile g{c, off, w, 0, {}};
        tile_group(g, c, w);
        P.tiles.push_back(g);
    }
    return P;
}
// butterfly passes of a 2^m-point transform above its low eight levels,
// top window first (forward order); tiles of at most 2^tile units
inline std::vector<BfPass> bf_passes(int m, int tile) {
    std::vector<BfPass> v;
    for (int top = m; top > 8;) {
        const int w = top - 8 < 8 ? top - 8 : 8, a = top - w;
        int tb = tile;
        if (tb > w + a - 1) tb = w + a - 1;
        const int least = w + 2;   // covers the RB ceil(w / RB) bits the stages need
        if (tb < least) tb = least;
        v.push_back(BfPass{m, a, w, tb});
        top = a;
    }
    return v;
}
constexpr int FFT_MAX_M = 27;
// a transform's size for that many coefficients
inline int fft_m_for(u64 nchunks_total) {
    int m = 1;
    while (((u64)1 << m) < nchunks_total) m++;
    return m;
}
// Wrapped products.  A product whose N = ca + cb - 1 chunk coefficients lie just above a
// power of two, 2^mp < N <= 2^mp + 2^mp/4, runs on 2^mp-point transforms
// instead of 2^(mp+1), plus a product at most half that size.  The 2^mp
// points are the span of the first mp Cantor basis elements, whose
// vanishing polynomial is
//     V(X) = sum over k with bits(k) inside bits(mp) of X^(2^k)
// (V_{i+1} = V_i^2 + V_i, since V_i(b_i) = 1 for the Cantor basis; the
// binomial coefficients mod 2 follow Lucas).  So pointwise products and
// the inverse give C mod V.  The e = N - 2^mp top coefficients
// C_high = C div X^(2^mp) come from the product of the top e chunks of
// each operand (pairs i + j >= 2^mp only involve those), a 2^ms-point
// product.  V's next term below X^(2^mp) is at most X^(2^(mp-1)), and
// deg C_high < e <= 2^(mp-2), so C div V = C_high and
//     C = (C mod V) + C_high * (V - X^(2^mp)) + C_high * X^(2^mp):
// C_high is XORed into the low coefficients at each offset 2^k, k a
// proper bit-subset of mp, and forms the coefficients from 2^mp up.
struct Wrap {
    bool on = false;
    int mp = 0, ms = 0;
    u64 e = 0;
};
// Wrapping pays where the 2^mp points it saves (of all products of a batch
// together) take longer than the top product: its chain of launches, as
// long as WRAP_CHAIN points, and a fourth more than its own points, as a
// smaller transform uses the chip less.  Wrapped and not, 2^20 coefficients
// and a 32nd more take 265 and 268 us, a 16th more 284 and 268; 2^21 and an
// eighth 439 and 419; 2^22 and an eighth 645 and 721, and a quarter 743 and
// 717; 2^23 and a 64th 928 and 1352.
constexpr u64 WRAP_CHAIN = 900000;
inline Wrap wrap_for(u64 ca, u64 cb, u64 nbatch = 1) {
    Wrap w;
    const u64 N = ca + cb - 1;
    const int m = fft_m_for(N);
    if (m < 12 || m - 1 > FFT_MAX_M) return w;
    const int mp = m - 1;
    const u64 n = (u64)1 << mp;
    if (N <= n) return w;
    const u64 e = N - n;
    if (e > n / 4 || ca > n || cb > n || e >= ca || e >= cb) return w;
    const int ms = fft_m_for(2 * e - 1);
    if (nbatch * n < WRAP_CHAIN + 5 * (nbatch << ms) / 4) return w;
    w.on = true;
    w.mp = mp;
    w.e = e;
    w.ms = ms;
    return w;
}
// The transforms of a launch are the rows of its grid, which has at most
// 65535, and a product has two of them: the pairs of one chain of launches.
constexpr unsigned MAX_PAIRS = 32767;
// the pairs j of a batch by their transform size m[j] (0: no transform), the
// largest first, at most MAX_PAIRS to a group
struct SizeGroup {
    int m;
    std::vector<int> pairs;
};
inline std::vector<SizeGroup> size_groups(const std::vector<int> &m) {
    std::vector<SizeGroup> v;
    for (int k = 31; k >= 1; k--) {
        const size_t first = v.size();
        for (int j = 0; j < (int)m.size(); j++) {
            if (m[j] != k) continue;
            if (v.size() == first || v.back().pairs.size() == MAX_PAIRS) v.push_back(SizeGroup{k, {}});
            v.back().pairs.push_back(j);
        }
    }
    return v;
}
// Of a batch of pairs of ca[j] and cb[j] chunks and transform sizes m[j],
// those formed without transforms, all in one launch: whole sizes, the
// smallest first, while their chunk pairs are at most DIRECT_PAIRS together.
// A size by transforms is a chain of launches of its own, 40 to 60 us however
// few its pairs; 2^25 chunk pairs take about 50 us (eight pairs of 2^15 ..
// 2^22 bits: 464 us, 586 all by transforms; one pair of 132,049 bits: 46 and
// 91), and where there are more the transforms' fewer operations count (64
// pairs of 44,497 bits: 80 us by transforms).
constexpr size_t DIRECT_PAIRS = (size_t)1 << 25;
constexpr int DIRECT_MAX_M = 15;   // of at most 2^15 + 1 chunks
inline std::vector<char> direct_pairs(const std::vector<int> &m, const std::vector<u64> &ca,
                                      const std::vector<u64> &cb) {
    u64 work[DIRECT_MAX_M + 1] = {}, all = 0;
    for (size_t j = 0; j < m.size(); j++)
        if (m[j] && m[j] <= DIRECT_MAX_M) work[m[j]] += ca[j] * cb[j];
    int most = 0;
    while (most < DIRECT_MAX_M && all + work[most + 1] <= DIRECT_PAIRS) all += work[++most];
    std::vector<char> v(m.size());
    for (size_t j = 0; j < m.size(); j++) v[j] = m[j] && m[j] <= most;
    return v;
}
// the subfield class of a window's twiddles: 8, 16 or 32
inline int bf_class(const BfPass &P) {
    const int bits = P.m - 1 - P.a;
    return bits <= 7 ? 8 : bits <= 15 ? 16 : 32;
}

// the tables, from the Cantor basis b[0..63]
inline u64 pow_of(u64 a, int n) {
    u64 r = 1;
    for (int i = 0; i < n; i++) r = gf64_mul(r, a);
    return r;
}
// rows of the inverse of the map bit i -> col[i] (n columns of n bits)
inline bool invert(const u64 *col, int n, u64 *icol) {
    std::vector<u64> a(col, col + n), e(n);
    for (int i = 0; i < n; i++) e[i] = 1ULL << i;
    for (int bit = 0; bit < n; bit++) {
        int p = -1;
        for (int i = bit; i < n; i++)
            if ((a[i] >> bit) & 1) { p = i; break; }
        if (p < 0) return false;
        std::swap(a[p], a[bit]);
        std::swap(e[p], e[bit]);
        for (int i = 0; i < n; i++)
            if (i != bit && ((a[i] >> bit) & 1)) { a[i] ^= a[bit]; e[i] ^= e[bit]; }
    }
    // a[i] = 1 << i now: icol[i] is the combination of columns that gives bit i
    for (int i = 0; i < n; i++) icol[i] = e[i];
    return true;
}
inline u64 apply(const u64 *col, u64 v) {
    u64 r = 0;
    for (int i = 0; v; i++, v >>= 1)
        if (v & 1) r ^= col[i];
    return r;
}
inline bool build_tables(const u64 *b, FftTables &T) {
    // tower halfword p, byte j2: bits 16 p + 8 j2 + i
    u64 tow[64], inv[64];
    for (int p = 0; p < 4; p++)
        for (int j = 0; j < 2; j++)
            for (int i = 0; i < 8; i++) {
                u64 v = b[i];
                if (p & 1) v = gf64_mul(v, b[8]);
                if (p & 2) v = gf64_mul(v, b[16]);
                if (j) v = gf64_mul(v, b[32]);
                tow[16 * p + 8 * j + i] = v;
            }
    if (!invert(tow, 64, inv)) return false;
    for (int k = 0; k < 8; k++)
        for (int v = 0; v < 256; v++) {
            T.emb[k][v] = apply(inv, (u64)v << (8 * k));
            T.une[k][v] = apply(tow, (u64)v << (8 * k));
        }
    // products in GF(2^8), bytes in the basis b[0..7]
    auto mul8 = [&](u32 x, u32 y) -> u32 {
        return (u32)apply(inv, gf64_mul(apply(tow, x), apply(tow, y)));
    };
    u32 prod[8][8];
    for (int i = 0; i < 8; i++)
        for (int j = 0; j < 8; j++) {
            prod[i][j] = mul8(1u << i, 1u << j);
            if (prod[i][j] > 255) return false;   // span(b[0..7]) is not a subfield
        }
    auto m8 = [&](u32 x, u32 y) {
        u32 r = 0;
        for (int i = 0; i < 8; i++)
            for (int j = 0; j < 8; j++)
                if (((x >> i) & 1) && ((y >> j) & 1)) r ^= prod[i][j];
        return r;
    };
    for (u32 v = 0; v < 256; v++) {
        u32 a[2] = {0, 0}, m[2] = {0, 0}, c = 0;
        for (u32 x = 0; x < 8; x++) {
            a[x >> 2] |= m8(v, x) << (8 * (x & 3));
            m[x >> 2] |= m8(v, x << 3) << (8 * (x & 3));
            if (x < 4) c |= m8(v, x << 6) << (8 * x);
        }
        T.mulA[v][0] = a[0]; T.mulA[v][1] = a[1]; T.mulA[v][2] = m[0]; T.mulA[v][3] = m[1];
        T.mulB[v] = c;
    }
    // twiddles: tower bytes of b[j + 1], which must lie in GF(2^32)
    const u32 c3 = (u32)apply(inv, b[7]);
    auto ent = [&](u64 w) {
        const u64 t = apply(inv, w);
        const u32 a0 = (u32)t & 255, a1 = (u32)(t >> 16) & 255, b0 = (u32)(t >> 32) & 255,
                  b1 = (u32)(t >> 48) & 255;
        const u64 wb = apply(tow, (u64)b0 | ((u64)b1 << 16));
        const u64 tq = apply(inv, gf64_mul(b[15], wb));   // c4 Wb
        const u32 q0 = (u32)tq & 255, q1 = (u32)(tq >> 16) & 255;
        const u32 r0 = a0 ^ b0, r1 = a1 ^ b1;
        const u32 p[3] = {a0, m8(c3, a1), a0 ^ a1}, q[3] = {q0, m8(c3, q1), q0 ^ q1},
                  r[3] = {r0, m8(c3, r1), r0 ^ r1};
        auto two = [](u32 x, u32 y) { return (x << 4) | (y << 20); };
        return TwEnt{two(p[0], p[2]), two(r[0], r[2]), two(p[1], r[1]), two(q[0], q[1]),
                     q[2] << 4, {}};
    };
    TwEnt bit[32] = {};
    for (int j = 0; j + 1 < 32; j++) {
        if (apply(inv, b[j + 1]) & 0xFF00FF00FF00FF00ULL) return false;
        bit[j] = ent(b[j + 1]);
    }
    for (int k = 0; k < 4; k++)
        for (int v = 0; v < 256; v++) {
            TwEnt e{};
            for (int j = 0; j < 8; j++)
                if ((v >> j) & 1) e = tw_xor(e, bit[8 * k + j]);
            T.tw[k][v] = e;
        }
    // GF(2^32): tower bytes (p = 0..3, u5^0) <-> powers of rho
    u64 rp[32], rt[32], ri[32];
    for (int i = 0; i < 32; i++) {
        rp[i] = pow_of(FFT_RHO, i);
        const u64 t = apply(inv, rp[i]);
        if (t & 0xFF00FF00FF00FF00ULL) return false;
        rt[i] = (t & 255) | ((t >> 8) & 0xFF00) | ((t >> 16) & 0xFF0000) | ((t >> 24) & 0xFF000000u);
    }
    if (!invert(rt, 32, ri)) return false;
    auto t32 = [&](u32 packed) {   // four tower bytes -> field element
        u64 t = 0;
        for (int p = 0; p < 4; p++) t |= (u64)((packed >> (8 * p)) & 255) << (16 * p);
        return apply(tow, t);
    };
    auto packed = [&](u64 f) {
        const u64 t = apply(inv, f);
        return (u32)((t & 255) | ((t >> 8) & 0xFF00) | ((t >> 16) & 0xFF0000) |
                     ((t >> 24) & 0xFF000000u));
    };
    for (int k = 0; k < 4; k++)
        for (u32 v = 0; v < 256; v++) {
            T.d32[k][v] = (u32)apply(ri, (u64)v << (8 * k));
            T.d5[k][v] = (u32)apply(ri, packed(gf64_mul(b[31], t32(v << (8 * k)))));
            T.b32[k][v] = (u32)apply(rt, (u64)v << (8 * k));
        }
    return true;
}
}  // namespace cantor_host
