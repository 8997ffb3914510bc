// class_log.hpp -- logarithms of GF(2^d), d <= 32, by conjugacy class,
// written once for device and host (the sieve's kernels include it, and a
// host build of the same functions is checked against plain discrete
// logarithms on the CPU, tests/test_class_log.py).
//
// With theta normal, w(y) = (Tr(theta^(2^i) y))_i, i < d, is a one-to-one
// linear image of the field in which squaring is a rotation by one bit, so
// the least rotation of w(y) names y's class {y^(2^k)} and the rotation
// that reaches it gives k.  Logarithms mod M = 2^d - 1 double with y
// squared, which is a rotation of the d-bit logarithm.  So one logarithm
// per class is enough: log y = rotr(T[least rotation of w(y)], k).  For
// classes of full length (y in no proper subfield) the least rotation is
// odd and below 2^(d-1): T has 2^(d-2) words, of which one in d/4 is used.
#pragma once
#include "gf2t_arith.hpp"
#include <algorithm>
#include <vector>

// a d-bit word repeated without end, its first 64 bits (first bit on top)
GF2T_HD u64 periodic64(u32 w, int d) {
    u64 a = (u64)w << (64 - d);
    for (int s = d; s < 64; s *= 2) a |= a >> s;
    return a;
}
// the 32 bits from bit k on, 1 <= k <= 31.  Two windows of one periodic
// word compare as the rotations they begin with, so no window is masked.
GF2T_HD u32 period_window(u64 a, int k) { return alignbit((u32)(a >> 32), (u32)a, (u32)(32 - k)); }

// ap: the rotations d/p, p prime, one byte each (0: none)
GF2T_HD u32 aperiodic_rotations(int d) {
    u32 ap = 0;
    int at = 0, n = d;
    for (int p = 2; p <= n; p++)
        if (n % p == 0) {
            ap |= (u32)(d / p) << at;
            at += 8;
            while (n % p == 0) n /= p;
        }
    return ap;
}
// j (d bits) is below all its other rotations: none is smaller (rotations
// past d repeat), and none of d/p equals it.  1.5 operations a rotation.
GF2T_HD bool lyndon_word(u32 j, int d, u32 ap) {
    const u64 a = periodic64(j, d);
    const u32 w0 = (u32)(a >> 32);
    u32 m = w0;
#pragma unroll
    for (int k = 1; k < 32; k++) {
        const u32 w = period_window(a, k);
        m = w < m ? w : m;
    }
    bool ok = m == w0;
    for (u32 x = ap; x; x >>= 8) ok = ok && period_window(a, (int)(x & 255)) != w0;
    return ok;
}
// w, the first n bits of a word, may begin a Lyndon word: no part of it
// from bit k on is below w's own beginning
GF2T_HD bool lyndon_prefix(u32 w, int n) {
    bool ok = true;
    for (int k = 1; k < n; k++) ok = ok && (w & ((1u << (n - k)) - 1)) >= (w >> k);
    return ok;
}
// the least rotation of a periodic word (its first 32 bits), and which
GF2T_HD u32 least_rotation(u64 a, int &k) {
    u32 m = (u32)(a >> 32);
    k = 0;
#pragma unroll
    for (int i = 1; i < 32; i++) {
        const u32 w = period_window(a, i);
        k = w < m ? i : k;
        m = w < m ? w : m;
    }
    return m;
}
// x * 2^k mod 2^d - 1 as d-bit words (0 <= k <= d <= 32)
GF2T_HD u32 rotl_d(u32 x, int k, int d) {
    const u64 t = (u64)x << k;
    return (u32)(t & (((u64)1 << d) - 1)) | (u32)(t >> d);
}
// T's index of the class whose least rotation begins with m
GF2T_HD u32 class_index(u32 m, int d) { return (m >> (33 - d)) & ((1u << (d - 2)) - 1); }

// Linear maps by bytes.  CL_NORM: w of an unreduced product (8 bytes);
// CL_RED: the reduction of its bits from d on (4 bytes); CL_DUAL: the
// vector (Tr(x^i b))_i of b (4 bytes), so Tr(a b) = parity(a & dual(b)).
constexpr u32 CL_NORM = 0, CL_RED = 2048, CL_DUAL = 3072, CL_MAP = 4096;
template <class Table>
GF2T_HD u32 map4(const Table &t, u32 x) {
    return t[x & 255] ^ t[256 + ((x >> 8) & 255)] ^ t[512 + ((x >> 16) & 255)] ^ t[768 + (x >> 24)];
}
template <class Table>
GF2T_HD u32 map8(const Table &t, u64 x) {
    return map4(t, (u32)x) ^ map4(t + 1024, (u32)(x >> 32));
}
GF2T_HD u32 red_product(u64 t, const u32 *red, int d) {
    return (u32)(t & (((u64)1 << d) - 1)) ^ map4(red, (u32)(t >> d));
}
// Tr(beta^k) for k < 64, bit k: beta^(8m + i) by its factors beta^(8m) and
// beta^i, the latter by their duals -- 6 products and 7 squares where 64
// powers took 64 products with a bit-serial reduction
GF2T_HD u64 trace_sequence(u32 beta, const u32 *red, const u32 *dual, int d) {
    auto mul = [&](u32 a, u32 b) { return red_product(clmul32(a, b), red, d); };
    auto sqr = [&](u32 a) { return red_product(spread32p(a), red, d); };
    u32 D[8];
    const u32 b2 = sqr(beta), b3 = mul(b2, beta), b4 = sqr(b2), b6 = sqr(b3);
    D[0] = map4(dual, 1u);
    D[1] = map4(dual, beta);
    D[2] = map4(dual, b2);
    D[3] = map4(dual, b3);
    D[4] = map4(dual, b4);
    D[5] = map4(dual, mul(b4, beta));
    D[6] = map4(dual, b6);
    D[7] = map4(dual, mul(b6, beta));
    u32 G[8];
    G[0] = 1;
    G[1] = sqr(b4);
    G[2] = sqr(G[1]);
    G[3] = mul(G[2], G[1]);
    G[4] = sqr(G[2]);
    G[5] = mul(G[4], G[1]);
    G[6] = sqr(G[3]);
    G[7] = mul(G[6], G[1]);
    u32 half[2] = {0, 0};
#pragma unroll
    for (int m = 0; m < 8; m++)
#pragma unroll
        for (int i = 0; i < 8; i++)
            half[m >> 2] |= (u32)(__builtin_popcount(G[m] & D[i]) & 1) << (8 * (m & 3) + i);
    return ((u64)half[1] << 32) | half[0];
}

// ---- progressions s j == v (mod M): s == v / j (mod n), n = M / gcd(j, M)
// p^e || M; inv = 1/p mod 2^32 and lim = floor((2^32 - 1) / p): x is a
// multiple of p iff x * inv mod 2^32 (then x / p) is at most lim
struct SievePrime {
    u32 p, inv, lim, e;
};
#if defined(__HIP_DEVICE_COMPILE__)
#define GF2T_ANY(x) __any(x)
#else
#define GF2T_ANY(x) (x)
#endif
// For N classes: v -> v / g for g = gcd(j, M), n = M / g; bit i of the
// result is cleared if g does not divide v[i] (no s).  unit: an integer
// below M, prime to it, that is j / g modulo n -- j / g + n t with t the
// primes that are in neither n nor j / g -- so its inverse modulo M serves
// modulo n, and the inverses of many classes are taken together.  A prime
// that divides no lane's j costs one multiplication.
template <int N>
GF2T_HD u32 progressions(u32 (&v)[N], const u32 (&j)[N], u32 (&n)[N], u32 (&unit)[N], u32 M,
                         const SievePrime *pr, int np) {
    u32 ok = ~0u, t[N];
#pragma unroll
    for (int c = 0; c < N; c++) {
        unit[c] = j[c];
        n[c] = M;
        t[c] = 1;
    }
    for (int i = 0; i < np; i++) {
        const SievePrime q = pr[i];
#pragma unroll
        for (int c = 0; c < N; c++) {
            bool all = true;
            for (u32 k = 0; k < q.e; k++) {
                const u32 x = unit[c] * q.inv, y = v[c] * q.inv;
                all = all && x <= q.lim;
                if (!GF2T_ANY(all)) break;
                if (all && y > q.lim) ok &= ~(1u << c);
                unit[c] = all ? x : unit[c];
                v[c] = all ? y : v[c];
                n[c] = all ? n[c] * q.inv : n[c];
            }
            if (GF2T_ANY(all) && all && unit[c] * q.inv > q.lim) t[c] *= q.p;
        }
    }
#pragma unroll
    for (int c = 0; c < N; c++) {
        const u64 x = (u64)n[c] * t[c] + unit[c];
        unit[c] = (u32)(x >= M ? x - M : x);
    }
    return ok;
}
// a b mod M = 2^d - 1, for a, b < M
GF2T_HD u32 mulmod_mersenne(u32 a, u32 b, int d, u32 M) {
    const u64 t = (u64)a * b;
    u64 x = (t & M) + (t >> d);
    return (u32)(x >= M ? x - M : x);
}

// ------------------------------------------------------- host: the tables
namespace class_host {
// the byte maps of GF(2^d); false if a trace does not lie in GF(2)
inline bool class_maps(u64 q, int d, u32 *map) {
    auto trace = [&](u64 y) {
        u64 acc = y;
        for (int k = 1; k < d; k++) { y = fmul64(y, y, q, d); acc ^= y; }
        return acc;
    };
    std::vector<u64> pw(2 * 64);   // x^b
    pw[0] = 1;
    for (int b = 1; b < 128; b++) pw[b] = (pw[b - 1] << 1) ^ (((pw[b - 1] >> (d - 1)) & 1) ? q : 0);
    u64 tmask = 0;   // bit i: Tr(x^i)
    for (int i = 0; i < d; i++) {
        const u64 t = trace(pw[i]);
        if (t > 1) return false;
        tmask |= t << i;
    }
    auto tr = [&](u64 y) { return (u32)(__builtin_popcountll(y & tmask) & 1); };
    auto dual = [&](u64 b) {   // bit i: Tr(x^i b)
        u32 x = 0;
        for (int i = 0; i < d; i++)
            if ((b >> i) & 1)
                for (int k = 0; k < d; k++) x ^= tr(pw[i + k]) << k;
        return x;
    };
    // theta: a normal element, of trace 1 -- at least one element in ten is
    // normal at these d, so scattered ones are tried; row i of w: the dual
    // of theta^(2^i)
    std::vector<u32> row(d);
    int rank = 0;
    for (u64 n = 1; rank < d; n++) {
        u64 t = (n * 0x9E3779B97F4A7C15ULL) >> (64 - d);
        if (!tr(t)) continue;
        for (int i = 0; i < d; i++) {
            row[i] = dual(t);
            t = fmul64(t, t, q, d);
        }
        std::vector<u32> m(row);
        for (rank = 0; rank < d; rank++) {
            int k = rank;
            while (k < d && !((m[k] >> rank) & 1)) k++;
            if (k == d) break;
            std::swap(m[k], m[rank]);
            for (int i = rank + 1; i < d; i++)
                if ((m[i] >> rank) & 1) m[i] ^= m[rank];
        }
    }
    auto bytes = [&](u32 *out, int nb, auto image) {   // image(b): of bit b
        for (int j = 0; j < nb; j++)
            for (u32 v = 0; v < 256; v++) {
                u32 x = 0;
                for (int k = 0; k < 8; k++)
                    if ((v >> k) & 1) x ^= image(8 * j + k);
                out[256 * j + v] = x;
            }
    };
    bytes(map + CL_NORM, 8, [&](int b) {
        u32 x = 0;
        for (int i = 0; i < d; i++) x |= (u32)(__builtin_popcountll(pw[b] & row[i]) & 1) << i;
        return x;
    });
    bytes(map + CL_RED, 4, [&](int b) { return (u32)pw[d + b]; });
    bytes(map + CL_DUAL, 4, [&](int b) { return b < d ? dual((u64)1 << b) : 0; });
    return true;
}
inline SievePrime sieve_prime(u32 p, u64 M) {
    u32 inv = p, e = 0;
    for (int k = 0; k < 5; k++) inv *= 2 - p * inv;   // 1/p mod 2^32
    for (u64 m = M; m % p == 0; m /= p) e++;
    return SievePrime{p, inv, 0xFFFFFFFFu / p, e};
}
}  // namespace class_host
