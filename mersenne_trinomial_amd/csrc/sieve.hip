// sieve.hip -- (a) Zech-log coarse sieve on gfx950.
//
// For each degree d: GF(2^d) = GF(2)[x]/q with q primitive, so g = x has
// order M = 2^d - 1.  An irreducible P of degree d with root beta = g^j
// divides x^r + x^s + 1 iff beta^r + beta^s = 1, i.e. j*s == Z(u) (mod M)
// with u = j*r mod M and Z the Zech logarithm Z(u) = log(g^u + 1): an
// arithmetic progression in s of modulus n = M / gcd(j, M).  One root per
// conjugacy class suffices: the class representative is the j that is
// strictly smaller than all its other rotations j*2^i mod M (a binary
// Lyndon word of length d), which also excludes every element of a
// proper subfield.  Each progression is marked into best[s] with an
// atomic min of (d << 48) | mask, i.e. smallest degree, then numerically
// least mask (reference: src/sieve_ref.cpp:1-30, src/coarse_sieve.cu:
// 237-299).
//
// Degrees up to 32 (class_log.hpp), on the device:
//   k_classes     the class representatives (Lyndon words) as a dense list,
//                 only below prefixes that can begin one
//   k_class_log   one logarithm per class: T[least rotation of w(g^j)], a
//                 table of 2^(d-2) words of which one in d/4 is written
//   k_zech        per class: Zech logarithm (one random gather of T) and
//                 the progression; classes whose progression reaches s <=
//                 smax are ballot-compacted into a queue (about 1.6% of
//                 them at d = 32 for smax = 68,139,920)
//   k_mark        per queued class: minimal polynomial by Berlekamp-Massey
//                 on Tr(beta^k), then the marks (inline up to 1024, longer
//                 progressions to k_mark_heavy); degrees up to 20 whose
//                 period M is at most smax mark one period instead, and
//   k_sweep       takes every s through the periods once, lowest degree
//                 first
// A table of all 2^d logarithms (16 GiB at d = 32) took three radix
// partition passes over 8-byte entries, 94 of 134 ms at degrees 2..32 over
// 68,139,920 s; one logarithm per class needs none of them.  Several small
// degrees run in one launch (blockIdx.y), and nothing waits for the host
// until all degrees are done.
#include "gf2t_internal.hpp"
#include "class_log.hpp"
#include "../../include/gf2t.h"
#include <vector>
#include <algorithm>
#include <cstring>
#include <mutex>

namespace {

constexpr u64 INLINE_MARKS = 1024;
constexpr u32 HEAVY_CAP = 1u << 22;

struct Heavy {
    u64 s_first, n, key;
};

// ------------------------------------------------------------ host field
u64 hclmul(u64 a, u64 b, u64 &hi) {
    u64 lo = 0;
    hi = 0;
    for (int i = 0; i < 64; i++)
        if ((b >> i) & 1) {
            lo ^= a << i;
            if (i) hi ^= a >> (64 - i);
        }
    return lo;
}
u64 hmulmod(u64 a, u64 b, u64 q, int d) {
    u64 hi, lo = hclmul(a, b, hi);
    for (int bit = 2 * d - 2; bit >= d; bit--) {
        u64 have = bit >= 64 ? (hi >> (bit - 64)) & 1 : (lo >> bit) & 1;
        if (!have) continue;
        int sh = bit - d;
        lo ^= q << sh;
        if (sh) hi ^= q >> (64 - sh);
    }
    return lo;
}
u64 hpgcd(u64 a, u64 b) {
    while (b) {
        int db = 63 - __builtin_clzll(b);
        while (a && 63 - __builtin_clzll(a) >= db) a ^= b << ((63 - __builtin_clzll(a)) - db);
        std::swap(a, b);
    }
    return a;
}
int hprimes(u64 m, u64 *ps) {
    int n = 0;
    for (u64 p = 2; p * p <= m; p += (p == 2 ? 1 : 2))
        if (m % p == 0) { ps[n++] = p; while (m % p == 0) m /= p; }
    if (m > 1) ps[n++] = m;
    return n;
}
// Rabin: x^(2^d) == x and gcd(x^(2^(d/p)) - x, q) = 1 for primes p | d
bool hirreducible(u64 q, int d) {
    u64 chain[65];
    u64 t = 2;
    chain[0] = t;
    for (int i = 1; i <= d; i++) { t = hmulmod(t, t, q, d); chain[i] = t; }
    if (chain[d] != 2) return false;
    u64 ps[16];
    int np = hprimes((u64)d, ps);
    for (int i = 0; i < np; i++)
        if (hpgcd(q, chain[d / ps[i]] ^ 2) != 1) return false;
    return true;
}
u64 hpow(u64 b, u64 e, u64 q, int d) {
    u64 r = 1;
    while (e) {
        if (e & 1) r = hmulmod(r, b, q, d);
        b = hmulmod(b, b, q, d);
        e >>= 1;
    }
    return r;
}
u64 primitive_poly(int d) {
    u64 M = ((u64)1 << d) - 1, ps[16];
    int np = hprimes(M, ps);
    for (u64 q = ((u64)1 << d) | 1; q < ((u64)2 << d); q += 2) {
        if (!hirreducible(q, d)) continue;
        bool prim = true;
        for (int i = 0; i < np && prim; i++)
            if (hpow(2, M / ps[i], q, d) == 1) prim = false;
        if (prim) return q;
    }
    return 0;
}
u64 gcd_host(u64 a, u64 b) {
    while (b) { u64 t = a % b; a = b; b = t; }
    return a;
}
int64_t mobius(u64 n) {
    int64_t mu = 1;
    for (u64 p = 2; p * p <= n; p++) {
        if (n % p) continue;
        n /= p;
        if (n % p == 0) return 0;
        mu = -mu;
    }
    if (n > 1) mu = -mu;
    return mu;
}
u64 irreducible_count(int d) {
    int64_t acc = 0;
    for (int k = 1; k <= d; k++)
        if (d % k == 0) acc += mobius((u64)k) * ((int64_t)1 << (d / k));
    return (u64)(acc / d);
}

// Per-degree host constants, computed once per process: the smallest
// primitive modulus q, the antilog tables g^k and g^(65536 k) (k < 2^16),
// the byte maps of class_log.hpp, and the primes of M.  The g^(65536 k)
// table steps by a fixed multiplier, which is linear over GF(2): four
// 256-entry byte tables make each step four lookups.
constexpr size_t DEG_TAB = 2 * 65536 + CL_MAP;   // words of a degree's tables
struct DegHost {
    bool ready = false, trace_ok = false;
    u64 q = 0;
    std::vector<u32> tab;   // g^k, g^(65536 k), byte maps
    std::vector<SievePrime> primes;
};
std::mutex g_deg_mu;
DegHost g_deg[33];

const DegHost &deg_host(int d) {
    std::lock_guard<std::mutex> lk(g_deg_mu);
    DegHost &H = g_deg[d];
    if (H.ready) return H;
    H.q = primitive_poly(d);
    H.tab.assign(DEG_TAB, 0);
    if (H.q) {
        const u64 q = H.q;
        u32 *lo = H.tab.data(), *hi = lo + 65536;
        u64 a = 1;
        for (u64 k = 0; k < 65536; k++) {
            lo[k] = (u32)a;
            a <<= 1;
            if ((a >> d) & 1) a ^= q;
        }
        const u64 g16 = a;   // g^65536
        u32 T[4][256];
        for (int j = 0; j < 4; j++)
            for (u64 v = 0; v < 256; v++) {
                u64 e = v << (8 * j);
                T[j][v] = (e >> d) ? 0u : (u32)hmulmod(e, g16, q, d);
            }
        u32 b = 1;
        for (u64 k = 0; k < 65536; k++) {
            hi[k] = b;
            b = T[0][b & 255] ^ T[1][(b >> 8) & 255] ^ T[2][(b >> 16) & 255] ^ T[3][b >> 24];
        }
        H.trace_ok = class_host::class_maps(q, d, hi + 65536);
        const u64 M = ((u64)1 << d) - 1;
        u64 ps[16];
        const int np = hprimes(M, ps);
        for (int i = 0; i < np; i++) H.primes.push_back(class_host::sieve_prime((u32)ps[i], M));
    }
    H.ready = true;
    return H;
}

// ---------------------------------------------------------- device side
struct MarkRec {
    u32 j, n, sf, pad;
};
constexpr int SV_PRIMES = 8;     // primes of 2^d - 1, d <= 32: at most 6
constexpr int PAT_MAX_D = 20;    // degrees that may mark one period
struct SieveDeg {                // one degree of a launch (blockIdx.y)
    int d, lb, np;               // lb: bits of a class word below its prefix
    u32 M, rmod, ap;
    u32 nprefix, per;            // prefixes, and how many a block takes
    u64 q, smax, ncls, qcap;
    const u32 *lo, *hi, *map;    // g^k, g^(k<<16), byte maps
    u32 *surv, *T, *pat;         // pat: marks of one period, or null
    MarkRec *queue;
    unsigned long long *cnt;     // CN_*
    SievePrime pr[SV_PRIMES];
};
enum { CN_SURV, CN_QUEUE, CN_HEAVY, CN_BAD, CN_N };

// exclusive prefix sum of v over the block (blockDim.x = T), and the total;
// wtot: T/64 words of LDS, free again after the caller's next barrier
template <int T>
__device__ unsigned block_excl_scan(unsigned v, unsigned *total, unsigned *wtot) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    unsigned x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const unsigned y = __shfl_up(x, o);
        if (lane >= o) x += y;
    }
    if (lane == 63) wtot[w] = x;
    __syncthreads();
    unsigned before = 0, tot = 0;
#pragma unroll
    for (int i = 0; i < T / 64; i++) {
        const unsigned t = wtot[i];
        if (i < w) before += t;
        tot += t;
    }
    *total = tot;
    return before + x - v;
}

// off[b] = sum of cnt[0..b) for the nb <= 8*T buckets of a block-level
// counting sort, all threads taking part (each sums a run of buckets,
// then one block scan); the caller waits at a barrier before reading off
template <int T>
__device__ void bucket_offsets(const unsigned *cnt, unsigned *off, unsigned nb, unsigned *wtot) {
    const unsigned per = (nb + T - 1) / T;
    const unsigned b0 = threadIdx.x * per;
    unsigned v = 0;
    for (unsigned i = 0; i < per; i++)
        if (b0 + i < nb) v += cnt[b0 + i];
    unsigned total;
    unsigned acc = block_excl_scan<T>(v, &total, wtot);
    for (unsigned i = 0; i < per; i++)
        if (b0 + i < nb) {
            off[b0 + i] = acc;
            acc += cnt[b0 + i];
        }
}

__global__ void k_fill_u32(unsigned *p, u64 n, unsigned v) {
    u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// A Lyndon word of length >= 2 starts with 0 and ends with 1, so only the
// odd j below 2^(d-1) are candidates: candidate c tests j = 2c + 1,
// c < 2^(d-2).  Each thread tests a run of LY_PER consecutive candidates
// against all d-1 rotations (no early exit: about one candidate in d/4 is
// a Lyndon word, so nearly every wave runs all rotations anyway; the
// LY_PER independent chains keep the SIMD busy), the block sums its
// counts, and one atomic per block reserves the block's output run.
// Survivors stay ascending within each block's run.
constexpr int LY_T = 256, LY_PER = 16;

template <class W>
__global__ __launch_bounds__(LY_T) void k_lyndon_t(int d, W M, W *__restrict__ surv,
                                                   unsigned long long *__restrict__ nsurv,
                                                   u64 cap) {
    __shared__ unsigned wtot[LY_T / 64];
    __shared__ unsigned long long bbase;
    const u64 ncand = (u64)1 << (d - 2);
    const u64 chunk = (u64)LY_T * LY_PER;
    for (u64 c0 = (u64)blockIdx.x * chunk; c0 < ncand; c0 += (u64)gridDim.x * chunk) {
        const u64 cb = c0 + (u64)threadIdx.x * LY_PER;
        W jv[LY_PER];
        bool ok[LY_PER];
#pragma unroll
        for (int i = 0; i < LY_PER; i++) {
            jv[i] = (W)(2 * (cb + i) + 1);
            ok[i] = cb + i < ncand;
        }
        for (int k = 1; k < d; k++) {
#pragma unroll
            for (int i = 0; i < LY_PER; i++)
                ok[i] = ok[i] && ((((jv[i] << k) | (jv[i] >> (d - k))) & M) > jv[i]);
        }
        unsigned keep = 0;
#pragma unroll
        for (int i = 0; i < LY_PER; i++) keep |= (unsigned)ok[i] << i;
        unsigned total;
        const unsigned pre = block_excl_scan<LY_T>((unsigned)__popc(keep), &total, wtot);
        if (threadIdx.x == 0) bbase = total ? atomicAdd(nsurv, (unsigned long long)total) : 0;
        __syncthreads();
        u64 pos = bbase + pre;
#pragma unroll
        for (int i = 0; i < LY_PER; i++)
            if ((keep >> i) & 1) {
                if (pos < cap) surv[pos] = jv[i];
                pos++;
            }
        __syncthreads();   // bbase and wtot are rewritten by the next chunk
    }
}

unsigned lyndon_blocks(int d) {
    const u64 chunks = ((((u64)1 << (d - 2)) + (u64)LY_T * LY_PER - 1) / ((u64)LY_T * LY_PER));
    return (unsigned)std::min<u64>(chunks, 8192);
}

constexpr int ZC_T = 256, ZC_PER = 4;   // classes per thread per round

// The classes of a degree: the Lyndon words of length d, which start with 0
// and end with 1, as a list.  A word is a prefix and its low lb bits; a
// block takes `per` prefixes, drops those that cannot begin a Lyndon word
// (nine in ten at d = 32), and its waves try the odd words below the
// others, 256 at a time.  Survivors gather in LDS, one output reservation
// per 4096 or more.  Bounded by VALU issue (1.5 operations a rotation):
// 0.7 ms at d = 32, where testing every odd word below 2^(d-1) took 6.0.
constexpr int CS_T = 256, CS_LB = 11, CS_STAGE = 8192;
__global__ __launch_bounds__(CS_T) void k_classes(const SieveDeg *__restrict__ degs) {
    const SieveDeg &P = degs[blockIdx.y];
    __shared__ u32 stage[CS_STAGE], list[CS_T];
    __shared__ unsigned nlist, nstage;
    __shared__ unsigned long long gpos;
    const int d = P.d, lb = P.lb;
    const u32 ap = P.ap, p0 = blockIdx.x * P.per;
    if (p0 >= P.nprefix) return;   // whole block
    if (threadIdx.x == 0) nlist = nstage = 0;
    __syncthreads();
    if (threadIdx.x < P.per && p0 + threadIdx.x < P.nprefix &&
        lyndon_prefix(p0 + threadIdx.x, d - lb))
        list[atomicAdd(&nlist, 1u)] = p0 + threadIdx.x;
    __syncthreads();
    const u32 n = nlist, ncand = 1u << (lb - 1);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (u32 r = 0; r < n; r += CS_T / 64) {
        const u32 k = r + wave;
        if (k < n) {
            const u32 base = (__builtin_amdgcn_readfirstlane(list[k]) << lb) | 1;
            for (u32 c0 = 0; c0 < ncand; c0 += 256) {
                bool ok[4];
                unsigned long long bal[4];
                unsigned tot = 0;
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const u32 c = c0 + 64 * q + lane;
                    ok[q] = c < ncand && lyndon_word(base + 2 * c, d, ap);
                    bal[q] = __ballot(ok[q]);
                    tot += (unsigned)__popcll(bal[q]);
                }
                unsigned at = 0;
                if (lane == 0) at = atomicAdd(&nstage, tot);
                at = __builtin_amdgcn_readfirstlane(at);
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    if (ok[q])
                        stage[at + (unsigned)__popcll(bal[q] & ((1ULL << lane) - 1))] =
                            base + 2 * (c0 + 64 * q + lane);
                    at += (unsigned)__popcll(bal[q]);
                }
            }
        }
        __syncthreads();
        const unsigned m = nstage;   // at most 4096 more per round
        if (m > CS_STAGE - 4096 || (r + CS_T / 64 >= n && m)) {
            if (threadIdx.x == 0) gpos = atomicAdd(P.cnt + CN_SURV, (unsigned long long)m);
            __syncthreads();
            for (unsigned i = threadIdx.x; i < m; i += CS_T)
                if (gpos + i < P.ncls) P.surv[gpos + i] = stage[i];
            if (threadIdx.x == 0) nstage = 0;
        }
        __syncthreads();
    }
}

// the classes found, at most the list's length
GF2T_DEV u64 class_count(const SieveDeg &P) {
    const u64 n = P.cnt[CN_SURV];
    return n < P.ncls ? n : P.ncls;
}

// T[class of g^j] = log of its least rotation, for every class.  Bounded by
// the VALU (a carry-less product, 31 rotations at 4 operations) and the
// antilog gathers while T stays in the caches, 16 ps a class up to d = 29;
// at d = 32 by the scattered 4-byte stores, 4.2 ms.  The table of all
// logarithms took 38 ms there.
constexpr int CL_T = 256, CL_PER = 4;
__global__ __launch_bounds__(CL_T) void k_class_log(const SieveDeg *__restrict__ degs) {
    const SieveDeg &P = degs[blockIdx.y];
    __shared__ u32 norm[2048];
    const u64 n = class_count(P), chunk = (u64)CL_T * CL_PER;
    if ((u64)blockIdx.x * chunk >= n) return;   // whole block
    for (u32 i = threadIdx.x; i < 2048; i += CL_T) norm[i] = P.map[CL_NORM + i];
    __syncthreads();
    const int d = P.d;
    for (u64 c0 = (u64)blockIdx.x * chunk; c0 < n; c0 += (u64)gridDim.x * chunk) {
        u32 j[CL_PER], hi[CL_PER], lo[CL_PER];
#pragma unroll
        for (int q = 0; q < CL_PER; q++) {
            const u64 t = c0 + (u64)q * CL_T + threadIdx.x;
            j[q] = t < n ? P.surv[t] : 0u;
        }
#pragma unroll
        for (int q = 0; q < CL_PER; q++) {
            hi[q] = P.hi[j[q] >> 16];
            lo[q] = P.lo[j[q] & 0xFFFF];
        }
#pragma unroll
        for (int q = 0; q < CL_PER; q++) {
            const u64 t = c0 + (u64)q * CL_T + threadIdx.x;
            int k;
            const u32 m = least_rotation(periodic64(map8((const u32 *)norm, clmul32(hi[q], lo[q])), d), k);
            if (t < n) P.T[class_index(m, d)] = rotl_d(j[q], k, d);
        }
    }
}

// Per class: Zech logarithm (one random gather), the progression
// s == s0 (mod n), and -- only for the few classes whose progression
// reaches s <= smax -- a queue entry, so that k_mark's minimal polynomials
// run on dense waves.  A thread takes PER classes (8, or 2 where there are
// too few to fill the chip and a launch is as long as one thread: 24 us
// and 13 for the degrees up to 20, but 38 and 80 at degree 25): their
// lookups are
// overlapped, and one Euclid inverts the product of their units (three
// products a class; a gcd, an inverse and two divisions a class before).
// Bounded by the VALU and the gathers: 3.3 ms at d = 32, 5.6 before.
constexpr int ZN_T = 256;
template <int ZN_PER>
__global__ __launch_bounds__(ZN_T) void k_zech(const SieveDeg *__restrict__ degs) {
    const SieveDeg &P = degs[blockIdx.y];
    __shared__ u32 norm[2048], zech[ZN_T * ZN_PER];
    __shared__ unsigned wtot[ZN_T / 64];
    __shared__ unsigned long long bbase;
    const u64 n = class_count(P), chunk = (u64)ZN_T * ZN_PER;
    if ((u64)blockIdx.x * chunk >= n) return;   // whole block
    for (u32 i = threadIdx.x; i < 2048; i += ZN_T) norm[i] = P.map[CL_NORM + i];
    __syncthreads();
    const int d = P.d;
    const u32 M = P.M;
    for (u64 c0 = (u64)blockIdx.x * chunk; c0 < n; c0 += (u64)gridDim.x * chunk) {
        // Zech logarithms, one class after another (all eight unrolled
        // together took 256 VGPRs and scratch): a gather is on its way
        // while the next class's rotation is found
        u32 back = 0;   // the rotation still to be undone of the last gather
        u32 got = 0;
#pragma unroll 1
        for (int q = 0; q <= ZN_PER; q++) {
            u32 next = 0, nback = 0;
            const u64 t = c0 + (u64)q * ZN_T + threadIdx.x;
            if (q < ZN_PER && t < n) {
                const u32 u = mulmod_mersenne(P.surv[t], P.rmod, d, M);   // beta^r = g^u, not 1: r is prime to M
                // w(1) is all ones
                const u32 w = map8((const u32 *)norm, clmul32(P.hi[u >> 16], P.lo[u & 0xFFFF])) ^ M;
                int k;
                next = P.T[class_index(least_rotation(periodic64(w, d), k), d)];
                nback = (u32)(d - k);
            }
            if (q) zech[(q - 1) * ZN_T + threadIdx.x] = rotl_d(got, (int)back, d);
            got = next;
            back = nback;
        }
        u32 j[ZN_PER], v[ZN_PER];   // v: log(beta^r + 1)
        unsigned live = 0;
#pragma unroll
        for (int q = 0; q < ZN_PER; q++) {
            const u64 t = c0 + (u64)q * ZN_T + threadIdx.x;
            live |= (unsigned)(t < n) << q;
            j[q] = t < n ? P.surv[t] : 1u;
            v[q] = zech[q * ZN_T + threadIdx.x];   // this thread's own
        }
        u32 un[ZN_PER], nn[ZN_PER], pre[ZN_PER];
        live &= progressions(v, j, nn, un, M, P.pr, P.np);
#pragma unroll
        for (int q = 0; q < ZN_PER; q++)
            pre[q] = q ? mulmod_mersenne(pre[q - 1], un[q], d, M) : un[q];
        u32 inv = inv32(pre[ZN_PER - 1], M);
        unsigned keep = 0;
#pragma unroll
        for (int q = ZN_PER - 1; q >= 0; q--) {
            const u32 iv = q ? mulmod_mersenne(inv, pre[q - 1], d, M) : inv;
            inv = mulmod_mersenne(inv, un[q], d, M);
            u32 s0 = mulmod_mersenne(iv, v[q], d, M);
            if (nn[q] != M) s0 %= nn[q];
            v[q] = s0 ? s0 : nn[q];                              // first s >= 1
            if (((live >> q) & 1) && v[q] <= P.smax) keep |= 1u << q;
        }
        unsigned total;
        const unsigned before = block_excl_scan<ZN_T>((unsigned)__popc(keep), &total, wtot);
        if (threadIdx.x == 0)
            bbase = total ? atomicAdd(P.cnt + CN_QUEUE, (unsigned long long)total) : 0;
        __syncthreads();
        u64 pos = bbase + before;
#pragma unroll
        for (int q = 0; q < ZN_PER; q++)
            if ((keep >> q) & 1) {
                if (pos < P.qcap) P.queue[pos] = MarkRec{j[q], nn[q], v[q], 0};
                pos++;
            }
        __syncthreads();   // bbase and wtot are rewritten by the next round
    }
}

// Per queued class: minimal polynomial, then the marks: of one period
// (P.pat), inline up to INLINE_MARKS, or through the heavy queue (hcount
// entries so far).  Bounded by the random read-modify-writes of best[]:
// 0.16 ms at d = 32 and 0.30 ms at d = 28, where each class's 64 products
// with a bit-serial reduction took 1.07 and 0.82.
constexpr int MK_T = 256;
__global__ __launch_bounds__(MK_T) void k_mark(const SieveDeg *__restrict__ degs,
                                               unsigned long long *__restrict__ best,
                                               Heavy *__restrict__ heavy,
                                               unsigned long long *__restrict__ hcount) {
    const SieveDeg &P = degs[blockIdx.y];
    __shared__ u32 map[CL_MAP - CL_RED];
    const u64 all = P.cnt[CN_QUEUE], nq = all < P.qcap ? all : P.qcap;
    if ((u64)blockIdx.x * MK_T >= nq) return;   // whole block
    for (u32 i = threadIdx.x; i < CL_MAP - CL_RED; i += MK_T) map[i] = P.map[CL_RED + i];
    __syncthreads();
    const u32 *red = map, *dual = map + (CL_DUAL - CL_RED);
    const int d = P.d;
    const u64 smax = P.smax;
    for (u64 t = (u64)blockIdx.x * MK_T + threadIdx.x; t < nq; t += (u64)gridDim.x * MK_T) {
        const MarkRec rec = P.queue[t];
        const u32 beta = red_product(clmul32(P.hi[rec.j >> 16], P.lo[rec.j & 0xFFFF]), red, d);
        const u64 mask = minpoly_seq(trace_sequence(beta, red, dual, d), d);
        if (mask == 0 || !((mask >> d) & 1) || !(mask & 1)) {
            atomicOr(P.cnt + CN_BAD, 1ULL);
            continue;
        }
        const unsigned long long key = ((unsigned long long)d << 48) | mask;
        const u64 n = rec.n, sf = rec.sf, count = (smax - sf) / n + 1;
        if (count > INLINE_MARKS) atomicAdd(P.cnt + CN_HEAVY, 1ULL);
        if (P.pat) {
            for (u32 s = sf == n ? 0u : (u32)sf; s < P.M; s += (u32)n) atomicMin(&P.pat[s], (u32)mask);
        } else if (count <= INLINE_MARKS) {
            for (u64 s = sf; s <= smax; s += 4 * n) {   // four loads on their way
                unsigned long long now[4];
#pragma unroll
                for (int i = 0; i < 4; i++) now[i] = s + i * n <= smax ? best[s + i * n] : 0;
#pragma unroll
                for (int i = 0; i < 4; i++)
                    if (now[i] > key) atomicMin(&best[s + i * n], key);
            }
        } else {
            const u64 idx = atomicAdd(hcount, 1ULL);
            if (idx < HEAVY_CAP) heavy[idx] = Heavy{sf, n, key};
            else atomicOr(P.cnt + CN_BAD, 2ULL);
        }
    }
}

// Degrees lo..hi marked one period each (pat).  2^d - 1 divides 2^e - 1
// where d divides e, so only the periods of the degrees e > hi / 2 are
// needed: k_fold_periods takes the marks of e's divisors into e's table,
// as keys d << 21 | mask, the lowest first.
struct PeriodArgs {
    const u32 *pat[PAT_MAX_D + 1];   // marks of degree d
    u32 *tab[PAT_MAX_D / 2];         // tables of the degrees first..hi
    u32 divs[PAT_MAX_D / 2];         // bit d: d divides that degree, and was marked
    int lo, hi, first;
};
__global__ void k_fold_periods(PeriodArgs A) {
    const int e = A.first + (int)blockIdx.y;
    const u32 M = (1u << e) - 1;
    for (u32 x = blockIdx.x * blockDim.x + threadIdx.x; x < M; x += gridDim.x * blockDim.x) {
        u32 key = ~0u;
        for (u32 w = A.divs[blockIdx.y]; w; w &= w - 1) {
            const int d = __builtin_ctz(w);
            const u32 m = A.pat[d][x % ((1u << d) - 1)];
            if (m != ~0u) {
                key = (u32)d << 21 | m;
                break;
            }
        }
        A.tab[blockIdx.y][x] = key;
    }
}
// Every s through those tables: the least key is the least factor of the
// degrees lo..hi.  One pass over best[], with its loads and stores, and
// the tables' loads, in order: 0.55 ms for 68,139,920 s and degrees 2..20,
// where marking the progressions one by one took 4.6.
// A thread takes `per` values of s, fewer where they would leave the chip
// idle (66,024 values: 36 us at 16 each, 5.6 us at one).
constexpr int SW_T = 256;
__global__ __launch_bounds__(SW_T) void k_sweep(PeriodArgs A, u64 smax, u32 per,
                                                unsigned long long *__restrict__ best) {
    constexpr int N = PAT_MAX_D / 2;
    __shared__ u32 base[N];   // the block's first s modulo each period
    const u64 s0 = 1 + (u64)blockIdx.x * SW_T * per;
    if (threadIdx.x < N && A.first + (int)threadIdx.x <= A.hi)
        base[threadIdx.x] = (u32)(s0 % (((u64)1 << (A.first + threadIdx.x)) - 1));
    __syncthreads();
    u32 x[N];
#pragma unroll
    for (int i = 0; i < N; i++)
        if (A.first + i <= A.hi) x[i] = (base[i] + threadIdx.x) % ((1u << (A.first + i)) - 1);
    for (u32 it = 0; it < per; it++) {
        const u64 s = s0 + it * SW_T + threadIdx.x;
        if (s > smax) return;
        const unsigned long long now = best[s];
        u32 key = ~0u;
#pragma unroll
        for (int i = 0; i < N; i++) {
            if (A.first + i > A.hi) break;
            const u32 M = (1u << (A.first + i)) - 1, m = A.tab[i][x[i]];
            key = m < key ? m : key;
            x[i] += SW_T % M;
            x[i] = x[i] >= M ? x[i] - M : x[i];
        }
        if (key == ~0u) continue;
        const unsigned long long k64 =
            ((unsigned long long)(key >> 21) << 48) | (key & ((1u << 21) - 1));
        if (now > k64) best[s] = k64;
    }
}

// nheavy: how many, or null and `known`
__global__ void k_mark_heavy(const Heavy *__restrict__ heavy,
                             const unsigned long long *__restrict__ count_at, unsigned known,
                             u64 smax, unsigned long long *__restrict__ best) {
    const unsigned nheavy = count_at ? (unsigned)(*count_at < HEAVY_CAP ? *count_at : HEAVY_CAP) : known;
    for (unsigned rec = blockIdx.y; rec < nheavy; rec += gridDim.y) {
        const Heavy h = heavy[rec];
        u64 count = (smax - h.s_first) / h.n + 1;
        for (u64 k = (u64)blockIdx.x * blockDim.x + threadIdx.x; k < count;
             k += (u64)gridDim.x * blockDim.x) {
            u64 s = h.s_first + k * h.n;
            if (best[s] > h.key) atomicMin(&best[s], (unsigned long long)h.key);
        }
    }
}

__global__ void k_zero_counters(unsigned long long *a, unsigned *b) {
    if (threadIdx.x < 4) a[threadIdx.x] = 0;
    if (threadIdx.x < 4) b[threadIdx.x] = 0;
}


struct DevBuf {
    void *p = nullptr;
    size_t bytes = 0;
    void release() {
        if (p) (void)hipFree(p);
        p = nullptr;
        bytes = 0;
    }
    int ensure(size_t b) {
        if (bytes >= b) return GF2T_OK;
        if (p) GF2T_HIP(hipFree(p));
        p = nullptr;
        bytes = 0;
        GF2T_HIP(hipMalloc(&p, b));
        bytes = b;
        return GF2T_OK;
    }
};

// ===================================================== degrees 33..36
// Elements of GF(2^d) are u64.  The log table holds d-bit exponents, so
// it is stored as the low 32 bits (L_lo, u32) plus the top four bits
// packed eight to a word (L_hi).  It is built by the same radix
// partition as above, except that the level-2 split runs one level-1
// bucket at a time, to a bucket-sized scratch region and back (two
// counting-sort passes), so the whole build needs 8 bytes per element
// plus the table (about 205 GB at d = 34, inside 288 GB).  Entries are
// (g^i mod 2^(d-8)) << 36 | i.
// Above d = 34 the table is built and used in value slices: slice k holds
// the logs of the field elements whose top byte lies in [k nb, (k+1) nb),
// nb = 256 / slices.  Each slice's partition pass generates every power
// but keeps only its own buckets, and the Zech pass of the slice resolves
// only the classes whose lookup value falls in it; the marking queue
// collects all slices' classes.  So the memory of d = 35 (two slices) and
// d = 36 (four) is that of d = 34, and the extra cost is one generation
// pass over the powers per slice.
constexpr int WIDE_MAX_D = 36;
constexpr int W_DENSE_D = 34;       // largest degree with the whole table at once
constexpr int W_SB = 15;            // values per placed slice: 2^15
constexpr int W_E = 8192;           // entries per block in passes 1 and 2
constexpr int W_T = 256;
constexpr int W_IB = 36;            // bits of i in an entry
constexpr int W_B1 = 8;             // level-1 bucket bits
constexpr int W_AB = 18;            // antilog table split: g^e = A1[e >> 18] * A0[e & (2^18 - 1)]

struct WParams {
    int d;
    u64 M, q, rmod, smax, tmask;
    const u64 *A0, *A1;
};

GF2T_DEV u64 antilog_w(const WParams &P, u64 e) {
    return fmul64(P.A1[e >> W_AB], P.A0[e & ((1u << W_AB) - 1)], P.q, P.d);
}

// block-wide exclusive scan of cnt[0..nb) (nb <= W_T * 16) into off;
// part: W_T / 64 words of LDS
__device__ void block_scan(const unsigned *cnt, unsigned *off, unsigned nb, unsigned *part) {
    bucket_offsets<W_T>(cnt, off, nb, part);
    __syncthreads();
}

// Pass 1 of the table build for the level-1 buckets [b0, b0 + nb): every
// power g^i is generated, and those whose top byte is in range are
// appended to bucket (top byte - b0) of out (2^(d-8) entries each).
__global__ __launch_bounds__(W_T) void k_w_part1(WParams P, unsigned long long *__restrict__ out,
                                                 unsigned *__restrict__ cursor,
                                                 unsigned *__restrict__ bad, unsigned b0,
                                                 unsigned nb) {
    __shared__ unsigned cnt[256], off[256], gbase[256], part[W_T];
    __shared__ unsigned long long stage[W_E];
    __shared__ unsigned char sbkt[W_E];   // bucket of each staged entry
    const int shift = P.d - W_B1;
    const u64 cap = (u64)1 << shift;
    const u64 i0 = (u64)blockIdx.x * W_E;
    cnt[threadIdx.x] = 0;
    __syncthreads();
    constexpr int PER = W_E / W_T;
    const u64 my0 = i0 + (u64)threadIdx.x * PER;
    unsigned rank[PER];
    u64 a0 = my0 < P.M ? antilog_w(P, my0) : 0, a = a0;
#pragma unroll
    for (int k = 0; k < PER; k++) {
        rank[k] = 0;
        const unsigned b = (unsigned)(a >> shift);
        if (my0 + k < P.M && b - b0 < nb) rank[k] = atomicAdd(&cnt[b], 1u);
        a <<= 1;
        if (a >> P.d) a ^= P.q;
    }
    __syncthreads();
    block_scan(cnt, off, 256, part);
    gbase[threadIdx.x] = cnt[threadIdx.x] ? atomicAdd(&cursor[threadIdx.x], cnt[threadIdx.x]) : 0;
    a = a0;
#pragma unroll
    for (int k = 0; k < PER; k++) {
        const unsigned b = (unsigned)(a >> shift);
        if (my0 + k < P.M && b - b0 < nb) {
            const unsigned at = off[b] + rank[k];
            stage[at] = ((unsigned long long)(a & (cap - 1)) << W_IB) | (my0 + k);
            sbkt[at] = (unsigned char)b;
        }
        a <<= 1;
        if (a >> P.d) a ^= P.q;
    }
    __syncthreads();
    const u64 nvalid = (u64)off[255] + cnt[255];   // entries staged in range
    for (u64 k = threadIdx.x; k < nvalid; k += W_T) {
        const unsigned b = sbkt[k];
        u64 pos = (u64)gbase[b] + (k - off[b]);
        if (pos >= cap) { atomicOr(bad, 4u); continue; }
        out[(u64)(b - b0) * cap + pos] = stage[k];
    }
}

// One counting-sort pass of the level-2 split, which runs as two such
// passes per level-1 bucket (about half the d - 23 level-2 bits each, so
// every block writes runs of 128-256 entries): source bucket blockIdx.y
// (src_cap entries apart; the first holds first_count) is partitioned by
// the nbits-bit digit at bit `shift` of the stored value into
// destination buckets src * 2^nbits + digit of dst_cap entries each.
constexpr int WS_MAXB = 128;  // digits per pass (2^7: degree 36 splits 13 bits as 7 + 6)
constexpr int WS_T = 512;     // threads per block
__global__ __launch_bounds__(WS_T) void k_w_split(const unsigned long long *__restrict__ in,
                                                 u64 src_cap, u64 first_count, int shift,
                                                 int nbits, unsigned long long *__restrict__ out,
                                                 u64 dst_cap, unsigned *__restrict__ cursor,
                                                 unsigned *__restrict__ bad) {
    __shared__ unsigned cnt[WS_MAXB], off[WS_MAXB], gbase[WS_MAXB], part[WS_T / 64];
    __shared__ unsigned long long stage[W_E];
    const unsigned nd = 1u << nbits;
    const unsigned src = blockIdx.y;
    const u64 count = src ? src_cap : first_count;
    const u64 k0 = (u64)blockIdx.x * W_E;
    if (k0 >= count) return;
    const u64 nvalid = (k0 + W_E <= count) ? W_E : count - k0;
    const unsigned long long *sp = in + (u64)src * src_cap + k0;
    const int dsh = W_IB + shift;
    for (unsigned b = threadIdx.x; b < nd; b += WS_T) cnt[b] = 0;
    __syncthreads();
    constexpr int PER = W_E / WS_T;
    unsigned rank[PER];
#pragma unroll
    for (int k = 0; k < PER; k++) {
        const u64 idx = (u64)k * WS_T + threadIdx.x;
        rank[k] = idx < nvalid ? atomicAdd(&cnt[(unsigned)(sp[idx] >> dsh) & (nd - 1)], 1u) : 0;
    }
    __syncthreads();
    bucket_offsets<WS_T>(cnt, off, nd, part);
    __syncthreads();
    for (unsigned b = threadIdx.x; b < nd; b += WS_T)
        gbase[b] = cnt[b] ? atomicAdd(&cursor[src * nd + b], cnt[b]) : 0;
#pragma unroll
    for (int k = 0; k < PER; k++) {
        const u64 idx = (u64)k * WS_T + threadIdx.x;
        if (idx < nvalid) {
            const unsigned long long e = sp[idx];
            stage[off[(unsigned)(e >> dsh) & (nd - 1)] + rank[k]] = e;
        }
    }
    __syncthreads();
    for (u64 k = threadIdx.x; k < nvalid; k += WS_T) {
        const unsigned long long e = stage[k];
        const unsigned b = (unsigned)(e >> dsh) & (nd - 1);
        const u64 pos = (u64)gbase[b] + (k - off[b]);
        if (pos >= dst_cap) { atomicOr(bad, 4u); continue; }
        out[((u64)src * nd + b) * dst_cap + pos] = e;
    }
}

// one block per run z of 2^W_SB values of the slice: L_lo and the
// packed top bits.  zero_first: the slice starts at value 0, which has no
// logarithm (its run holds 2^W_SB - 1 entries; L[0] is left 0)
__global__ __launch_bounds__(1024) void k_w_place(const unsigned long long *__restrict__ in,
                                                  u32 *__restrict__ Llo, u32 *__restrict__ Lhi,
                                                  int zero_first) {
    extern __shared__ u32 wtile[];
    u32 *lo = wtile, *hi = wtile + (1u << W_SB);          // hi: 4 bits per value
    const u64 cap = (u64)1 << W_SB;
    const u64 z = blockIdx.x;
    const bool has_zero = zero_first && z == 0;
    const u64 count = has_zero ? cap - 1 : cap;
    const unsigned long long *src = in + z * cap;
    for (u64 k = threadIdx.x; k < cap / 8; k += blockDim.x) hi[k] = 0;
    if (has_zero && threadIdx.x == 0) lo[0] = 0;
    __syncthreads();
    for (u64 k = threadIdx.x; k < count; k += blockDim.x) {
        unsigned long long e = src[k];
        u32 v = (u32)(e >> W_IB) & (u32)(cap - 1);
        u64 i = e & (((u64)1 << W_IB) - 1);
        lo[v] = (u32)i;
        atomicOr(&hi[v >> 3], (u32)((i >> 32) & 15) << (4 * (v & 7)));
    }
    __syncthreads();
    for (u64 k = threadIdx.x; k < cap; k += blockDim.x) Llo[z * cap + k] = lo[k];
    for (u64 k = threadIdx.x; k < cap / 8; k += blockDim.x) Lhi[z * (cap / 8) + k] = hi[k];
}

struct MarkRecW {
    u64 j, n, sf;
};

// as k_zech: ZC_PER classes per thread, lookups first, one reservation
// per block; only the classes whose lookup value y = beta^r + 1 lies in
// the table slice [ybase, ybase + yspan) are resolved
__global__ __launch_bounds__(ZC_T) void k_zech_w(WParams P, const u64 *__restrict__ surv,
                                                 u64 nsurv, const u32 *__restrict__ Llo,
                                                 const u32 *__restrict__ Lhi,
                                                 MarkRecW *__restrict__ queue,
                                                 unsigned long long *__restrict__ nqueue,
                                                 u64 qcap, u64 ybase, u64 yspan) {
    __shared__ unsigned wtot[ZC_T / 64];
    __shared__ unsigned long long bbase;
    const u64 chunk = (u64)ZC_T * ZC_PER;
    for (u64 c0 = (u64)blockIdx.x * chunk; c0 < nsurv; c0 += (u64)gridDim.x * chunk) {
        u64 j[ZC_PER], y[ZC_PER], v[ZC_PER];
        bool live[ZC_PER];
#pragma unroll
        for (int q = 0; q < ZC_PER; q++) {
            const u64 t = c0 + (u64)q * ZC_T + threadIdx.x;
            live[q] = t < nsurv;
            j[q] = live[q] ? surv[t] : 1;
        }
#pragma unroll
        for (int q = 0; q < ZC_PER; q++) {
            const u64 u = mulmod64(j[q], P.rmod, P.M);
            live[q] = live[q] && u;                    // u = 0: beta^r = 1, never a root
            y[q] = (antilog_w(P, u ? u : 1) ^ 1u) - ybase;
            live[q] = live[q] && y[q] < yspan;         // resolved by this slice's table
        }
#pragma unroll
        for (int q = 0; q < ZC_PER; q++)
            v[q] = live[q] ? ((u64)Llo[y[q]] |
                              ((u64)((Lhi[y[q] >> 3] >> (4 * (y[q] & 7))) & 15) << 32))
                           : 0;
        unsigned keep = 0;
        MarkRecW rec[ZC_PER];
#pragma unroll
        for (int q = 0; q < ZC_PER; q++) {
            rec[q] = MarkRecW{0, 0, 0};
            if (!live[q]) continue;
            const u64 gg = gcd64(j[q], P.M);
            if (v[q] % gg) continue;
            const u64 n = P.M / gg;
            const u64 iv = inv64((j[q] / gg) % n, n);
            const u64 s0 = mulmod64(iv, v[q] / gg, n);
            const u64 sf = s0 ? s0 : n;
            if (sf <= P.smax) {
                keep |= 1u << q;
                rec[q] = MarkRecW{j[q], n, sf};
            }
        }
        unsigned total;
        const unsigned pre = block_excl_scan<ZC_T>((unsigned)__popc(keep), &total, wtot);
        if (threadIdx.x == 0) bbase = total ? atomicAdd(nqueue, (unsigned long long)total) : 0;
        __syncthreads();
        u64 pos = bbase + pre;
#pragma unroll
        for (int q = 0; q < ZC_PER; q++)
            if ((keep >> q) & 1) {
                if (pos < qcap) queue[pos] = rec[q];
                pos++;
            }
        __syncthreads();
    }
}

__global__ void k_mark_w(WParams P, const MarkRecW *__restrict__ queue, u64 nq,
                         unsigned long long *__restrict__ best, Heavy *__restrict__ heavy,
                         unsigned *__restrict__ nheavy, unsigned *__restrict__ bad) {
    u64 t = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nq) return;
    const MarkRecW rec = queue[t];
    const int d = P.d;
    u64 mask = minpoly_bm64(antilog_w(P, rec.j), P.q, d, P.tmask);
    if (mask == 0 || !((mask >> d) & 1) || !(mask & 1)) { atomicAdd(bad, 1u); return; }
    unsigned long long key = ((unsigned long long)d << 48) | mask;
    u64 count = (P.smax - rec.sf) / rec.n + 1;
    if (count <= INLINE_MARKS) {
        for (u64 s = rec.sf; s <= P.smax; s += rec.n)
            if (best[s] > key) atomicMin(&best[s], key);
    } else {
        unsigned idx = atomicAdd(nheavy, 1u);
        if (idx < HEAVY_CAP) heavy[idx] = Heavy{rec.sf, rec.n, key};
        else atomicAdd(bad, 2u);
    }
}

struct WideHost {
    bool ready = false, trace_ok = false;
    u64 q = 0, tmask = 0;
    std::vector<u64> a0, a1;
};
std::mutex g_wide_mu;
WideHost g_wide[WIDE_MAX_D + 1];

const WideHost &wide_host(int d) {
    std::lock_guard<std::mutex> lk(g_wide_mu);
    WideHost &H = g_wide[d];
    if (H.ready) return H;
    H.q = primitive_poly(d);
    const size_t na = (size_t)1 << W_AB;
    H.a0.assign(na, 0);
    H.a1.assign(na, 0);
    if (H.q) {
        const u64 q = H.q;
        u64 a = 1;
        for (size_t k = 0; k < na; k++) {
            H.a0[k] = a;
            a <<= 1;
            if ((a >> d) & 1) a ^= q;
        }
        const u64 gstep = a;   // g^(2^18); multiplying by it is linear: byte tables
        u64 T[5][256];
        for (int j = 0; j < 5; j++)
            for (u64 v = 0; v < 256; v++) {
                u64 e = v << (8 * j);
                T[j][v] = (e >> d) ? 0 : hmulmod(e, gstep, q, d);
            }
        u64 b = 1;
        for (size_t k = 0; k < na; k++) {
            H.a1[k] = b;
            b = T[0][b & 255] ^ T[1][(b >> 8) & 255] ^ T[2][(b >> 16) & 255] ^
                T[3][(b >> 24) & 255] ^ T[4][(b >> 32) & 255];
        }
        H.trace_ok = true;
        for (int i = 0; i < d; i++) {
            u64 y = (u64)1 << i, acc = y;
            for (int k = 1; k < d; k++) { y = hmulmod(y, y, q, d); acc ^= y; }
            if (acc > 1) { H.trace_ok = false; break; }
            H.tmask |= acc << i;
        }
    }
    H.ready = true;
    return H;
}

struct SieveWork {
    DevBuf bClass, bHeavy, bTab, bCnt, bPat, bDegs;
    u64 tab_ready = 0;   // degrees whose tables bTab holds
    DevBuf wP1, wTmp, wLlo, wLhi, wSurv, wQueue, wTab, wCur;   // degrees 33..34
};
std::mutex g_sw_mu;
SieveWork *g_sw = nullptr;   // never destroyed at exit: the runtime may be gone by then

}  // namespace

extern "C" int gf2t_sieve_release(void) {
    std::lock_guard<std::mutex> lk(g_sw_mu);
    if (g_sw) {
        for (DevBuf *b : {&g_sw->bClass, &g_sw->bHeavy, &g_sw->bTab, &g_sw->bCnt, &g_sw->bPat,
                          &g_sw->bDegs, &g_sw->wP1, &g_sw->wTmp, &g_sw->wLlo, &g_sw->wLhi,
                          &g_sw->wSurv, &g_sw->wQueue, &g_sw->wTab, &g_sw->wCur})
            b->release();
        g_sw->tab_ready = 0;
    }
    return GF2T_OK;
}

extern "C" uint64_t gf2t_primitive_poly(int d) {
    if (d < 2 || d > 40) return 0;
    return primitive_poly(d);
}

namespace {
// per-degree phase timers, destroyed on every return path
struct SieveEvents {
    hipEvent_t e[33][4] = {};
    ~SieveEvents() {
        for (auto &g : e)
            for (hipEvent_t x : g)
                if (x) (void)hipEventDestroy(x);
    }
};

constexpr size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }

// Degrees that run in one launch: up to 20, 21..23, then each by itself (a degree-24 launch fills the card).  A launch waits for nothing
// on the host, and costs about 5 us however little it does.
int group_end(int d, int dmax) {
    return std::min(dmax, d <= PAT_MAX_D ? PAT_MAX_D : d <= 23 ? 23 : d);
}

// bytes of a degree's class table, class list and marking queue
struct NarrowBytes {
    size_t T, surv, queue;
    size_t all() const { return T + surv + queue; }
};
NarrowBytes narrow_bytes(int d) {
    const u64 ncls = irreducible_count(d);
    return {align256(((size_t)1 << (d - 2)) * 4), align256(ncls * 4), align256(ncls * sizeof(MarkRec))};
}

// The arrays of the largest group.  They are carved out of the wide log
// table whenever that is allocated and large enough, so a sieve to degree
// 34 never holds both.
int narrow_mem(int dmin, int dmax, char *&mem) {
    SieveWork &W = *g_sw;
    size_t bytes = 0;
    for (int d = dmin; d <= dmax;) {
        const int e = group_end(d, dmax);
        size_t b = 0;
        for (; d <= e; d++) b += narrow_bytes(d).all();
        bytes = std::max(bytes, b);
    }
    if (W.wLlo.bytes >= bytes) {
        mem = (char *)W.wLlo.p;
        return GF2T_OK;
    }
    if (int rc = W.bClass.ensure(bytes)) return rc;
    mem = (char *)W.bClass.p;
    return GF2T_OK;
}

// degrees dmin..dmax <= 32 (u32 field elements); g_sw_mu held by the caller
int sieve_narrow(uint64_t r, int dmin, int dmax, uint64_t smax, uint64_t *dbest,
                 gf2t_sieve_stats *stats) {
    SieveWork &W = *g_sw;
    int status = GF2T_OK, rc;
    // the degrees before the first that cannot be done
    for (int d = dmin; d <= dmax; d++) {
        const u64 M = ((u64)1 << d) - 1, rmod = r % M;
        const DegHost &H = deg_host(d);
        if (!H.q || gcd_host(rmod ? rmod : M, M) != 1) {
            gf2t::set_error("gf2t_sieve: d=%d: gcd(r, 2^d-1) != 1, unsupported r", d);
            status = GF2T_EINVAL;
        } else if (!H.trace_ok || H.primes.size() > SV_PRIMES) {
            gf2t::set_error("gf2t_sieve: d=%d: trace not in GF(2)", d);
            status = GF2T_EINTERNAL;
        }
        if (status != GF2T_OK) {
            dmax = d - 1;
            break;
        }
    }
    if (dmax < dmin) return status;
    char *mem;
    if ((rc = narrow_mem(dmin, dmax, mem))) return rc;
    if ((rc = W.bTab.ensure(33 * DEG_TAB * sizeof(u32)))) return rc;
    if ((rc = W.bHeavy.ensure((size_t)HEAVY_CAP * sizeof(Heavy)))) return rc;
    if ((rc = W.bPat.ensure(((size_t)4 << PAT_MAX_D) * sizeof(u32)))) return rc;   // marks, tables
    if ((rc = W.bDegs.ensure(33 * sizeof(SieveDeg)))) return rc;
    if ((rc = W.bCnt.ensure(34 * CN_N * 8))) return rc;
    u32 *tabs = (u32 *)W.bTab.p, *pats = (u32 *)W.bPat.p;
    unsigned long long *cnt = (unsigned long long *)W.bCnt.p;   // by degree; then the heavy queue's
    unsigned long long *hcount = cnt + 33 * CN_N;
    Heavy *heavy = (Heavy *)W.bHeavy.p;
    SieveDeg degs[33];
    for (int d = dmin; d <= dmax;) {
        char *at = mem;
        for (const int e = group_end(d, dmax); d <= e; d++) {
            const DegHost &H = deg_host(d);
            u32 *tab = tabs + (size_t)d * DEG_TAB;
            if (!((W.tab_ready >> d) & 1)) {
                GF2T_HIP(hipMemcpy(tab, H.tab.data(), DEG_TAB * sizeof(u32), hipMemcpyHostToDevice));
                W.tab_ready |= 1ULL << d;
            }
            const NarrowBytes nb = narrow_bytes(d);
            SieveDeg &P = degs[d];
            P.d = d;
            P.lb = std::min(CS_LB, d - 1);
            P.np = (int)H.primes.size();
            P.M = (u32)(((u64)1 << d) - 1);
            P.rmod = (u32)(r % P.M);
            P.ap = aperiodic_rotations(d);
            P.nprefix = 1u << (d - P.lb - 1);
            P.per = std::min<u32>(CS_T, std::max<u32>(4, P.nprefix / 2048));
            P.q = H.q;
            P.smax = smax;
            P.ncls = P.qcap = irreducible_count(d);
            P.lo = tab;
            P.hi = tab + 65536;
            P.map = tab + 2 * 65536;
            P.T = (u32 *)at;
            P.surv = (u32 *)(at + nb.T);
            P.queue = (MarkRec *)(at + nb.T + nb.surv);
            at += nb.all();
            P.pat = d <= PAT_MAX_D && P.M <= smax ? pats + ((size_t)1 << d) : nullptr;
            P.cnt = cnt + d * CN_N;
            for (int i = 0; i < P.np; i++) P.pr[i] = H.primes[i];
        }
    }
    SieveEvents evs;
    hipEvent_t(&ev)[33][4] = evs.e;   // [first degree of a group]
    if (stats)
        for (int d = dmin; d <= dmax; d = group_end(d, dmax) + 1)
            for (auto &e : ev[d]) GF2T_HIP(hipEventCreate(&e));
    SieveDeg *ddegs = (SieveDeg *)W.bDegs.p;
    GF2T_HIP(hipMemcpyAsync(ddegs + dmin, degs + dmin, (dmax - dmin + 1) * sizeof(SieveDeg),
                            hipMemcpyHostToDevice, 0));
    hipLaunchKernelGGL(k_fill_u32, dim3(2), dim3(256), 0, 0, (unsigned *)cnt, (u64)34 * CN_N * 2, 0u);
    for (int d = dmin; d <= dmax;) {
        const int e = group_end(d, dmax);
        const unsigned ny = (unsigned)(e - d + 1);
        const SieveDeg *g = ddegs + d;
        u64 bc = 0, bl = 0, bm = 0, most = 0;
        PeriodArgs A{};
        A.lo = d;
        A.hi = d - 1;
        for (int k = d; k <= e; k++) {
            const SieveDeg &P = degs[k];
            bc = std::max<u64>(bc, (P.nprefix + P.per - 1) / P.per);
            bl = std::max<u64>(bl, (P.ncls + CL_T * CL_PER - 1) / (CL_T * CL_PER));
            most = std::max(most, P.ncls);
            bm = std::max<u64>(bm, (P.ncls + MK_T - 1) / MK_T);
            if (P.pat) {
                A.pat[k] = P.pat;
                A.hi = k;
            }
        }
        if (stats) GF2T_HIP(hipEventRecord(ev[d][0], 0));
        hipLaunchKernelGGL(k_classes, dim3((unsigned)bc, ny), dim3(CS_T), 0, 0, g);
        hipLaunchKernelGGL(k_class_log, dim3((unsigned)std::min<u64>(bl, 4096), ny), dim3(CL_T), 0, 0, g);
        if (stats) GF2T_HIP(hipEventRecord(ev[d][1], 0));
        const u64 zper = most >= ((u64)8 * ZN_T * 64) ? 8 : 2;
        const dim3 gz((unsigned)std::min<u64>((most + ZN_T * zper - 1) / (ZN_T * zper), 4096), ny);
        if (zper == 8) hipLaunchKernelGGL(k_zech<8>, gz, dim3(ZN_T), 0, 0, g);
        else hipLaunchKernelGGL(k_zech<2>, gz, dim3(ZN_T), 0, 0, g);
        const bool periods = A.hi >= A.lo;
        if (periods) {
            const u64 n = (u64)2 << A.hi;
            hipLaunchKernelGGL(k_fill_u32, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, 0, pats, n, ~0u);
            A.first = std::max(A.lo, A.hi / 2 + 1);
            for (int k = A.first; k <= A.hi; k++) {
                for (int j = A.lo; j <= k; j++)
                    if (k % j == 0) A.divs[k - A.first] |= 1u << j;
                A.tab[k - A.first] = pats + ((size_t)2 << PAT_MAX_D) + ((size_t)1 << k);
            }
        }
        hipLaunchKernelGGL(k_mark, dim3((unsigned)std::min<u64>(bm, 2048), ny), dim3(MK_T), 0, 0, g,
                           (unsigned long long *)dbest, heavy, hcount);
        if (stats) GF2T_HIP(hipEventRecord(ev[d][2], 0));
        if (periods) {
            const u64 n = ((u64)1 << A.hi) / 1024;
            hipLaunchKernelGGL(k_fold_periods,
                               dim3((unsigned)std::max<u64>(1, n), (unsigned)(A.hi - A.first + 1)),
                               dim3(256), 0, 0, A);
            const u32 per = (u32)std::min<u64>(16, smax / (SW_T * 2048) + 1);
            hipLaunchKernelGGL(k_sweep, dim3((unsigned)((smax + SW_T * per - 1) / (SW_T * per))),
                               dim3(SW_T), 0, 0, A, smax, per, (unsigned long long *)dbest);
        }
        hipLaunchKernelGGL(k_mark_heavy, dim3(64, 16), dim3(256), 0, 0, heavy, hcount, 0u, smax,
                           (unsigned long long *)dbest);
        if (e < dmax)   // the next group's heavy queue
            hipLaunchKernelGGL(k_fill_u32, dim3(1), dim3(64), 0, 0, (unsigned *)hcount, (u64)2, 0u);
        if (stats) GF2T_HIP(hipEventRecord(ev[d][3], 0));
        GF2T_CHECK_LAUNCH("sieve degrees");
        d = e + 1;
    }
    unsigned long long h[33 * CN_N];
    GF2T_HIP(hipMemcpy(h, cnt, sizeof(h), hipMemcpyDeviceToHost));
    for (int d = dmin; d <= dmax; d++) {
        const unsigned long long *c = h + d * CN_N;
        const SieveDeg &P = degs[d];
        if (c[CN_SURV] != P.ncls) {
            gf2t::set_error("gf2t_sieve: d=%d: %llu classes, expected %llu", d, c[CN_SURV],
                            (unsigned long long)P.ncls);
            return GF2T_EINTERNAL;
        }
        if (c[CN_BAD]) {
            gf2t::set_error("gf2t_sieve: d=%d: %s", d,
                            (c[CN_BAD] & 1) ? "minimal polynomial not over GF(2)"
                                            : "heavy queue overflow");
            return GF2T_EINTERNAL;
        }
    }
    if (!stats) return status;
    for (int d = dmin; d <= dmax;) {   // degrees that ran together share the time by their size
        const int f = d, e = group_end(d, dmax);
        float ms[3];
        for (int i = 0; i < 3; i++) GF2T_HIP(hipEventElapsedTime(&ms[i], ev[f][i], ev[f][i + 1]));
        for (; d <= e; d++) {
            gf2t_sieve_stats &S = stats[d];
            const float part = (float)((double)((u64)1 << d) / (double)(((u64)2 << e) - ((u64)1 << f)));
            S.d = d;
            S.q = degs[d].q;
            S.classes = h[d * CN_N + CN_SURV];
            S.marking = h[d * CN_N + CN_QUEUE];
            S.heavy = h[d * CN_N + CN_HEAVY];
            S.ms_table = ms[0] * part;
            S.ms_classes = ms[1] * part;
            S.ms_heavy = ms[2] * part;
        }
    }
    return status;
}

// slices of the degree-d log table: the whole table up to W_DENSE_D, then
// the fewest slices that keep a slice at 2^W_DENSE_D values; at least
// g_min_slices (a test knob, gf2t_tune "sieve_slices")
int g_min_slices = 1;
int g_wide_from = 33;   // first degree of the 64-bit path (gf2t_tune "sieve_wide_from")
int slices_for(int d) {
    int n = d > W_DENSE_D ? 1 << (d - W_DENSE_D) : 1;
    while (n < g_min_slices && n < 256) n <<= 1;
    return n;
}

// the tables of the 64-bit path up to degree dmax (one slice's worth)
int wide_mem(int dmax) {
    SieveWork &W = *g_sw;
    int rc;
    const u64 N = (u64)1 << std::min(dmax, W_DENSE_D);          // values per slice, at most
    if ((rc = W.wP1.ensure(N * 8))) return rc;
    if ((rc = W.wTmp.ensure((((u64)1 << dmax) >> W_B1) * 8))) return rc;   // one level-1 bucket
    if ((rc = W.wLlo.ensure(N * 4))) return rc;
    if ((rc = W.wLhi.ensure(N / 2))) return rc;
    if ((rc = W.wTab.ensure(2 * ((size_t)1 << W_AB) * 8))) return rc;
    // cursors: 256 level-1 buckets, then one per level-2 bucket of a
    // level-1 bucket (2^(d - 8 - 15) at the largest d)
    const size_t n2 = (size_t)1 << std::max(0, dmax - W_B1 - W_SB);
    if ((rc = W.wCur.ensure((256 + n2) * 4))) return rc;
    if ((rc = W.bHeavy.ensure((size_t)HEAVY_CAP * sizeof(Heavy)))) return rc;
    if ((rc = W.bCnt.ensure(34 * CN_N * 8))) return rc;
    return GF2T_OK;
}

int sieve_wide(uint64_t r, int dmin, int dmax, uint64_t smax, uint64_t *dbest,
               gf2t_sieve_stats *stats) {
    SieveWork &W = *g_sw;
    int rc;
    if ((rc = wide_mem(dmax))) return rc;
    static std::once_flag lds_once;
    static hipError_t lds_err = hipSuccess;
    const int place_lds = (int)((((size_t)1 << W_SB) + ((size_t)1 << W_SB) / 8) * sizeof(u32));
    std::call_once(lds_once, [place_lds] {
        lds_err = hipFuncSetAttribute((const void *)k_w_place,
                                      hipFuncAttributeMaxDynamicSharedMemorySize, place_lds);
    });
    GF2T_HIP(lds_err);
    unsigned long long *cnt64 = (unsigned long long *)W.bCnt.p;
    unsigned *cnt32 = (unsigned *)((char *)W.bCnt.p + 32);
    unsigned *cur1 = (unsigned *)W.wCur.p, *cur2 = cur1 + 256;
    unsigned long long *P1 = (unsigned long long *)W.wP1.p, *tmp = (unsigned long long *)W.wTmp.p;
    u32 *Llo = (u32 *)W.wLlo.p, *Lhi = (u32 *)W.wLhi.p;
    u64 *A0 = (u64 *)W.wTab.p, *A1 = A0 + ((size_t)1 << W_AB);
    Heavy *heavy = (Heavy *)W.bHeavy.p;
    constexpr int MAX_SL = 16;
    hipEvent_t ev[4 + 2 * MAX_SL];
    for (auto &e : ev) GF2T_HIP(hipEventCreate(&e));
    struct Destroy {
        hipEvent_t *e;
        int n;
        ~Destroy() {
            for (int i = 0; i < n; i++) hipEventDestroy(e[i]);
        }
    } destroy{ev, 4 + 2 * MAX_SL};
    int status = GF2T_OK;
    for (int d = dmin; d <= dmax && status == GF2T_OK; d++) {
        const u64 M = ((u64)1 << d) - 1;
        const WideHost &H = wide_host(d);
        const u64 q = H.q, rmod = r % M;
        const int nsl = slices_for(d);
        if (d - W_B1 - W_SB < 2 || nsl > MAX_SL || 256 % nsl) {
            gf2t::set_error("gf2t_sieve: d=%d: the 64-bit path needs d >= 25 and at most %d "
                            "slices", d, MAX_SL);
            status = GF2T_EINVAL;
            break;
        }
        if (!q || gcd_host(rmod ? rmod : M, M) != 1) {
            gf2t::set_error("gf2t_sieve: d=%d: gcd(r, 2^d-1) != 1, unsupported r", d);
            status = GF2T_EINVAL;
            break;
        }
        if (!H.trace_ok) {
            gf2t::set_error("gf2t_sieve: d=%d: trace not in GF(2)", d);
            status = GF2T_EINTERNAL;
            break;
        }
        GF2T_HIP(hipMemcpy(A0, H.a0.data(), H.a0.size() * 8, hipMemcpyHostToDevice));
        GF2T_HIP(hipMemcpy(A1, H.a1.data(), H.a1.size() * 8, hipMemcpyHostToDevice));
        WParams P{d, M, q, rmod, smax, H.tmask, A0, A1};
        const u64 ncls = irreducible_count(d);
        const u64 qcap = ncls / 16 + 65536;
        if ((rc = W.wSurv.ensure((ncls + 64) * 8))) { status = rc; break; }
        if ((rc = W.wQueue.ensure(qcap * sizeof(MarkRecW)))) { status = rc; break; }
        u64 *surv = (u64 *)W.wSurv.p;
        MarkRecW *queue = (MarkRecW *)W.wQueue.p;

        // the classes (Lyndon words) first: every slice resolves its share
        hipLaunchKernelGGL(k_zero_counters, dim3(1), dim3(64), 0, 0, cnt64, cnt32);
        GF2T_HIP(hipEventRecord(ev[0], 0));
        hipLaunchKernelGGL(k_lyndon_t<u64>, dim3(lyndon_blocks(d)), dim3(LY_T), 0, 0, d, M, surv,
                           cnt64, (u64)(ncls + 64));
        GF2T_CHECK_LAUNCH("k_lyndon_w");
        unsigned long long hs[2];
        GF2T_HIP(hipMemcpy(hs, cnt64, 16, hipMemcpyDeviceToHost));
        const u64 nsurv = hs[0];
        if (nsurv != ncls) {
            gf2t::set_error("gf2t_sieve: d=%d: %llu classes, expected %llu", d,
                            (unsigned long long)nsurv, (unsigned long long)ncls);
            status = GF2T_EINTERNAL;
            break;
        }
        GF2T_HIP(hipEventRecord(ev[1], 0));
        const int nb = 256 / nsl;
        const u64 cap1 = (u64)1 << (d - W_B1);                 // values per level-1 bucket
        const int B2 = d - W_B1 - W_SB, B2a = (B2 + 1) / 2, B2b = B2 - B2a;
        if ((1 << B2a) > WS_MAXB || W.wCur.bytes < (256 + ((size_t)1 << B2)) * 4) {
            gf2t::set_error("gf2t_sieve: d=%d: level-2 split of %d bits beyond the cursor or "
                            "digit tables", d, B2);
            status = GF2T_EINTERNAL;
            break;
        }
        const u64 capA = cap1 >> B2a;
        const u64 zb = std::min<u64>((nsurv + (u64)ZC_T * ZC_PER - 1) / ((u64)ZC_T * ZC_PER),
                                     1u << 16);
        for (int sl = 0; sl < nsl && status == GF2T_OK; sl++) {
            const unsigned b0 = (unsigned)(sl * nb);
            GF2T_HIP(hipEventRecord(ev[4 + 2 * sl], 0));
            // log table slice: partition pass 1 (this slice's buckets),
            // level-2 split per bucket, placement
            hipLaunchKernelGGL(k_fill_u32, dim3(1), dim3(256), 0, 0, cur1, (u64)256, 0u);
            hipLaunchKernelGGL(k_w_part1, dim3((unsigned)((M + W_E - 1) / W_E)), dim3(W_T), 0, 0,
                               P, P1, cur1, cnt32 + 1, b0, (unsigned)nb);
            GF2T_CHECK_LAUNCH("k_w_part1");
            // level 2 per level-1 bucket: bucket -> scratch by the high half
            // of the level-2 bits, scratch -> bucket by the low half
            for (unsigned b1 = b0; b1 < b0 + (unsigned)nb; b1++) {
                const u64 count = b1 ? cap1 : cap1 - 1;   // value 0 never occurs
                unsigned long long *bk = P1 + (u64)(b1 - b0) * cap1;
                hipLaunchKernelGGL(k_fill_u32, dim3(1), dim3(256), 0, 0, cur2, (u64)(1u << B2a), 0u);
                hipLaunchKernelGGL(k_w_split, dim3((unsigned)((count + W_E - 1) / W_E), 1),
                                   dim3(WS_T), 0, 0, bk, cap1, count, W_SB + B2b, B2a, tmp, capA,
                                   cur2, cnt32 + 1);
                hipLaunchKernelGGL(k_fill_u32, dim3((unsigned)(((1u << B2) + 255) / 256)),
                                   dim3(256), 0, 0, cur2, (u64)(1u << B2), 0u);
                hipLaunchKernelGGL(k_w_split, dim3((unsigned)((capA + W_E - 1) / W_E), 1u << B2a),
                                   dim3(WS_T), 0, 0, tmp, capA, b1 ? capA : capA - 1, W_SB, B2b,
                                   bk, (u64)1 << W_SB, cur2, cnt32 + 1);
            }
            GF2T_CHECK_LAUNCH("k_w_split");
            hipLaunchKernelGGL(k_w_place, dim3((unsigned)(((u64)nb * cap1) >> W_SB)), dim3(1024),
                               (size_t)place_lds, 0, P1, Llo, Lhi, sl == 0 ? 1 : 0);
            GF2T_CHECK_LAUNCH("k_w_place");
            GF2T_HIP(hipEventRecord(ev[5 + 2 * sl], 0));
            unsigned chk[2];
            GF2T_HIP(hipMemcpy(chk, cnt32, 8, hipMemcpyDeviceToHost));
            if (chk[1]) {
                gf2t::set_error("gf2t_sieve: d=%d: log table partition overflow", d);
                status = GF2T_EINTERNAL;
                break;
            }
            hipLaunchKernelGGL(k_zech_w, dim3((unsigned)zb), dim3(ZC_T), 0, 0, P, surv, nsurv, Llo,
                               Lhi, queue, cnt64 + 1, qcap, (u64)b0 * cap1, (u64)nb * cap1);
            GF2T_CHECK_LAUNCH("k_zech_w");
        }
        if (status != GF2T_OK) break;
        GF2T_HIP(hipMemcpy(hs, cnt64, 16, hipMemcpyDeviceToHost));
        if (hs[1] > qcap) {
            gf2t::set_error("gf2t_sieve: d=%d: marking queue overflow (%llu)", d,
                            (unsigned long long)hs[1]);
            status = GF2T_EINTERNAL;
            break;
        }
        const u64 nq = hs[1];
        if (nq) {
            hipLaunchKernelGGL(k_mark_w, dim3((unsigned)((nq + 255) / 256)), dim3(256), 0, 0, P,
                               queue, nq, (unsigned long long *)dbest, heavy, cnt32, cnt32 + 1);
            GF2T_CHECK_LAUNCH("k_mark_w");
        }
        GF2T_HIP(hipEventRecord(ev[2], 0));
        unsigned h32[2];
        GF2T_HIP(hipMemcpy(h32, cnt32, 8, hipMemcpyDeviceToHost));
        if (h32[1]) {
            gf2t::set_error("gf2t_sieve: d=%d: %s", d,
                            (h32[1] & 1) ? "minimal polynomial not over GF(2)"
                                         : "heavy queue overflow");
            status = GF2T_EINTERNAL;
            break;
        }
        const unsigned nheavy = h32[0];
        if (nheavy) {
            unsigned gy = nheavy < 65535 ? nheavy : 65535;
            hipLaunchKernelGGL(k_mark_heavy, dim3(64, gy), dim3(256), 0, 0, heavy, nullptr, nheavy,
                               smax, (unsigned long long *)dbest);
            GF2T_CHECK_LAUNCH("k_mark_heavy");
        }
        GF2T_HIP(hipEventRecord(ev[3], 0));
        GF2T_HIP(hipEventSynchronize(ev[3]));
        if (stats) {
            gf2t_sieve_stats &S = stats[d];
            S.d = d;
            S.q = q;
            S.classes = nsurv;
            S.marking = nq;
            S.heavy = nheavy;
            // table: the slices' builds; classes: the rest up to marking
            float tab = 0, all = 0, x;
            for (int sl = 0; sl < nsl; sl++) {
                GF2T_HIP(hipEventElapsedTime(&x, ev[4 + 2 * sl], ev[5 + 2 * sl]));
                tab += x;
            }
            GF2T_HIP(hipEventElapsedTime(&all, ev[0], ev[2]));
            S.ms_table = tab;
            S.ms_classes = all - tab;
            GF2T_HIP(hipEventElapsedTime(&S.ms_heavy, ev[2], ev[3]));
        }
    }
    return status;
}
}  // namespace

// gf2t_tune keys of the sieve (test knobs): "sieve_wide_from" = first
// degree of the 64-bit path (25..33, default 33), "sieve_slices" = least
// number of log-table slices (1..16, a power of two)
int gf2t_sieve_tune(const char *key, int64_t v) {
    std::lock_guard<std::mutex> lk(g_sw_mu);
    if (!strcmp(key, "sieve_wide_from") && v >= 25 && v <= 33) {
        g_wide_from = (int)v;
        return GF2T_OK;
    }
    if (!strcmp(key, "sieve_slices") && v >= 1 && v <= 16 && !(v & (v - 1))) {
        g_min_slices = (int)v;
        return GF2T_OK;
    }
    gf2t::set_error("gf2t_tune: %s needs 25..33 (sieve_wide_from) or a power of two 1..16 "
                    "(sieve_slices)", key);
    return GF2T_EINVAL;
}
int gf2t_sieve_tune_get(const char *key, int64_t *v) {
    std::lock_guard<std::mutex> lk(g_sw_mu);
    if (!strcmp(key, "sieve_wide_from")) { *v = g_wide_from; return GF2T_OK; }
    if (!strcmp(key, "sieve_slices")) { *v = g_min_slices; return GF2T_OK; }
    return GF2T_EINVAL;
}

extern "C" int gf2t_sieve(uint64_t r, int dmin, int dmax, uint64_t smax, uint64_t *dbest,
                          gf2t_sieve_stats *stats) {
    if (dmin < 2) dmin = 2;
    if (dmax > WIDE_MAX_D || dmin > dmax || !dbest || smax < 1) {
        gf2t::set_error("gf2t_sieve: need 2 <= dmin <= dmax <= %d, smax >= 1, dbest",
                        WIDE_MAX_D);
        return GF2T_EINVAL;
    }
    // device tables stay allocated between calls (grow-only; freed by
    // gf2t_sieve_release), so repeated sieves pay no allocation
    std::lock_guard<std::mutex> lk(g_sw_mu);
    if (!g_sw) g_sw = new SieveWork();
    int status = GF2T_OK;
    const int wf = g_wide_from;
    if (dmax >= 33) {
        // the degree-<=32 arrays live inside the wide tables from here on
        g_sw->bClass.release();
        status = wide_mem(dmax);
    }
    if (status == GF2T_OK && dmin < wf)
        status = sieve_narrow(r, dmin, std::min(dmax, wf - 1), smax, dbest, stats);
    if (status == GF2T_OK && dmax >= wf)
        status = sieve_wide(r, std::max(dmin, wf), dmax, smax, dbest, stats);
    return status;
}
