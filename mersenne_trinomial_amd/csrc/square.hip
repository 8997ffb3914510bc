// square.hip -- (b) squaring + trinomial fold on gfx950.
//
// F <- F^2 mod T, T = x^r + x^s + 1, 1 <= s, 2s < r.  Squaring over GF(2)
// is the bit spread SP (SP[2k] = F bit k, SP[odd] = 0); the fold
// x^e -> x^(e-r) + x^(e-r+s) applied twice reduces SP (degree <= 2r-2)
// to r bits.  Writing SP = L + x^r H, H = H_lo + x^(r-s) H_hi:
//   F^2 mod T = SP[0,r) + SP[r,2r-1)>>r + SP[r,2r-s)>>(r-s)
//             + SP[2r-s,2r-1)>>(2r-s) + SP[2r-s,2r-1)>>(2r-2s)
// (the same five windows as the reference's fused kernel,
// src/tsfactor.cu:128-186).  Each output word is written by exactly one
// lane (gather form), so there are no write races.
//
// Mapping: one lane produces one 128-bit output pair (two words) from
// 64-bit input windows; waves cover 64 consecutive pairs = 1 KiB of
// output, so stores and the dominant loads are fully coalesced.  Per
// residue-step the kernel moves 16*nw algorithmic bytes (read F, write
// F^2); the second read of the upper input half by window 3 hits in
// L2 / Infinity Cache.
#include "gf2t_internal.hpp"
#include "host_poly.hpp"
#include "../../include/gf2t.h"
#include <vector>
#include <algorithm>
#include <numeric>
#include <cstring>
#include <cstdlib>
#include <atomic>
#include <mutex>
#include <new>

namespace {

constexpr int SQ_THREADS = 256;

// W12 (template argument of the squaring kernels): the window words are
// read as one 12-byte load; the host sets it when no residue of the launch
// has r a multiple of 64 (sq_w12_ok)
template <bool W12>
__global__ __launch_bounds__(SQ_THREADS) void k_square_fold(
        const u64 *__restrict__ in, u64 *__restrict__ out, const SqConst c) {
    size_t i = (size_t)blockIdx.x * SQ_THREADS + threadIdx.x;
    if (i >= (c.nw + 1) / 2) return;
    u64 o0, o1;
    square_fold_pair_fast<W12>(in, c, i, o0, o1);
    out[2 * i] = o0;
    if (2 * i + 1 < c.nw) out[2 * i + 1] = o1;
}

__device__ __forceinline__ u32 uniform32(u32 v) { return __builtin_amdgcn_readfirstlane(v); }

struct SqDesc {
    const u64 *in;
    u64 *out;
    SqConst c;
    int m;              // squarings of the first launch; the others take two or three
    int back;           // the chain ends in the scratch buffer (in, of an odd launch)
    const int *order;   // block -> tile (-1 idle), or null for identity
    Sq2Chain h;         // two-squaring tile layout
    PowOrder p;         // order of the ranges of F^8 windows
};

// output pair i (one 16-byte store when both words exist)
template <bool NT>
__device__ __forceinline__ void store_pair(u64 *out_, size_t nw, size_t i, u64 o0, u64 o1) {
    typedef u64 v2u __attribute__((ext_vector_type(2)));
    GF2T_GLOBAL u64 *out = (GF2T_GLOBAL u64 *)out_;
    if (2 * i + 1 < nw) {
        GF2T_GLOBAL v2u *p = (GF2T_GLOBAL v2u *)(out + 2 * i);
        if (NT) __builtin_nontemporal_store(v2u{o0, o1}, p);
        else *p = v2u{o0, o1};
    } else {
        if (NT) __builtin_nontemporal_store(o0, out + 2 * i);
        else out[2 * i] = o0;
    }
}

// batched: blockIdx.y selects the residue, blockIdx.x a tile of
// SQ_THREADS*PPT output pairs (pairs j*SQ_THREADS + lane for j < PPT)
template <int PPT, bool NT, bool W12>
__global__ __launch_bounds__(SQ_THREADS) void k_square_fold_batch(
        const SqDesc *__restrict__ desc) {
    const SqDesc d = desc[blockIdx.y];
    int t = (int)blockIdx.x;
    if (d.order) {
        t = __builtin_amdgcn_readfirstlane(d.order[blockIdx.x]);   // one value per block
        if (t < 0) return;
    }
    const size_t np = (d.c.nw + 1) / 2;
    const size_t t0 = (size_t)t * SQ_THREADS * PPT;
    if (t0 >= np) return;
    // one region for the whole tile (all but a few tiles per residue)
    const int treg = sq_tile_region(d.c, t0, t0 + SQ_THREADS * PPT < np ? t0 + SQ_THREADS * PPT : np);
    const SqArrayT<W12> src{d.in, d.c.nw};
    // streaming stores: F^2 is not re-read before the next launch (one
    // 16-byte store per pair; residue buffers are 16-byte aligned)
    if (treg < 3) {
        sq_variant(treg, d.c, [&](auto v) {
#pragma unroll
            for (int j = 0; j < PPT; j++) {
                const size_t i = t0 + (size_t)j * SQ_THREADS + threadIdx.x;
                if (i < np) {
                    u64 o0, o1;
                    v.pair(src, d.c, (u32)i, o0, o1);
                    store_pair<NT>(d.out, d.c.nw, i, o0, o1);
                }
            }
        });
    } else {
        for (int j = 0; j < PPT; j++) {
            const size_t i = t0 + (size_t)j * SQ_THREADS + threadIdx.x;
            if (i < np) {
                u64 o0, o1;
                square_fold_pair_masked(src, d.c, i, o0, o1);
                store_pair<NT>(d.out, d.c.nw, i, o0, o1);
            }
        }
    }
}

// ---- two squarings per launch: H = (F^2)^2 mod T
// One tile, the output pairs [i0, i1) (at most SQ2_TP): the G phase forms
// the windows of pl.compute, one G pair per thread and window, into the
// plan's LDS slots; the H phase then reads G through the window copies of
// the plan.  Only the loads of windows 1 and 2, which every tile forms, go
// first; the others are loaded as they are formed, which keeps the
// work-unit loop at 53 VGPRs (8 waves per SIMD) where loading every window
// first needs 84 -- and gains nothing where tiles are few either (the 12
// tiles of a 756839-bit residue: 176 us either way for 40 squarings).
template <bool NT, bool W12>
__device__ __forceinline__ void square2_run(const u64 *__restrict__ in, u64 *__restrict__ out,
                                            const SqConst &c, size_t i0, size_t i1, int treg,
                                            const Sq2Plan &pl, u64 *gw) {
    static_assert(SQ_THREADS == SQ2_GP && 2 * SQ_THREADS >= SQ2_TP + 7, "tile shape");
    typedef u64 v2u __attribute__((ext_vector_type(2)));
    const SqArrayT<W12> fsrc{in, c.nw};
    int greg[SQ2_WINS];
    SqRawPair raw[SQ2_WINS];
#pragma unroll
    for (int k = 0; k < SQ2_WINS; k++) {
        const u64 p0 = pl.base[k] >> 1;
        greg[k] = ((pl.compute >> k) & 1) ? sq_tile_region(c, p0, p0 + SQ2_GP) : -1;
    }
#pragma unroll
    for (int k = 0; k < 2; k++)
        if (greg[k] >= 0 && greg[k] < 3)
            raw[k] = sq_raw_pair(fsrc, c, (u32)((pl.base[k] >> 1) + threadIdx.x), greg[k]);
#pragma unroll
    for (int k = 0; k < SQ2_WINS; k++) {
        if (greg[k] < 0) continue;
        u64 o0, o1;
        if (greg[k] < 3) {
            if (k >= 2)
                raw[k] = sq_raw_pair(fsrc, c, (u32)((pl.base[k] >> 1) + threadIdx.x), greg[k]);
            sq_combine_pair(raw[k], c, greg[k], o0, o1);
        } else {
            sq2_g_pair_clipped(fsrc, c, (pl.base[k] >> 1) + threadIdx.x, o0, o1);
        }
        *(v2u *)(gw + pl.at[k] + 2 * threadIdx.x) = v2u{o0, o1};
    }
    __syncthreads();
    const Sq2Tile src = sq2_tile(gw, pl);
    // pair slots from i0 rounded down to a 128-byte line: each wave stores
    // whole lines (non-temporal stores of part of a line go to memory
    // as partial writes); the slots below i0 idle
    const size_t ib = i0 & ~(size_t)7;
    if (treg < 3) {
        sq_variant(treg, c, [&](auto v) {
            for (int j = 0; j < 2; j++) {
                const size_t i = ib + (size_t)j * SQ_THREADS + threadIdx.x;
                if (i >= i0 && i < i1) {
                    u64 o0, o1;
                    v.pair(src, c, (u32)i, o0, o1);
                    store_pair<NT>(out, c.nw, i, o0, o1);
                }
            }
        });
    } else {
        for (int j = 0; j < 2; j++) {
            const size_t i = ib + (size_t)j * SQ_THREADS + threadIdx.x;
            if (i >= i0 && i < i1) {
                u64 o0, o1;
                square_fold_pair_masked(src, c, i, o0, o1);
                store_pair<NT>(out, c.nw, i, o0, o1);
            }
        }
    }
}
// the plain tile number `tile` (pairs from tile * SQ2_TP on)
template <bool NT, bool W12>
__device__ __forceinline__ void square2_tile(const u64 *__restrict__ in, u64 *__restrict__ out,
                                             const SqConst &c, size_t tile, u64 *gw) {
    const size_t np = (c.nw + 1) / 2;
    const size_t i0 = tile * SQ2_TP;
    if (i0 >= np) return;   // whole block
    const size_t i1 = i0 + SQ2_TP < np ? i0 + SQ2_TP : np;
    const int treg = sq_tile_region(c, i0, i1);
    square2_run<NT, W12>(in, out, c, i0, i1, treg, sq2_plan(c, i0, sq2_need(treg)), gw);
}
// work unit u: its tiles one after another, each taking windows 3 and 5
// from the copies of the tile before it where the plan says so
template <bool NT, bool W12>
__device__ __forceinline__ void square2_unit(const u64 *__restrict__ in, u64 *__restrict__ out,
                                             const SqConst &c, const Sq2Chain &h, u32 u,
                                             u64 *gw) {
    Sq2Unit w;
    if (!sq2_unit(h, u, w)) return;   // whole block
    u32 prev_need = 0, prev_base4 = 0;
    for (u32 j = w.j0; j < w.j1; j++) {
        if (j > w.j0) __syncthreads();   // the previous H phase is done with the slots
        const u32 i0 = w.start + j * h.period;
        const u32 i1 = i0 + w.width < h.np ? i0 + w.width : h.np;
        const int treg = sq_tile_region(c, i0, i1);
        const u32 need = sq2_need(treg);
        const Sq2Plan pl = sq2_chain_plan(c, h, i0, w.width, need, j - w.j0, prev_need, prev_base4);
        square2_run<NT, W12>(in, out, c, i0, i1, treg, pl, gw);
        prev_need = need;
        prev_base4 = pl.base[3];
    }
}

// batched: blockIdx.y selects the residue, blockIdx.x the work unit.
// Eight waves per SIMD (106 SGPRs would allow seven; 23 of them then live
// in VGPR lanes, no scratch): about 2% faster per launch.
template <bool NT, bool W12>
__global__ __launch_bounds__(SQ_THREADS) __attribute__((amdgpu_waves_per_eu(8))) void
k_square2_fold_batch(
        const SqDesc *__restrict__ desc) {
    __shared__ __align__(16) u64 gw[SQ2_WINS * SQ2_LEN];
    const SqDesc d = desc[blockIdx.y];
    square2_unit<NT, W12>(d.in, d.out, d.c, d.h, blockIdx.x, gw);
}
// The same, and the residues with m = 1 advance by one squaring: the first
// launch of a batch whose chains differ in length, so that every later one
// advances all of its chains by two.
template <bool NT, bool W12>
__global__ __launch_bounds__(SQ_THREADS) void k_square12_fold_batch(
        const SqDesc *__restrict__ desc) {
    __shared__ __align__(16) u64 gw[SQ2_WINS * SQ2_LEN];
    const SqDesc d = desc[blockIdx.y];
    if (d.m == 2) {
        square2_unit<NT, W12>(d.in, d.out, d.c, d.h, blockIdx.x, gw);
        return;
    }
    for (u32 i = blockIdx.x * SQ_THREADS + threadIdx.x; i < d.h.np; i += gridDim.x * SQ_THREADS) {
        u64 o0, o1;
        square_fold_pair_fast<W12>(d.in, d.c, i, o0, o1);
        store_pair<NT>(d.out, d.c.nw, i, o0, o1);
    }
}

// ---- F^8 by direct windows: three squarings per launch
// A block takes a range of units of 2^M words of 32 output bits.  Its list
// of windows (pow_window: about 31 for M = 3, their shifts uniform) is
// sorted by class and dealt to its waves in equal parts -- by class the
// fullest wave had 7 of them -- and what a wave has of a class is XORed
// into that class's words in LDS, which are then merged.  For three
// squarings that is 216 VALU operations a pair of words in all, the list
// among them (0.5 per cycle per CU: not the issue limit), where a tile of the
// two-squaring kernel takes 174 for two and copies in LDS; but a tile reads
// each word about once, this about four times, from the caches while they
// hold the launch's residues: three squarings take 4.2 us where one launch
// is all latency (756839 bits; two took 9), 14 us for one full-size residue
// (two: 16), 92 us for 8 (two: 74) and 800 us for 64 (two: 455).  Past the
// 256 MiB cache, which eight full-size residues and their copies fill, two
// at a time are faster: 12 squarings of 8, 9, 16 and 32 of them take 396,
// 497, 871 and 1712 us by three and 469, 460, 729 and 1370 by two, 24 of 24
// and 26 residues of 44,497,001 bits 724 and 916 by three and 860 of the 26
// by two.  (Residues small enough to run in rows, 13,466,917 bits, keep the
// threes faster a little longer: 96 of them 874 us against 970.)
constexpr int PW_T = 512, PW_LIST = 128;
template <int M, int U>
constexpr u32 pw_units() { return 64u * U * (8 >> M); }
// LDS word of unit x of a class, a range having `units`: with four units
// per lane, by their place in the four and padded, so that neither the
// lanes' XORs nor the merge's reads meet in a bank
template <int U>
__device__ __forceinline__ u32 pw_word(u32 x) {
    return U == 4 ? (x >> 8) * 320 + (x & 3) * 80 + ((x & 255) >> 2) : x;
}
template <int M, int U>
constexpr u32 pw_class_words() { return U == 4 ? pw_units<M, U>() / 256 * 320 : pw_units<M, U>(); }
template <int M, int U>
__device__ __forceinline__ void power_range(const u64 *__restrict__ in, u64 *__restrict__ out,
                                            const SqConst &c, u32 blk, u32 *lds) {
    typedef u32 v2u __attribute__((ext_vector_type(2), aligned(4)));
    typedef u32 v4u __attribute__((ext_vector_type(4)));
    typedef u32 v4a __attribute__((ext_vector_type(4), aligned(4)));
    static_assert(U == 1 || U == 4, "units per lane");
    constexpr int NC = 1 << M;
    constexpr u32 UB = pw_units<M, U>(), UC = pw_class_words<M, U>();
    const u32 nd = 2 * (u32)c.nw, i0 = blk * UB;
    if ((u64)i0 * NC >= nd) return;   // whole block
    u32 *acc = lds, *lk = lds + UC * NC, *li = lk + PW_LIST;
    int *lo = (int *)(li + PW_LIST), *hi = lo + PW_LIST;
    u32 *cnt = (u32 *)(hi + PW_LIST);   // [class], [8 + class]: whole, masked
    if (threadIdx.x < 16) cnt[threadIdx.x] = 0;
    for (u32 x = threadIdx.x; x < UC * NC; x += PW_T) acc[x] = 0;
    __syncthreads();
    PowWin w;
    u32 rank = 0;
    const bool got = threadIdx.x < 256 &&
                     pow_window<M>(c.r, c.s, threadIdx.x >> 4, threadIdx.x & 15, (u64)i0 * NC * 32,
                                   ((u64)i0 + UB) * NC * 32, w);
    if (got) rank = atomicAdd(&cnt[w.cls + (w.part ? 8 : 0)], 1u);
    __syncthreads();
    u32 before = 0, nfull = 0, npart = 0;   // before this thread's pair in the list
#pragma unroll
    for (int k = 0; k < NC; k++) {
        const u32 f = cnt[k], m = cnt[8 + k];
        nfull += f;
        npart += m;
        if (got && k < (int)w.cls) before += w.part ? m : f;
    }
    if (got) {
        const u32 at = before + rank + (w.part ? nfull : 0);
        lk[at] = w.kw;
        li[at] = w.sh | w.cls << 8;
        lo[at] = w.lo;
        hi[at] = w.hi;
    }
    __syncthreads();
    nfull = uniform32(nfull);
    npart = uniform32(npart);
    const int lane = threadIdx.x & 63, wave = uniform32(threadIdx.x >> 6);
    const u32 part = wave & (NC - 1), group = wave >> M;   // the waves of a group share its units
    const u32 ub = i0 + group * 64 * U;
    const GF2T_GLOBAL u32 *f = (const GF2T_GLOBAL u32 *)in;
    u32 A[U];
#pragma unroll
    for (int u = 0; u < U; u++) A[u] = 0;
    u32 cls = 0;
    auto flush = [&](u32 next) {   // A into class cls's words
#pragma unroll
        for (int u = 0; u < U; u++) {
            atomicXor(&acc[cls * UC + pw_word<U>(group * 64 * U + (U == 4 ? 4 * lane + u : lane))], A[u]);
            A[u] = 0;
        }
        cls = next;
    };
    const u32 f0 = part * nfull / NC, n = (part + 1) * nfull / NC - f0;   // at most 16
    const u32 ek = lane < (int)n ? lk[f0 + lane] : 0, es = lane < (int)n ? li[f0 + lane] : 0;
    constexpr int Q = 4;   // windows whose loads are in flight together
    for (u32 q = 0; q < n; q += Q) {
        v4u x[Q];
        u32 y[Q], e[Q];
#pragma unroll
        for (int t = 0; t < Q; t++) {
            if (q + t >= n) break;
            e[t] = __builtin_amdgcn_readlane(es, (int)(q + t));
            const GF2T_GLOBAL u32 *p = f + (size_t)ub + (u32)__builtin_amdgcn_readlane(ek, (int)(q + t));
            // (of a window that ends on a word, the word after may lie
            // past the residue)
            const bool over = (e[t] & 31) != 0;
            y[t] = 0;
            if (U == 4) {
                x[t] = *(const GF2T_GLOBAL v4a *)(p + 4 * lane);
                if (over && lane == 63) y[t] = p[256];
            } else if (over) {
                const v2u v = *(const GF2T_GLOBAL v2u *)(p + lane);
                x[t].x = v.x;
                y[t] = v.y;
            } else {
                x[t].x = p[lane];
            }
        }
#pragma unroll
        for (int t = 0; t < Q; t++) {
            if (q + t >= n) break;
            if (e[t] >> 8 != cls) flush(e[t] >> 8);
            const u32 sh = e[t] & 31;
            const v4u v = x[t];
            if (U == 4) {
                // the next lane's first word (wave_shl:1), lane 63's its own y
                const u32 nx = (u32)__builtin_amdgcn_update_dpp((int)y[t], (int)v.x, 0x130, 0xf, 0xf, false);
                A[0] ^= alignbit(v.y, v.x, sh);
                A[1 % U] ^= alignbit(v.z, v.y, sh);
                A[2 % U] ^= alignbit(v.w, v.z, sh);
                A[3 % U] ^= alignbit(nx, v.w, sh);
            } else {
                A[0] ^= alignbit(y[t], v.x, sh);
            }
        }
    }
    const u32 p0 = nfull + part * npart / NC, p1 = nfull + (part + 1) * npart / NC;
    for (u32 at = p0; at < p1; at++) {
        const u32 kw = uniform32(lk[at]), e = uniform32(li[at]);
        const int l = (int)uniform32((u32)lo[at]), h = (int)uniform32((u32)hi[at]);
        if (e >> 8 != cls) flush(e >> 8);
        u32 x[U], y[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const u64 j = (u64)ub + (U == 4 ? 4 * lane + u : lane) + kw;
            x[u] = f[j < nd ? (u32)j : nd - 1];
            y[u] = f[j + 1 < nd ? (u32)j + 1 : nd - 1];
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            const u32 i = ub - i0 + (U == 4 ? 4 * lane + u : lane);
            A[u] ^= alignbit(y[u], x[u], e & 31) & pow_mask<M>((int)(i * NC * 32), cls, l, h);
        }
    }
    flush(0);
    __syncthreads();
    for (u32 k = wave * 64; k < UB; k += PW_T) {
        const u32 i = i0 + k + lane;
        u32 a[NC], o[NC];
#pragma unroll
        for (int t = 0; t < NC; t++) a[t] = acc[t * UC + pw_word<U>(k + lane)];
        class_merge(a, o);
        u32 *dst = (u32 *)out + (size_t)i * NC;
        if ((u64)(i + 1) * NC <= nd) {
            if (M == 1) {
                *(u64 *)dst = ((u64)o[1] << 32) | o[0];
            } else {
#pragma unroll
                for (int t = 0; t < NC; t += 4) *(v4u *)(dst + t) = v4u{o[t], o[t + 1], o[t + 2], o[t + 3]};
            }
        } else {
#pragma unroll
            for (int t = 0; t < NC; t++)
                if ((u64)i * NC + t < nd) dst[t] = o[t];
        }
    }
}
// ranges (2^16 output bits) of a launch
inline u64 pow_ranges(size_t nw) { return (nw + 1023) / 1024; }
constexpr u64 PW_FULL = 128;    // from which a block takes a range (U = 4)
constexpr u64 PW_MOST = 16640;  // above which two squarings per launch are faster
constexpr u64 PW_SHORT = 13500;  // above which they are for some short chains
// ranges of a residue from which they run in columns: it exceeds the 4 MiB
// L2 of an XCD (12 squarings of 8 residues of 44,497,001 bits: 174 us in
// plain order, 150 us in columns; of 64 of 3,021,377 bits: 249 and 274)
constexpr u64 PW_COLS = 512;
// Squarings per launch.  Where a launch's residues and their copies no
// longer fit the 256 MiB cache, one of three squarings takes a fourth longer
// than one of two, and the copy back after an odd number of launches three
// fourths of that: chains of up to 4, 7 and 8 squarings are shorter by two
// (7 squarings of 8 residues of 136,279,841 bits: 274 us, by three 318; of 6
// residues: 224, by three 220).  two, three: the chains' costs, each times
// its residue's length.
inline u64 pow_cost(u64 steps, u64 per) {
    const u64 l = (steps + per - 1) / per;
    return (per == 3 ? 5 : 4) * l + 3 * (l & 1);
}
inline int pow_per(u64 ranges, u64 two, u64 three) {
    return ranges > PW_MOST || (ranges > PW_SHORT && two <= three) ? 2 : 3;
}
// A single squaring by windows is as long as three where residues come from
// memory: from PW_COLS ranges on the one-squaring kernels take it
// (136,279,841 bits: 19.1 us against 20.4, s = 1 17.1 against 19.7; below,
// 20,000,003 bits: 8.7 against 7.7).
inline bool pow_one(u64 ranges) { return ranges < PW_COLS; }
template <int U>
constexpr size_t pw_lds() { return (8 * pw_class_words<3, U>() + 4 * PW_LIST + 16) * 4; }

// 2^m-th powers of a residue
template <bool COLS>
__device__ __forceinline__ u32 pw_block(const PowOrder &p) {
    return COLS ? pow_range(p, blockIdx.x) : blockIdx.x;
}
template <int U, bool COLS>
__global__ __launch_bounds__(PW_T) void k_power(const u64 *__restrict__ in, u64 *__restrict__ out,
                                                const SqConst c, const PowOrder p, int m) {
    __shared__ __align__(16) u32 lds[pw_lds<U>() / 4];
    const u32 x = pw_block<COLS>(p);
    if (m == 3) power_range<3, U>(in, out, c, x, lds);
    else if (m == 2) power_range<2, U>(in, out, c, x, lds);
    else power_range<1, U>(in, out, c, x, lds);
}
// of the residues of a batch (blockIdx.y); the first launch advances each
// by d.m squarings, so that every later one takes three of all
template <int U, bool COLS, bool FIRST>
__global__ __launch_bounds__(PW_T) void k_power_batch(const SqDesc *__restrict__ desc) {
    __shared__ __align__(16) u32 lds[pw_lds<U>() / 4];
    const SqDesc &d = desc[blockIdx.y];
    const u32 x = pw_block<COLS>(d.p);
    if (!FIRST || d.m == 3) power_range<3, U>(d.in, d.out, d.c, x, lds);
    else if (d.m == 2) power_range<2, U>(d.in, d.out, d.c, x, lds);
    else power_range<1, U>(d.in, d.out, d.c, x, lds);
}
// blocks for 2^m-th powers of nw words
template <int U, bool COLS>
u64 power_blocks(size_t nw, int m, const PowOrder &p) {
    static_assert(pw_units<3, 4>() * 256 == 65536 && pw_units<1, 4>() * 64 == 65536, "PowOrder");
    if (COLS) return 8 * (u64)p.per;
    const u64 units = (2 * (u64)nw + (1u << m) - 1) >> m, ub = 64ull * U * (8 >> m);
    return (units + ub - 1) / ub;
}

// the values that ended in the scratch buffers, back to the residues: of
// the entries `in` -> `out`, those marked back (one launch instead of a
// device copy of 4 us for each)
__global__ __launch_bounds__(SQ_THREADS) void k_batch_back(const SqDesc *__restrict__ desc) {
    const SqDesc &d = desc[blockIdx.y];
    if (!d.back) return;
    typedef u64 v2u __attribute__((ext_vector_type(2)));
    const u32 n2 = (u32)(d.c.nw / 2);   // 16-byte words (buffers are 16-byte aligned)
    const v2u *in = (const v2u *)d.in;
    v2u *out = (v2u *)d.out;
    for (u32 i = blockIdx.x * SQ_THREADS + threadIdx.x; i < n2; i += gridDim.x * SQ_THREADS)
        out[i] = in[i];
    if ((d.c.nw & 1) && blockIdx.x == 0 && threadIdx.x == 0) d.out[d.c.nw - 1] = d.in[d.c.nw - 1];
}

// ---- whole chains of small residues
// A residue whose two copies fit in LDS (r up to 655,232) runs its whole
// chain in one block, one squaring per barrier, between the copies: no
// launch and no memory traffic per step.  Bounded by the issue of one
// CU and the barrier: 0.85 us per squaring at 132049 bits and 2.2 us at
// 640,000, where by launches two squarings took 9.5 us, all of it latency
// (40 squarings: 191 -> 34 us, and 183 -> 90 us).  By launches of three
// squarings 40 take about 57 us at any such size, and a few squarings less
// (6 of 262,144 bits 8.2 us against 12.4, 40 56 against 54), so residues above
// CH_ONE words go that way unless there are CH_FEW of them: a batch of 16 of
// 300,000 bits takes 63 us in LDS and 83 by launches (40 squarings, upload
// and wait among them), 16 of 640,000 135 and 120, 32 of them 136 and 173, and
// of 64 137 and 202.  512 residues of 600,000 bits are 512 blocks, one per CU
// at a time: 276 us against 1085 us.
constexpr int CH_THREADS = 1024;
constexpr size_t CH_LDS = 160 * 1024;
constexpr size_t CH_WORDS = CH_LDS / 16 - 2;   // words of a residue, at most
constexpr size_t CH_ONE = 4096;                // of a few residues, at most
constexpr int CH_FEW = 16;
constexpr u64 CH_STEPS = 4096;                 // squarings per launch, at most
struct ChainDesc {
    u64 *res;
    SqConst c;
    u64 steps;
};
struct SqLds {   // a residue's copy in LDS, two words past its end readable
    const u32 *p;
    __device__ void raw3(int, u32 q, u32, u32 &a, u32 &b, u32 &c) const {
        a = p[q];
        b = p[q + 1];
        c = p[q + 2];
    }
};
// `steps` squarings from cur, the copies changing places; K pairs per
// thread, their window addresses and masks in registers
template <int K, int RP, int SP>
__device__ __forceinline__ u64 *chain_steps(u64 *cur, u64 *oth, const SqConst &c, u32 np, u32 steps,
                                            const SqClip (&clip)[K], const u32 (&need)[K]) {
    typedef u64 v2u __attribute__((ext_vector_type(2)));
    const u32 nthr = blockDim.x, wave0 = uniform32(threadIdx.x & ~63u);
    for (u32 k = 0; k < steps; k++) {
        const SqLds src{(const u32 *)cur};
#pragma unroll
        for (int j = 0; j < K; j++) {
            if (wave0 + j * nthr >= np) break;   // whole wave
            u64 o0, o1;
            sq_pair_clipped<RP, SP>(src, c, clip[j], need[j], o0, o1);
            const u32 i = threadIdx.x + j * nthr;
            if (i < np) *(v2u *)(oth + 2 * i) = v2u{o0, o1};
        }
        __syncthreads();
        u64 *t = cur;
        cur = oth;
        oth = t;
    }
    return cur;
}
// list (or one, where list is null): one residue per block, at most
// `most` squarings of its chain from squaring number `done` on
template <int K>
__global__ __launch_bounds__(CH_THREADS) void k_square_chain(const ChainDesc *__restrict__ list,
                                                             const ChainDesc one, u64 done,
                                                             u64 most) {
    extern __shared__ __align__(16) u64 ch_lds[];
    const ChainDesc d = list ? list[blockIdx.x] : one;
    if (d.steps <= done) return;   // whole block
    const u64 left = d.steps - done;
    const u32 steps = (u32)(left < most ? left : most);
    const u32 nw = (u32)d.c.nw, np = (nw + 1) / 2, nthr = blockDim.x;
    u64 *cur = ch_lds, *oth = ch_lds + 2 * np + 2;
    for (u32 w = threadIdx.x; w < nw; w += nthr) cur[w] = d.res[w];
    SqClip clip[K];
    u32 need[K];
#pragma unroll
    for (int j = 0; j < K; j++) {
        const u32 i = threadIdx.x + j * nthr;
        clip[j] = sq_clip(d.c, i < np ? i : np);   // past the end: every mask empty
        need[j] = 0;
#pragma unroll
        for (int k = 0; k < 5; k++)
            if (__ballot((clip[j].m[k][0] | clip[j].m[k][1]) != 0)) need[j] |= 1u << k;
    }
    __syncthreads();
    switch ((int)((d.c.r & 1) << 1) + (int)(d.c.s & 1)) {
    case 0: cur = chain_steps<K, 0, 0>(cur, oth, d.c, np, steps, clip, need); break;
    case 1: cur = chain_steps<K, 0, 1>(cur, oth, d.c, np, steps, clip, need); break;
    case 2: cur = chain_steps<K, 1, 0>(cur, oth, d.c, np, steps, clip, need); break;
    default: cur = chain_steps<K, 1, 1>(cur, oth, d.c, np, steps, clip, need); break;
    }
    for (u32 w = threadIdx.x; w < nw; w += nthr) d.res[w] = cur[w];
}
template <bool W12>
__global__ __launch_bounds__(SQ_THREADS) void k_square2_fold(
        const u64 *__restrict__ in, u64 *__restrict__ out, const SqConst c, const Sq2Chain h) {
    __shared__ __align__(16) u64 gw[SQ2_WINS * SQ2_LEN];
    square2_unit<false, W12>(in, out, c, h, blockIdx.x, gw);
}

// slab of n residues (pitch words apart), residue y with s = svec[y / group],
// advanced by two squarings: the h-table step of the blocked DDF taken
// twice in one pass.  Tiles beyond the residue exit before any barrier.
__device__ __forceinline__ u64 uniform_u64(u64 v) {
    return ((u64)__builtin_amdgcn_readfirstlane((u32)(v >> 32)) << 32) |
           __builtin_amdgcn_readfirstlane((u32)v);
}
// One tile of one residue per block: y = blockIdx.z * gridDim.y +
// blockIdx.y (a loop over residues here held its whole state across
// iterations, at 160-210 VGPRs and 2-3 waves per SIMD, against 47 and 8
// without it).
template <bool W12>
__global__ __launch_bounds__(SQ_THREADS) void k_square2_fold_slab_g(
        const u64 *__restrict__ in, u64 *__restrict__ out, u64 pitch, u64 r,
        const u64 *__restrict__ svec, unsigned n, unsigned group) {
    __shared__ __align__(16) u64 gw[SQ2_WINS * SQ2_LEN];
    const unsigned y = blockIdx.z * gridDim.y + blockIdx.y;
    if (y >= n) return;   // whole block
    const SqConst c = sq_const(r, uniform_u64(svec[y / group]));
    square2_tile<false, W12>(in + (u64)y * pitch, out + (u64)y * pitch, c, blockIdx.x, gw);
}

// The same two squarings of a slab in work units (as the batched kernel):
// desc[g] holds group g's constants and tile layout, computed on the host
// once per cohort (gf2t_sq2_slab_plan); blockIdx.x is the work unit.
struct Sq2SlabDesc {
    SqConst c;
    Sq2Chain h;
};
template <bool NT, bool W12>
__global__ __launch_bounds__(SQ_THREADS) __attribute__((amdgpu_waves_per_eu(8))) void
k_square2_fold_slab_u(const u64 *__restrict__ in, u64 *__restrict__ out, u64 pitch,
                      const Sq2SlabDesc *__restrict__ desc, unsigned n, unsigned group, u32 len) {
    __shared__ __align__(16) u64 gw[SQ2_WINS * SQ2_LEN];
    const unsigned y = blockIdx.z * gridDim.y + blockIdx.y;
    if (y >= n) return;   // whole block
    Sq2SlabDesc d = desc[y / group];
    if (d.h.len > len) d.h.len = len;   // a launch of few tiles: shorter units
    square2_unit<NT, W12>(in + (u64)y * pitch, out + (u64)y * pitch, d.c, d.h, blockIdx.x, gw);
}

// slab: residue y at in + y*pitch, its s in svec[y]
__global__ __launch_bounds__(SQ_THREADS) void k_square_fold_slab(
        const u64 *__restrict__ in, u64 *__restrict__ out, u64 pitch, u64 r,
        const u64 *__restrict__ svec) {
    const SqConst c = sq_const(r, svec[blockIdx.y]);
    size_t i = (size_t)blockIdx.x * SQ_THREADS + threadIdx.x;
    if (i >= (c.nw + 1) / 2) return;
    in += (u64)blockIdx.y * pitch;
    out += (u64)blockIdx.y * pitch;
    u64 o0, o1;
    square_fold_pair_fast(in, c, i, o0, o1);
    out[2 * i] = o0;
    if (2 * i + 1 < c.nw) out[2 * i + 1] = o1;
}

__global__ __launch_bounds__(SQ_THREADS) void k_fold(
        const u64 *__restrict__ p, size_t pw, u64 L, u64 *__restrict__ out,
        size_t nw, u64 r, u64 s) {
    size_t w = (size_t)blockIdx.x * SQ_THREADS + threadIdx.x;
    if (w >= nw) return;
    out[w] = fold_word(p, pw, L, r, s, w);
}

// dst ^= x*src mod T
__global__ __launch_bounds__(SQ_THREADS) void k_mulx_xor(
        u64 *__restrict__ dst, const u64 *__restrict__ src, size_t nw, u64 r,
        u64 s) {
    size_t w = (size_t)blockIdx.x * SQ_THREADS + threadIdx.x;
    if (w >= nw) return;
    u64 a = src[w];
    u64 prev = w ? src[w - 1] : 0;
    u64 v = (a << 1) | (prev >> 63);
    if (w == (size_t)(r >> 6)) v &= ~(1ULL << (r & 63));
    u64 wrap = (src[(r - 1) >> 6] >> ((r - 1) & 63)) & 1;   // coeff of x^(r-1)
    if (w == 0) v ^= wrap;
    if (w == (size_t)(s >> 6)) v ^= wrap << (s & 63);
    dst[w] ^= v;
}

__global__ void k_set_word0(u64 *p, size_t nw, u64 v0) {
    size_t w = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (w < nw) p[w] = w ? 0 : v0;
}

__global__ void k_xor_word0(u64 *p, u64 v) {
    if (blockIdx.x == 0 && threadIdx.x == 0) p[0] ^= v;
}

// r below 2^34: the kernels address a residue with 32-bit byte offsets
bool valid_rs(u64 r, u64 s) { return r >= 3 && r < (1ULL << 34) && s >= 1 && 2 * s < r; }

// tuning knobs of the batched squaring (gf2t_tune / GF2T_SQ_PPT, GF2T_SQ_ORDER)
int g_sq_ppt = -1, g_sq_order = -1, g_sq_nt = -1, g_sq_fuse = -1;
// two squarings per launch wherever a chain has two steps left
bool sq_fuse() {
    if (g_sq_fuse < 0) {
        const char *e = getenv("GF2T_SQ_FUSE");
        g_sq_fuse = e ? atoi(e) : 1;
    }
    return g_sq_fuse != 0;
}
bool sq_nt() {
    if (g_sq_nt < 0) {
        const char *e = getenv("GF2T_SQ_NT");
        g_sq_nt = e ? atoi(e) : 1;
    }
    return g_sq_nt != 0;
}
void sq_tuning(int &ppt, int &order) {
    if (g_sq_ppt < 0) {
        const char *e = getenv("GF2T_SQ_PPT");
        g_sq_ppt = e ? atoi(e) : 2;
    }
    if (g_sq_order < 0) {
        const char *e = getenv("GF2T_SQ_ORDER");
        g_sq_order = e ? atoi(e) : 0;
    }
    ppt = (g_sq_ppt == 2 || g_sq_ppt == 4) ? g_sq_ppt : 1;
    order = g_sq_order ? 1 : 0;
}

// 16-byte vector copy, four loads in flight per lane
template <bool NT>
__global__ __launch_bounds__(256) void k_stream_copy(const ulonglong2 *__restrict__ src,
                                                     ulonglong2 *__restrict__ dst, size_t n) {
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (; i + 3 * stride < n; i += 4 * stride) {
        ulonglong2 v[4] = {src[i], src[i + stride], src[i + 2 * stride], src[i + 3 * stride]};
#pragma unroll
        for (int k = 0; k < 4; k++) {
            if (NT) {
                typedef u64 v2u __attribute__((ext_vector_type(2)));
                __builtin_nontemporal_store(v2u{v[k].x, v[k].y}, (v2u *)&dst[i + k * stride]);
            } else {
                dst[i + k * stride] = v[k];
            }
        }
    }
    for (; i < n; i += stride) dst[i] = src[i];
}

unsigned blocks_for(size_t work, int threads) {
    return (unsigned)((work + threads - 1) / threads);
}

}  // namespace

extern "C" int gf2t_square_fold(const uint64_t *din, uint64_t *dout, uint64_t r,
                                uint64_t s, void *stream) {
    if (!valid_rs(r, s) || !din || !dout || din == dout) {
        gf2t::set_error("gf2t_square_fold: need r >= 3, 1 <= s, 2s < r, din != dout");
        return GF2T_EINVAL;
    }
    SqConst c = sq_const(r, s);
    if (sq_w12_ok(r))
        hipLaunchKernelGGL(k_square_fold<true>, dim3(blocks_for((c.nw + 1) / 2, SQ_THREADS)),
                           dim3(SQ_THREADS), 0, (hipStream_t)stream, din, dout, c);
    else
        hipLaunchKernelGGL(k_square_fold<false>, dim3(blocks_for((c.nw + 1) / 2, SQ_THREADS)),
                           dim3(SQ_THREADS), 0, (hipStream_t)stream, din, dout, c);
    GF2T_CHECK_LAUNCH("k_square_fold");
    return GF2T_OK;
}

namespace {
// chains of n residues (list in device memory, or one) of at most nw words
// and `steps` squarings, in LDS
int run_chains(const ChainDesc *list, const ChainDesc &one, unsigned n, size_t nw, u64 steps,
               hipStream_t st) {
    const size_t np = (nw + 1) / 2, lds = 2 * (2 * np + 2) * 8;
    const unsigned threads = (unsigned)std::min<size_t>(CH_THREADS, (np + 63) & ~(size_t)63);
    const int K = (int)((np + threads - 1) / threads);   // 1..5
    const auto kernel = K == 1 ? k_square_chain<1> : K == 2 ? k_square_chain<2>
                        : K == 3 ? k_square_chain<3> : k_square_chain<5>;
    // more than 64 KiB of LDS has to be allowed, once per kernel and device
    static std::atomic<unsigned> allowed[64];
    int dev = 0;
    GF2T_HIP(hipGetDevice(&dev));
    if (dev >= 64 || !((allowed[dev].load() >> K) & 1)) {
        GF2T_HIP(hipFuncSetAttribute((const void *)kernel,
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)CH_LDS));
        if (dev < 64) allowed[dev].fetch_or(1u << K);
    }
    for (u64 k = 0; k < steps; k += CH_STEPS)
        hipLaunchKernelGGL(kernel, dim3(n), dim3(threads), lds, st, list, one, k, CH_STEPS);
    GF2T_CHECK_LAUNCH("k_square_chain");
    return GF2T_OK;
}
}  // namespace

extern "C" int gf2t_square_fold_steps(uint64_t *dres, uint64_t *dtmp, uint64_t r,
                                      uint64_t s, uint64_t steps, void *stream) {
    if (!valid_rs(r, s) || !dres || !dtmp || dres == dtmp) {
        gf2t::set_error("gf2t_square_fold_steps: bad arguments");
        return GF2T_EINVAL;
    }
    SqConst c = sq_const(r, s);
    size_t nw = c.nw;
    hipStream_t st = (hipStream_t)stream;
    if (nw <= CH_ONE && sq_fuse() && steps > 3)
        return run_chains(nullptr, ChainDesc{dres, c, steps}, 1, nw, steps, st);
    u64 *a = dres, *b = dtmp;
    const bool fuse = sq_fuse(), w12 = sq_w12_ok(r);
    const PowOrder po = pow_order(nw, s);
    const u64 ranges = pow_ranges(nw), tiles = sq2_tiles(sq2_chain(c));
    const Sq2Chain h2 = sq2_chain(c, sq2_chain_len(tiles));
    const dim3 g2((unsigned)sq2_units(h2)), g1(blocks_for((nw + 1) / 2, SQ_THREADS));
    const int per = !fuse ? 1 : pow_per(ranges, pow_cost(steps, 2), pow_cost(steps, 3));
    u64 launches = 0;
    for (u64 k = 0; k < steps; launches++) {
        // by three: what is left over first
        const int m = per == 3 && (steps - k) % 3 ? (int)((steps - k) % 3) : per;
        if (per == 2 && steps - k >= 2) {
            if (w12)
                hipLaunchKernelGGL(k_square2_fold<true>, g2, dim3(SQ_THREADS), 0, st, a, b, c, h2);
            else
                hipLaunchKernelGGL(k_square2_fold<false>, g2, dim3(SQ_THREADS), 0, st, a, b, c, h2);
            k += 2;
        } else if (per == 3 && (m > 1 || pow_one(ranges))) {
            auto launch = [&](auto kernel, u64 blocks) {
                hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(PW_T), 0, st, a, b, c, po, m);
            };
            if (ranges >= PW_COLS) launch(k_power<4, true>, power_blocks<4, true>(nw, m, po));
            else if (ranges >= PW_FULL) launch(k_power<4, false>, power_blocks<4, false>(nw, m, po));
            else launch(k_power<1, false>, power_blocks<1, false>(nw, m, po));
            k += m;
        } else {
            if (w12)
                hipLaunchKernelGGL(k_square_fold<true>, g1, dim3(SQ_THREADS), 0, st, a, b, c);
            else
                hipLaunchKernelGGL(k_square_fold<false>, g1, dim3(SQ_THREADS), 0, st, a, b, c);
            k += 1;
        }
        std::swap(a, b);
    }
    GF2T_CHECK_LAUNCH("k_square_fold");
    if (launches & 1) GF2T_HIP(hipMemcpyAsync(dres, dtmp, nw * 8, hipMemcpyDeviceToDevice, st));
    return GF2T_OK;
}

namespace {
// descriptor and tile-order tables for the batched chain, cached and
// grown on demand
struct BatchScratch {
    unsigned char *d = nullptr;   // cap bytes
    int *ord = nullptr;
    size_t cap = 0, ocap = 0;
    int dev = -1;
    std::mutex mu;   // held by a call until its launches are done
} g_batch;

template <int PPT, bool W12>
void launch_batch(unsigned gx, unsigned active, const SqDesc *tab, hipStream_t st) {
    if (sq_nt())
        hipLaunchKernelGGL((k_square_fold_batch<PPT, true, W12>), dim3(gx, active),
                           dim3(SQ_THREADS), 0, st, tab);
    else
        hipLaunchKernelGGL((k_square_fold_batch<PPT, false, W12>), dim3(gx, active),
                           dim3(SQ_THREADS), 0, st, tab);
}
template <bool W12>
void launch_batch12(unsigned gx, unsigned active, const SqDesc *tab, hipStream_t st) {
    if (sq_nt())
        hipLaunchKernelGGL((k_square12_fold_batch<true, W12>), dim3(gx, active), dim3(SQ_THREADS),
                           0, st, tab);
    else
        hipLaunchKernelGGL((k_square12_fold_batch<false, W12>), dim3(gx, active), dim3(SQ_THREADS),
                           0, st, tab);
}
template <bool W12>
void launch_batch2(unsigned gx, unsigned active, const SqDesc *tab, hipStream_t st) {
    if (sq_nt())
        hipLaunchKernelGGL((k_square2_fold_batch<true, W12>), dim3(gx, active), dim3(SQ_THREADS),
                           0, st, tab);
    else
        hipLaunchKernelGGL((k_square2_fold_batch<false, W12>), dim3(gx, active),
                           dim3(SQ_THREADS), 0, st, tab);
}
template <int U, bool COLS>
void launch_power(bool first, unsigned gx, unsigned active, const SqDesc *tab, hipStream_t st) {
    if (first)
        hipLaunchKernelGGL((k_power_batch<U, COLS, true>), dim3(gx, active), dim3(PW_T), 0, st, tab);
    else
        hipLaunchKernelGGL((k_power_batch<U, COLS, false>), dim3(gx, active), dim3(PW_T), 0, st, tab);
}
}  // namespace

namespace gf2t_host {
bool square_fuse_enabled() { return sq_fuse(); }
}

int gf2t_fft_set_tile_bits(int m, int64_t T);   // fft.hip
int gf2t_fft_tile_bits(int m);
int gf2t_fft_set_ept(int64_t ept);                // fft.hip
int gf2t_fft_ept();
int gf2t_fft_set_low_bits(int64_t c);             // fft.hip
int gf2t_fft_low_bits();
int gf2t_hm_set_zc_words(int64_t words);          // fft.hip
int64_t gf2t_hm_zc_words();
int gf2t_sieve_tune(const char *key, int64_t v);   // sieve.hip
int gf2t_sieve_tune_get(const char *key, int64_t *v);

extern "C" int gf2t_tune(const char *key, int64_t value) {
    if (!key) return GF2T_EINVAL;
    if (!strncmp(key, "fft_tile_", 9) && key[9]) {
        char *end = nullptr;
        long m = strtol(key + 9, &end, 10);
        if (*end == 0) return gf2t_fft_set_tile_bits((int)m, value);
    }
    if (!strcmp(key, "sieve_wide_from") || !strcmp(key, "sieve_slices"))
        return gf2t_sieve_tune(key, value);
    if (!strncmp(key, "block_m_", 8) && key[8]) {
        char *end = nullptr;
        long k = strtol(key + 8, &end, 10);
        if (*end == 0 && gf2t_host::set_tuned_block_m((int)k, (int)value)) return GF2T_OK;
        gf2t::set_error("gf2t_tune: block_m_<k> needs 2 <= k <= 40 and 0 <= m <= 64");
        return GF2T_EINVAL;
    }
    if (!strcmp(key, "sq_ppt")) { g_sq_ppt = (int)value; return GF2T_OK; }
    if (!strcmp(key, "sq_order")) { g_sq_order = (int)value; return GF2T_OK; }
    if (!strcmp(key, "sq_nt")) { g_sq_nt = (int)value; return GF2T_OK; }
    if (!strcmp(key, "sq_fuse")) { g_sq_fuse = (int)value; return GF2T_OK; }
    if (!strcmp(key, "gcd_dev_bits")) {
        gf2t_host::set_device_product_bits(value > 0 ? (uint64_t)value : 0);
        return GF2T_OK;
    }
    if (!strcmp(key, "gcd_base_bits")) {
        if (gf2t_host::set_gcd_base_bits(value)) return GF2T_OK;
        gf2t::set_error("gf2t_tune: gcd_base_bits needs 128 <= bits <= 65536");
        return GF2T_EINVAL;
    }
    if (!strcmp(key, "gcd_school_words")) {
        if (gf2t_host::set_school_words(value)) return GF2T_OK;
        gf2t::set_error("gf2t_tune: gcd_school_words needs 8 <= words <= 512");
        return GF2T_EINVAL;
    }
    if (!strcmp(key, "fft_ept")) return gf2t_fft_set_ept(value);
    if (!strcmp(key, "fft_low_bits")) return gf2t_fft_set_low_bits(value);
    if (!strcmp(key, "hm_zc_words")) return gf2t_hm_set_zc_words(value);
    if (!strcmp(key, "scan_stagger")) {
        if (value < -1 || value > 64) {
            gf2t::set_error("gf2t_tune: scan_stagger needs -1 <= value <= 64");
            return GF2T_EINVAL;
        }
        gf2t_host::set_scan_stagger((int)value);
        return GF2T_OK;
    }
    gf2t::set_error("gf2t_tune: unknown key '%s'", key);
    return GF2T_EINVAL;
}

extern "C" int gf2t_tune_get(const char *key, int64_t *value) {
    if (!key || !value) return GF2T_EINVAL;
    int ppt = 0, order = 0;
    sq_tuning(ppt, order);
    if (!strcmp(key, "sq_ppt")) { *value = ppt; return GF2T_OK; }
    if (!strcmp(key, "sq_order")) { *value = order; return GF2T_OK; }
    if (!strcmp(key, "sq_nt")) { *value = sq_nt() ? 1 : 0; return GF2T_OK; }
    if (!strcmp(key, "sq_fuse")) { *value = sq_fuse() ? 1 : 0; return GF2T_OK; }
    if (!strcmp(key, "gcd_dev_bits")) {
        *value = (int64_t)gf2t_host::device_product_bits();
        return GF2T_OK;
    }
    if (!strcmp(key, "gcd_base_bits")) {
        *value = gf2t_host::gcd_base_bits();
        return GF2T_OK;
    }
    if (!strcmp(key, "gcd_school_words")) {
        *value = gf2t_host::school_words();
        return GF2T_OK;
    }
    if (!strcmp(key, "fft_ept")) {
        *value = gf2t_fft_ept();
        return GF2T_OK;
    }
    if (!strcmp(key, "fft_low_bits")) {
        *value = gf2t_fft_low_bits();
        return GF2T_OK;
    }
    if (!strcmp(key, "hm_zc_words")) {
        *value = gf2t_hm_zc_words();
        return GF2T_OK;
    }
    if (!strcmp(key, "scan_stagger")) {
        *value = gf2t_host::scan_stagger();
        return GF2T_OK;
    }
    if (!strcmp(key, "sieve_wide_from") || !strcmp(key, "sieve_slices"))
        return gf2t_sieve_tune_get(key, value);
    if (!strncmp(key, "fft_tile_", 9) && key[9]) {
        char *end = nullptr;
        long m = strtol(key + 9, &end, 10);
        if (*end == 0 && gf2t_fft_tile_bits((int)m)) {
            *value = gf2t_fft_tile_bits((int)m);
            return GF2T_OK;
        }
    }
    if (!strncmp(key, "block_m_", 8) && key[8]) {
        char *end = nullptr;
        long k = strtol(key + 8, &end, 10);
        if (*end == 0 && k >= 2 && k <= 40) {
            *value = gf2t_host::tuned_block_m(1ULL << k);
            return GF2T_OK;
        }
    }
    gf2t::set_error("gf2t_tune_get: unknown key '%s'", key);
    return GF2T_EINVAL;
}

extern "C" int gf2t_square_fold_batch(uint64_t *const *dres, uint64_t *const *dtmp,
                                      const uint64_t *r, const uint64_t *s,
                                      const uint64_t *steps, int n, void *stream) {
    if (n < 0 || (n > 0 && (!dres || !dtmp || !r || !s || !steps))) {
        gf2t::set_error("gf2t_square_fold_batch: bad arguments");
        return GF2T_EINVAL;
    }
    if (n == 0) return GF2T_OK;
    if (n > 65535) {
        gf2t::set_error("gf2t_square_fold_batch: at most 65535 residues per call");
        return GF2T_ERANGE;
    }
    for (int i = 0; i < n; i++)
        if (!valid_rs(r[i], s[i]) || !dres[i] || !dtmp[i] || dres[i] == dtmp[i] ||
            (((uintptr_t)dres[i] | (uintptr_t)dtmp[i]) & 15)) {
            gf2t::set_error("gf2t_square_fold_batch: residue %d has bad r/s/buffers "
                            "(distinct, 16-byte aligned)", i);
            return GF2T_EINVAL;
        }
    hipStream_t st = (hipStream_t)stream;
    int ppt, order;
    sq_tuning(ppt, order);
    const bool fuse = sq_fuse();
    int dev = 0;
    GF2T_HIP(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lock(g_batch.mu);
    if (g_batch.dev != dev) {   // (what another device holds stays there)
        g_batch.d = nullptr;
        g_batch.ord = nullptr;
        g_batch.cap = g_batch.ocap = 0;
        g_batch.dev = dev;
    }
    // residues whose chain runs in LDS, and the others, by launches: those
    // with most launches first, so that the residues still active at a
    // launch are a prefix (uneven frontiers, per-s early exit)
    std::vector<int> ord;
    std::vector<ChainDesc> chains;
    size_t chain_nw = 0;
    u64 chain_steps = 0;
    int larger = 0;   // residues that fit in LDS, above CH_ONE
    for (int i = 0; i < n; i++)
        larger += steps[i] && words_of(r[i]) > CH_ONE && words_of(r[i]) <= CH_WORDS;
    for (int i = 0; i < n; i++) {
        const size_t nw = words_of(r[i]);
        if (!steps[i]) continue;
        if (fuse && nw <= (larger < CH_FEW ? CH_ONE : CH_WORDS)) {
            chains.push_back(ChainDesc{dres[i], sq_const(r[i], s[i]), steps[i]});
            chain_nw = std::max(chain_nw, nw);
            chain_steps = std::max<u64>(chain_steps, steps[i]);
        } else {
            ord.push_back(i);
        }
    }
    u64 ranges = 0, most_ranges = 0, tiles2 = 0;   // of all residues by launches; of the largest
    u64 two = 0, three = 0;   // their costs by two and by three squarings a launch
    if (fuse)
        for (int i : ord) {
            const SqConst c = sq_const(r[i], s[i]);
            ranges += pow_ranges(c.nw);
            most_ranges = std::max(most_ranges, pow_ranges(c.nw));
            two += c.nw * pow_cost(steps[i], 2);
            three += c.nw * pow_cost(steps[i], 3);
            tiles2 += sq2_tiles(sq2_chain(c));
        }
    // squarings per launch, and a chain's launches
    const u64 per = !fuse ? 1 : (u64)pow_per(ranges, two, three);
    auto nlaunch = [&](int i) { return (steps[i] + per - 1) / per; };
    std::stable_sort(ord.begin(), ord.end(), [&](int a, int b) { return nlaunch(a) > nlaunch(b); });
    std::stable_sort(chains.begin(), chains.end(), [](const ChainDesc &a, const ChainDesc &b) {
        return a.steps * a.c.nw > b.steps * b.c.nw;
    });
    const int nl = (int)ord.size();
    // descriptors of the launches (even, then odd ones), then the chains
    const size_t chain_at = 2 * (size_t)nl * sizeof(SqDesc);
    const size_t need = chain_at + chains.size() * sizeof(ChainDesc);
    std::vector<size_t> ooff(nl, 0);
    std::vector<int> otab;
    size_t gx = 0, gx1 = 0;
    const u64 tile_pairs = (u64)SQ_THREADS * ppt;
    for (int k = 0; k < nl; k++) {
        SqConst c = sq_const(r[ord[k]], s[ord[k]]);
        u64 T = ((c.nw + 1) / 2 + tile_pairs - 1) / tile_pairs;
        if (order) {
            TileOrder o = tile_order(T, sq_delta_pairs(c), tile_pairs);
            ooff[k] = otab.size();
            for (u64 x = 0; x < 8 * o.P; x++) otab.push_back((int)tile_of(o, x));
            gx = std::max<size_t>(gx, 8 * o.P);
        } else {
            gx = std::max<size_t>(gx, T);
        }
    }
    if (g_batch.cap < need) {
        if (g_batch.d) (void)hipFree(g_batch.d);
        g_batch.d = nullptr;
        g_batch.cap = 0;
        GF2T_HIP(hipMalloc((void **)&g_batch.d, need));
        g_batch.cap = need;
    }
    // a block index beyond a residue's own table must idle: pad each
    // residue's table to gx entries
    if (order && nl) {
        std::vector<int> padded((size_t)nl * gx, -1);
        for (int k = 0; k < nl; k++) {
            size_t len = (k + 1 < nl ? ooff[k + 1] : otab.size()) - ooff[k];
            std::copy(otab.begin() + ooff[k], otab.begin() + ooff[k] + len,
                      padded.begin() + (size_t)k * gx);
        }
        otab.swap(padded);
        if (g_batch.ocap < otab.size()) {
            if (g_batch.ord) (void)hipFree(g_batch.ord);
            g_batch.ord = nullptr;
            g_batch.ocap = 0;
            GF2T_HIP(hipMalloc(&g_batch.ord, otab.size() * sizeof(int)));
            g_batch.ocap = otab.size();
        }
        GF2T_HIP(hipMemcpyAsync(g_batch.ord, otab.data(), otab.size() * sizeof(int),
                                hipMemcpyHostToDevice, st));
    }
    std::vector<unsigned char> h(need);
    SqDesc *hd = (SqDesc *)h.data();
    const int shape = most_ranges >= PW_COLS ? 2 : ranges >= PW_FULL ? 1 : 0;
    const u32 len2 = sq2_chain_len(tiles2);
    u64 gx2 = 0;            // work units of the residue with the most
    u64 gx3 = 0, gxf = 0;   // its blocks of F^8 windows, and in the first launch
    bool odd = false;       // some chain's first launch takes fewer than the others
    bool ones = per > 1;    // every chain's takes one
    bool w12 = true;   // 12-byte window loads: no r of the launches a multiple of 64
    bool back = false; // some chain ends in dtmp
    for (int k = 0; k < nl; k++) {
        const int i = ord[k];
        const SqConst c = sq_const(r[i], s[i]);
        const int *ot = order ? g_batch.ord + (size_t)k * gx : nullptr;
        const Sq2Chain h2 = sq2_chain(c, len2);
        const PowOrder po = pow_order(c.nw, c.s);
        const int m = (int)(steps[i] % per ? steps[i] % per : per);
        const int bk = (int)(nlaunch(i) & 1);
        new (hd + k) SqDesc{dres[i], dtmp[i], c, m, bk, ot, h2, po};        // even launches
        new (hd + nl + k) SqDesc{dtmp[i], dres[i], c, (int)per, bk, ot, h2, po};   // odd launches
        odd = odd || m != (int)per;
        ones = ones && m == 1;
        back = back || bk;
        gx2 = std::max(gx2, sq2_units(h2));
        auto blocks = [&](int m) {
            return shape == 2 ? power_blocks<4, true>(c.nw, m, po)
                   : shape == 1 ? power_blocks<4, false>(c.nw, m, po) : power_blocks<1, false>(c.nw, m, po);
        };
        gx3 = std::max(gx3, blocks(3));
        gxf = std::max(gxf, blocks(m));
        w12 = w12 && sq_w12_ok(r[i]);
        gx1 = std::max<size_t>(gx1, ((c.nw + 1) / 2 + SQ_THREADS - 1) / SQ_THREADS);
    }
    if (!chains.empty()) std::memcpy(h.data() + chain_at, chains.data(), chains.size() * sizeof(ChainDesc));
    if (need == 0) return GF2T_OK;   // no squaring to do
    GF2T_HIP(hipMemcpyAsync(g_batch.d, h.data(), need, hipMemcpyHostToDevice, st));
    if (!chains.empty()) {
        int rc = run_chains((const ChainDesc *)(g_batch.d + chain_at), chains[0],
                            (unsigned)chains.size(), chain_nw, chain_steps, st);
        if (rc) return rc;
    }
    // Every launch advances all live chains together, by `per` squarings (in
    // the first by what a chain's length leaves over); a chain's value is in
    // dtmp after an odd number of launches.
    const SqDesc *dd = (const SqDesc *)g_batch.d;
    int active = nl;
    for (u64 l = 0; active > 0; l++) {
        const SqDesc *tab = dd + ((l & 1) ? nl : 0);
        const bool first = l == 0 && odd;
        if (per == 1 || (l == 0 && ones && !(per == 3 && pow_one(most_ranges)))) {
            if (ppt == 4 && w12) launch_batch<4, true>((unsigned)gx, active, tab, st);
            else if (ppt == 4) launch_batch<4, false>((unsigned)gx, active, tab, st);
            else if (ppt == 2 && w12) launch_batch<2, true>((unsigned)gx, active, tab, st);
            else if (ppt == 2) launch_batch<2, false>((unsigned)gx, active, tab, st);
            else if (w12) launch_batch<1, true>((unsigned)gx, active, tab, st);
            else launch_batch<1, false>((unsigned)gx, active, tab, st);
        } else if (per == 3) {
            const unsigned g = (unsigned)(first ? gxf : gx3);
            if (shape == 2) launch_power<4, true>(first, g, active, tab, st);
            else if (shape == 1) launch_power<4, false>(first, g, active, tab, st);
            else launch_power<1, false>(first, g, active, tab, st);
        } else if (per == 2 && first) {
            // enough blocks for the one-squaring residues' pairs in a few rounds
            const unsigned g = (unsigned)std::max<u64>(gx2, (gx1 + 7) / 8);
            if (w12) launch_batch12<true>(g, active, tab, st);
            else launch_batch12<false>(g, active, tab, st);
        } else {
            if (w12) launch_batch2<true>((unsigned)gx2, active, tab, st);
            else launch_batch2<false>((unsigned)gx2, active, tab, st);
        }
        while (active > 0 && nlaunch(ord[active - 1]) == l + 1) active--;
    }
    if (back)
        hipLaunchKernelGGL(k_batch_back, dim3((unsigned)std::min<size_t>((gx1 + 1) / 2, 1024), nl),
                           dim3(SQ_THREADS), 0, st, dd + nl);
    GF2T_CHECK_LAUNCH("k_square_fold_batch");
    // the host tables must outlive the async copies
    GF2T_HIP(hipStreamSynchronize(st));
    return GF2T_OK;
}

extern "C" int gf2t_fold(const uint64_t *dsrc, uint64_t src_bits, uint64_t *dout,
                         uint64_t r, uint64_t s, void *stream) {
    if (!valid_rs(r, s) || !dsrc || !dout || dsrc == dout || src_bits > 2 * r - 1) {
        gf2t::set_error("gf2t_fold: need valid r/s, src_bits <= 2r-1, dsrc != dout");
        return GF2T_EINVAL;
    }
    size_t nw = words_of(r), pw = words_of(src_bits);
    hipLaunchKernelGGL(k_fold, dim3(blocks_for(nw, SQ_THREADS)), dim3(SQ_THREADS), 0,
                       (hipStream_t)stream, dsrc, pw, src_bits, dout, nw, r, s);
    GF2T_CHECK_LAUNCH("k_fold");
    return GF2T_OK;
}

extern "C" int gf2t_mulx_xor(uint64_t *ddst, const uint64_t *dsrc, uint64_t r,
                             uint64_t s, void *stream) {
    if (!valid_rs(r, s) || !ddst || !dsrc || ddst == dsrc) {
        gf2t::set_error("gf2t_mulx_xor: bad arguments");
        return GF2T_EINVAL;
    }
    size_t nw = words_of(r);
    hipLaunchKernelGGL(k_mulx_xor, dim3(blocks_for(nw, SQ_THREADS)), dim3(SQ_THREADS), 0,
                       (hipStream_t)stream, ddst, dsrc, nw, r, s);
    GF2T_CHECK_LAUNCH("k_mulx_xor");
    return GF2T_OK;
}

extern "C" int gf2t_set_x(uint64_t *dp, size_t nw, void *stream) {
    if (!dp || nw == 0) { gf2t::set_error("gf2t_set_x: bad arguments"); return GF2T_EINVAL; }
    hipLaunchKernelGGL(k_set_word0, dim3(blocks_for(nw, 256)), dim3(256), 0,
                       (hipStream_t)stream, dp, nw, 2ULL);
    GF2T_CHECK_LAUNCH("k_set_word0");
    return GF2T_OK;
}

extern "C" int gf2t_set_one(uint64_t *dp, size_t nw, void *stream) {
    if (!dp || nw == 0) { gf2t::set_error("gf2t_set_one: bad arguments"); return GF2T_EINVAL; }
    hipLaunchKernelGGL(k_set_word0, dim3(blocks_for(nw, 256)), dim3(256), 0,
                       (hipStream_t)stream, dp, nw, 1ULL);
    GF2T_CHECK_LAUNCH("k_set_word0");
    return GF2T_OK;
}

extern "C" int gf2t_xor_x(uint64_t *dp, void *stream) {
    if (!dp) { gf2t::set_error("gf2t_xor_x: null pointer"); return GF2T_EINVAL; }
    hipLaunchKernelGGL(k_xor_word0, dim3(1), dim3(64), 0, (hipStream_t)stream, dp, 2ULL);
    GF2T_CHECK_LAUNCH("k_xor_word0");
    return GF2T_OK;
}

extern "C" int gf2t_square_fold_slab(const uint64_t *din, uint64_t *dout, size_t pitch,
                                     uint64_t r, const uint64_t *ds, int n, void *stream) {
    size_t nw = words_of(r);
    if (!din || !dout || !ds || din == dout || r < 3 || pitch < nw || n < 0 || n > 65535) {
        gf2t::set_error("gf2t_square_fold_slab: bad arguments");
        return GF2T_EINVAL;
    }
    if (n == 0) return GF2T_OK;
    unsigned gx = blocks_for((nw + 1) / 2, SQ_THREADS);
    hipLaunchKernelGGL(k_square_fold_slab, dim3(gx, n), dim3(SQ_THREADS), 0,
                       (hipStream_t)stream, din, dout, (u64)pitch, r, ds);
    GF2T_CHECK_LAUNCH("k_square_fold_slab");
    return GF2T_OK;
}

extern "C" int gf2t_stream_copy(void *dst, const void *src, size_t bytes, void *stream) {
    if (!dst || !src || (bytes & 15) || (((uintptr_t)dst | (uintptr_t)src) & 15)) {
        gf2t::set_error("gf2t_stream_copy: 16-byte aligned pointers and size required");
        return GF2T_EINVAL;
    }
    size_t n = bytes / 16;
    // one 4-load iteration per lane: the widest grid reads fastest here
    // (5.46 TB/s copying 4.36 GB, against 4.87 TB/s with 8192 blocks)
    unsigned blocks = (unsigned)std::min<size_t>((n + 1023) / 1024, (size_t)1 << 20);
    if (sq_nt())
        hipLaunchKernelGGL(k_stream_copy<true>, dim3(blocks ? blocks : 1), dim3(256), 0,
                           (hipStream_t)stream, (const ulonglong2 *)src, (ulonglong2 *)dst, n);
    else
        hipLaunchKernelGGL(k_stream_copy<false>, dim3(blocks ? blocks : 1), dim3(256), 0,
                           (hipStream_t)stream, (const ulonglong2 *)src, (ulonglong2 *)dst, n);
    GF2T_CHECK_LAUNCH("k_stream_copy");
    return GF2T_OK;
}

extern "C" int gf2t_square2_fold_slab_g(const uint64_t *din, uint64_t *dout, size_t pitch,
                                        uint64_t r, const uint64_t *ds, size_t n, int group,
                                        void *stream) {
    size_t nw = words_of(r);
    if (!din || !dout || !ds || din == dout || r < 5 || r >= (1ULL << 34) || pitch < nw ||
        (pitch & 1) || (((uintptr_t)din | (uintptr_t)dout) & 15) || group < 1 ||
        n > 0xFFFFFFFFu) {
        gf2t::set_error("gf2t_square2_fold_slab_g: bad arguments (even pitch, 16-byte "
                        "aligned slabs)");
        return GF2T_EINVAL;
    }
    if (n == 0) return GF2T_OK;
    const unsigned gx = (unsigned)(((nw + 1) / 2 + SQ2_TP - 1) / SQ2_TP);
    const unsigned gy = n < 65535 ? (unsigned)n : 65535u;
    const unsigned gz = (unsigned)((n + gy - 1) / gy);
    if (sq_w12_ok(r))
        hipLaunchKernelGGL(k_square2_fold_slab_g<true>, dim3(gx, gy, gz), dim3(SQ_THREADS), 0,
                           (hipStream_t)stream, din, dout, (u64)pitch, r, ds, (unsigned)n,
                           (unsigned)group);
    else
        hipLaunchKernelGGL(k_square2_fold_slab_g<false>, dim3(gx, gy, gz), dim3(SQ_THREADS), 0,
                           (hipStream_t)stream, din, dout, (u64)pitch, r, ds, (unsigned)n,
                           (unsigned)group);
    GF2T_CHECK_LAUNCH("k_square2_fold_slab_g");
    return GF2T_OK;
}

// ---- two squarings of a slab in work units, with per-group layouts
struct gf2t_sq2_slab_plan {
    u64 r = 0;
    size_t cap = 0, ngroups = 0;
    unsigned gx[SQ2_CHAIN + 1] = {};   // work units of the group with the most, by unit length
    u64 tiles = 0;                     // tiles of that group
    Sq2SlabDesc *d = nullptr;
    std::vector<Sq2SlabDesc> h;   // host copy (source of the last upload)
};

extern "C" int gf2t_sq2_slab_plan_set(gf2t_sq2_slab_plan *p, const uint64_t *hs, size_t ngroups,
                                      void *stream) {
    if (!p || !hs || ngroups == 0 || ngroups > p->cap) {
        gf2t::set_error("gf2t_sq2_slab_plan_set: bad arguments (at most %zu groups)",
                        p ? p->cap : (size_t)0);
        return GF2T_EINVAL;
    }
    for (size_t g = 0; g < ngroups; g++)
        if (!valid_rs(p->r, hs[g])) {
            gf2t::set_error("gf2t_sq2_slab_plan_set: group %zu has bad s", g);
            return GF2T_EINVAL;
        }
    // the previous upload may still be in flight from h: let it finish
    // before h changes
    GF2T_HIP(hipStreamSynchronize((hipStream_t)stream));
    unsigned gx[SQ2_CHAIN + 1] = {};
    u64 tiles = 0;
    for (size_t g = 0; g < ngroups; g++) {
        const SqConst c = sq_const(p->r, hs[g]);
        p->h[g] = Sq2SlabDesc{c, sq2_chain(c)};
        tiles = std::max(tiles, sq2_tiles(p->h[g].h));
        for (u32 len = 1; len <= SQ2_CHAIN; len++)
            gx[len] = std::max(gx[len], (unsigned)sq2_units(sq2_chain(c, len)));
    }
    GF2T_HIP(hipMemcpyAsync(p->d, p->h.data(), ngroups * sizeof(Sq2SlabDesc),
                            hipMemcpyHostToDevice, (hipStream_t)stream));
    p->ngroups = ngroups;
    std::copy(gx, gx + SQ2_CHAIN + 1, p->gx);
    p->tiles = tiles;
    return GF2T_OK;
}

extern "C" int gf2t_sq2_slab_plan_create(uint64_t r, const uint64_t *hs, size_t ngroups,
                                         gf2t_sq2_slab_plan **plan) {
    if (!plan || !hs || ngroups == 0 || r < 5 || r >= (1ULL << 34)) {
        gf2t::set_error("gf2t_sq2_slab_plan_create: bad arguments");
        return GF2T_EINVAL;
    }
    *plan = nullptr;
    gf2t_sq2_slab_plan *p = new gf2t_sq2_slab_plan;
    p->r = r;
    p->cap = ngroups;
    p->h.resize(ngroups);
    hipError_t e = hipMalloc((void **)&p->d, ngroups * sizeof(Sq2SlabDesc));
    if (e != hipSuccess) {
        delete p;
        return gf2t::hip_fail(e, "hipMalloc", __FILE__, __LINE__);
    }
    int rc = gf2t_sq2_slab_plan_set(p, hs, ngroups, nullptr);
    if (rc == GF2T_OK) rc = hipStreamSynchronize(nullptr) == hipSuccess ? GF2T_OK : GF2T_EHIP;
    if (rc) {
        (void)hipFree(p->d);
        delete p;
        return rc;
    }
    *plan = p;
    return GF2T_OK;
}

extern "C" int gf2t_sq2_slab_plan_destroy(gf2t_sq2_slab_plan *p) {
    if (!p) return GF2T_OK;
    if (p->d) (void)hipFree(p->d);
    delete p;
    return GF2T_OK;
}

extern "C" int gf2t_square2_fold_slab_p(const gf2t_sq2_slab_plan *p, const uint64_t *din,
                                        uint64_t *dout, size_t pitch, size_t n, int group,
                                        void *stream) {
    if (!p || !din || !dout || din == dout || group < 1 || pitch < words_of(p->r) ||
        (pitch & 1) || (((uintptr_t)din | (uintptr_t)dout) & 15) || n > 0xFFFFFFFFu ||
        (n + (size_t)group - 1) / (size_t)group > p->ngroups) {
        gf2t::set_error("gf2t_square2_fold_slab_p: bad arguments (even pitch, 16-byte aligned "
                        "slabs, n / group within the plan's groups)");
        return GF2T_EINVAL;
    }
    if (n == 0) return GF2T_OK;
    const unsigned gy = n < 65535 ? (unsigned)n : 65535u;
    const unsigned gz = (unsigned)((n + gy - 1) / gy);
    const u32 len = sq2_chain_len(p->tiles * n);
    const dim3 grid(p->gx[len], gy, gz);
    const bool w12 = sq_w12_ok(p->r), nt = sq_nt();
    hipStream_t st = (hipStream_t)stream;
    if (nt && w12)
        hipLaunchKernelGGL((k_square2_fold_slab_u<true, true>), grid, dim3(SQ_THREADS), 0, st, din,
                           dout, (u64)pitch, p->d, (unsigned)n, (unsigned)group, len);
    else if (nt)
        hipLaunchKernelGGL((k_square2_fold_slab_u<true, false>), grid, dim3(SQ_THREADS), 0, st,
                           din, dout, (u64)pitch, p->d, (unsigned)n, (unsigned)group, len);
    else if (w12)
        hipLaunchKernelGGL((k_square2_fold_slab_u<false, true>), grid, dim3(SQ_THREADS), 0, st,
                           din, dout, (u64)pitch, p->d, (unsigned)n, (unsigned)group, len);
    else
        hipLaunchKernelGGL((k_square2_fold_slab_u<false, false>), grid, dim3(SQ_THREADS), 0, st,
                           din, dout, (u64)pitch, p->d, (unsigned)n, (unsigned)group, len);
    GF2T_CHECK_LAUNCH("k_square2_fold_slab_u");
    return GF2T_OK;
}
