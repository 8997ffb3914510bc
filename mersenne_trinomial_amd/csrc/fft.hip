// fft.hip -- (c) Cantor additive FFT over GF(2^64) and GF(2)[x] products
// on gfx950.
//
// Transform (same evaluation points and natural output order as the
// reference's CantorFFT, src/gf2_cantor_engine.h:125-188): output i is
// the chunk polynomial evaluated at sum_{bits k of i} b[k] of the Cantor
// basis.  Two parts:
//   1. the basis conversion (cantor.hpp): from powers of X to the products
//      of the subspace polynomials s_k, XORs only, O(m log m) of them per
//      coefficient.  Of a product's operands it runs on their 32-bit
//      chunks, before they become field elements.
//   2. butterflies, level L on index bit L: e1 = g + W(t) h, e2 = e1 + h
//      with W(t) = sum_{bits k of t} b[k+1], t = index >> (L+1); forward
//      L = m-1 down to 0.  Elements are in the tower basis of cantor.hpp,
//      two to a unit of four words; a thread holds four units and takes two
//      levels between two exchanges through LDS; a pass over memory
//      takes eight levels.
#include "gf2t_internal.hpp"
#include "cantor.hpp"
#include "../../include/gf2t.h"
#include <vector>
#include <mutex>
#include <condition_variable>
#include <cstring>
#include <algorithm>
#include <atomic>
#include <cstddef>

namespace {

using cantor_host::FFT_MAX_M;
// of the knobs fft_tile_<m> (see passes_for) and fft_low_bits (no effect)
constexpr int FFT_TILE_BITS = 13, FFT_MIN_TILE_BITS = 6;
constexpr int FFT_LOW_BITS = 4;
constexpr int PACK_LIST = 12;   // four matrix entries + four vector pairs
constexpr int CONV_ONE_TILE = 13;   // largest conversion done in one tile
constexpr int CONV_TILE32 = 13, CONV_TILE64 = 12;

__constant__ TwEnt c_tw[4][256];
__device__ FftTables g_tab;

// One operand of a transform: n 32-bit chunks at src (the last masked to
// mask, xor0 XORed into the first), and the buffer its converted
// coefficients go to (8-byte aligned: they are read two at a time).
struct Operand {
    const u32 *src;
    u32 *lch;
    u64 n;
    u32 mask, xor0;
};
// The operands of a launch, blockIdx selecting one: a list in the launch
// arguments (list = null, group = 0), a list in device memory, or two
// groups of `group` operands, sources sstride[.] and buffers lstride apart.
struct Operands {
    const Operand *list;
    u32 group;
    u64 sstride[2], lstride;   // 32-bit words
    Operand op[PACK_LIST];
};
GF2T_DEV Operand operand(const Operands &o, u32 y) {
    if (o.list) return o.list[y];
    if (!o.group) return o.op[y];
    const u32 g = y / o.group, i = y - g * o.group;
    Operand r = o.op[g];
    r.src += (u64)i * (g ? o.sstride[1] : o.sstride[0]);
    r.lch += (u64)i * o.lstride;
    return r;
}
// chunk k, zero from n on
GF2T_DEV u32 chunk(const Operand &o, u64 k) {
    if (k >= o.n) return 0;
    u32 v = o.src[k];
    if (k == o.n - 1) v &= o.mask;
    if (k == 0) v ^= o.xor0;
    return v;
}

// where a conversion reads and writes: an operand's chunks (the first
// launch from src, the others in place in lch), or a transform's elements
struct ChunkIo {
    Operand o;
    bool first;
    typedef u32 type;
    GF2T_DEV bool any(u64 i) const { return i < o.n; }
    GF2T_DEV u32 load(u64 i) const {
        if (first) return chunk(o, i);
        return i < o.n ? o.lch[i] : 0;
    }
    GF2T_DEV void store(u64 i, u32 v) const {
        if (i < o.n) o.lch[i] = v;
    }
};
struct ElemIo {
    u64 *f;
    u64 n;
    typedef u64 type;
    GF2T_DEV bool any(u64) const { return true; }
    GF2T_DEV u64 load(u64 i) const { return i < n ? f[i] : 0; }
    GF2T_DEV void store(u64 i, u64 v) const {
        if (i < n) f[i] = v;
    }
};

constexpr int CONV_THREADS = 256;
constexpr u32 CONV_EDGE_RHO = 4;   // columns of the edges per block

// One group of K expansion steps (ConvStep): blockIdx.y is the block of
// 2^K rows; the first colblocks blocks take a skewed column per thread,
// all rows of it in registers, in place; the others the columns at the
// rows' ends, in LDS.
template <int K, bool INV, class Io>
GF2T_DEV void conv_step_block(const Io &io, const ConvStep &s, u32 colblocks,
                              typename Io::type *lds) {
    typedef typename Io::type E;
    constexpr int R = 1 << K;
    const u64 base = (u64)blockIdx.y << (s.hb + K);
    if (!io.any(base)) return;   // whole block
    if (blockIdx.x < colblocks) {
        const u32 t = blockIdx.x * CONV_THREADS + threadIdx.x;
        if (t >= conv_full(s)) return;
        E x[R];
#pragma unroll
        for (int k = 0; k < R; k++) x[k] = io.load(base + ((u64)k << s.hb) + conv_col(s, t, k));
#pragma unroll
        for (int j = 0; j < K; j++) {
            const int e = INV ? j : K - 1 - j;
#pragma unroll
            for (int k = 0; k < R; k++)
                if ((k >> e) & 1) x[k ^ (1 << e)] ^= x[k];
        }
#pragma unroll
        for (int k = 0; k < R; k++) io.store(base + ((u64)k << s.hb) + conv_col(s, t, k), x[k]);
        return;
    }
    // edge: rho0 .. rho0 + nr of the unit, R x R coefficients each
    const u32 unit = 1u << s.ub, nr = unit < CONV_EDGE_RHO ? unit : CONV_EDGE_RHO;
    const int lr = s.ub < 2 ? s.ub : 2;
    const u32 rho0 = (blockIdx.x - colblocks) * nr;
    const u32 total = (u32)(R * R) << lr;
    constexpr int PER = (R * R * CONV_EDGE_RHO + CONV_THREADS - 1) / CONV_THREADS;
    E v[PER];
    auto mem = [&](u32 i) {
        const u32 rho = i & (nr - 1), q = (i >> lr) & (R - 1), k = i >> (lr + K);
        return base + ((u64)k << s.hb) + conv_edge(s, (int)k, q, rho0 + rho);
    };
#pragma unroll
    for (int j = 0; j < PER; j++) {
        const u32 i = threadIdx.x + j * CONV_THREADS;
        v[j] = i < total ? io.load(mem(i)) : 0;
    }
#pragma unroll
    for (int j = 0; j < PER; j++) {
        const u32 i = threadIdx.x + j * CONV_THREADS;
        if (i < total) lds[i] = v[j];
    }
    __syncthreads();
    for (int j = 0; j < K; j++) {
        const int e = INV ? j : K - 1 - j;
        for (u32 i = threadIdx.x; i < total / 2; i += CONV_THREADS) {
            const u32 rho = i & (nr - 1);
            conv_edge_pair([&](u32 l) -> E & { return lds[(l << lr) | rho]; }, K, e, INV, i >> lr);
        }
        __syncthreads();
    }
#pragma unroll
    for (int j = 0; j < PER; j++) {
        const u32 i = threadIdx.x + j * CONV_THREADS;
        if (i < total) io.store(mem(i), lds[i]);
    }
}
template <int K>
__global__ __launch_bounds__(CONV_THREADS) void k_conv_step32(const Operands ops, const ConvStep s,
                                                              u32 colblocks, int first) {
    __shared__ u32 lds[(1 << (2 * K)) * CONV_EDGE_RHO];
    conv_step_block<K, false>(ChunkIo{operand(ops, blockIdx.z), first != 0}, s, colblocks, lds);
}
template <int K, bool INV>
__global__ __launch_bounds__(CONV_THREADS) void k_conv_step64(u64 *__restrict__ f, u64 f_stride,
                                                              const ConvStep s, u32 colblocks) {
    __shared__ u64 lds[(1 << (2 * K)) * CONV_EDGE_RHO];
    conv_step_block<K, INV>(ElemIo{f + (u64)blockIdx.z * f_stride, ~0ULL}, s, colblocks, lds);
}

// The conversion's other part: a tile in LDS (one coefficient in 17 left
// out, so that the threads' runs of sixteen fall on different banks),
// 16 coefficients per thread, stage by stage in registers.
GF2T_DEV u32 conv_pad(u32 i) { return i + (i >> 4); }
template <bool INV, class Io>
GF2T_DEV void conv_tile_block(const Io &io, const ConvTile &t, typename Io::type *lds) {
    typedef typename Io::type E;
    const u64 base = tile_base(t, blockIdx.x);
    if (!io.any(base)) return;   // whole block
    const u32 q = threadIdx.x, nthr = blockDim.x;   // 16 coefficients each
    E v[16];
#pragma unroll
    for (int j = 0; j < 16; j++) v[j] = io.load(base + tile_mem(t, q + j * nthr));
#pragma unroll
    for (int j = 0; j < 16; j++) lds[conv_pad(q + j * nthr)] = v[j];
    __syncthreads();
    for (int i = 0; i < t.n; i++) {
        const ConvStep s = t.st[INV ? t.n - 1 - i : i];
        conv_tile_stage<INV, E>([&](u32 l) -> E & { return lds[conv_pad(l)]; }, q, nthr, s);
        __syncthreads();
    }
#pragma unroll
    for (int j = 0; j < 16; j++)
        io.store(base + tile_mem(t, q + j * nthr), lds[conv_pad(q + j * nthr)]);
}
__global__ __launch_bounds__(512) void k_conv_tile32(const Operands ops, const ConvTile t,
                                                     int first) {
    extern __shared__ u32 lds32[];
    conv_tile_block<false>(ChunkIo{operand(ops, blockIdx.y), first != 0}, t, lds32);
}
template <bool INV>
__global__ __launch_bounds__(512) void k_conv_tile64(u64 *__restrict__ f, u64 f_stride, u64 n,
                                                     const ConvTile t) {
    extern __shared__ u64 lds64[];
    conv_tile_block<INV>(ElemIo{f + (u64)blockIdx.y * f_stride, n}, t, lds64);
}

// ------------------------------------------------------ small transforms
// A whole transform of up to 2^FFT_SMALL points in one block, in the
// polynomial basis: the conversion's one tile, then the butterflies with
// GF(2^64) products.  Such a transform is all latency: by the kernels below
// it is two or three launches, each of which first copies up to 37 KB of
// tables (2^2 points: 10.3 us and 3.0 here, 2^8 16.8 and 9.5, 2^10 21.8 and
// 15.0; 2^11, two elements a thread, 25.5 and 24).
constexpr int FFT_SMALL = 10;
struct SmallFft {
    int m;
    u64 b[FFT_SMALL];   // W(t) = sum of b[k] over the bits k of t
    ConvTile t;
};
template <bool INV>
__global__ __launch_bounds__(1 << (FFT_SMALL - 1)) void k_fft_small(u64 *__restrict__ f,
                                                                    const SmallFft A) {
    __shared__ u64 lds[(1 << FFT_SMALL) + (1 << (FFT_SMALL - 4))];
    auto x = [&](u32 i) -> u64 & { return lds[conv_pad(i)]; };
    const u32 n = 1u << A.m, tile = n < 16 ? 16 : n, q = threadIdx.x, nthr = blockDim.x;
    for (u32 i = q; i < tile; i += nthr) x(i) = i < n ? f[i] : 0;
    __syncthreads();
    auto convert = [&] {
        for (int i = 0; i < A.t.n; i++) {
            if (q < tile / 16) conv_tile_stage<INV, u64>(x, q, tile / 16, A.t.st[INV ? A.t.n - 1 - i : i]);
            __syncthreads();
        }
    };
    if (!INV) convert();
    for (int i = 0; i < A.m; i++) {
        const int L = INV ? i : A.m - 1 - i;
        for (u32 k = q; k < n / 2; k += nthr) {
            const u32 t = k >> L, at = k + (t << L);
            u64 g = x(at), h = x(at + (1u << L)), w = 0;
            for (int j = 0; j < A.m - 1 - L; j++) w ^= (t >> j) & 1 ? A.b[j] : 0;
            if (INV) h ^= g;
            if (L < A.m - 1) g ^= gf64_mul(w, h);
            if (!INV) h ^= g;
            x(at) = g;
            x(at + (1u << L)) = h;
        }
        __syncthreads();
    }
    if (INV) convert();
    for (u32 i = q; i < n; i += nthr) f[i] = x(i);
}

// ------------------------------------------------------------ butterflies
// n 16-byte words from memory to LDS, four loads in flight per thread
GF2T_DEV void copy_lds(void *dst_, const void *src_, u32 n) {
    uint4 *dst = (uint4 *)dst_;
    const uint4 *src = (const uint4 *)src_;
    const u32 nthr = blockDim.x;
    for (u32 i = threadIdx.x; i < n; i += 4 * nthr) {
        const u32 i1 = i + nthr, i2 = i1 + nthr, i3 = i2 + nthr, e = n - 1;
        const uint4 v0 = src[i], v1 = src[i1 < e ? i1 : e], v2 = src[i2 < e ? i2 : e],
                    v3 = src[i3 < e ? i3 : e];
        dst[i] = v0;
        if (i1 < n) dst[i1] = v1;
        if (i2 < n) dst[i2] = v2;
        if (i3 < n) dst[i3] = v3;
    }
}
// LDS copies of the GF(2^8) multiply tables and, behind them, the GF(2^32)
// basis tables (FftTables' first members)
struct MulLds {
    uint4 A[256];
    u32 B[256];
    GF2T_DEV Mul8 operator()(u32 off) const {
        const unsigned char *p = reinterpret_cast<const unsigned char *>(A);
        const uint4 a = *reinterpret_cast<const uint4 *>(p + off);
        return Mul8{a.x, a.y, a.z, a.w,
                    *reinterpret_cast<const u32 *>(p + sizeof(A) + (off >> 2))};
    }
};
struct ProdLds {
    u32 d32[4][256], d5[4][256], b32[4][256];
};
static_assert(sizeof(MulLds) + sizeof(ProdLds) == offsetof(FftTables, emb), "table layout");
// what a pass reads and writes: units; the chunks of an operand (lch:
// converted ones); elements in the polynomial basis
enum { IO_UNITS = 0, IO_CHUNKS = 1, IO_LCH = 2, IO_PLAIN = 3 };

// transform buffers are the caller's: 8-byte aligned
typedef u32 G4 __attribute__((ext_vector_type(4), aligned(8)));
typedef u64 G2 __attribute__((ext_vector_type(2), aligned(8)));
typedef u64 Emb[256];
GF2T_DEV U4 load_unit(const U4 *f, u32 i, int io, const Operand &o, const Emb *emb) {
    if (io == IO_UNITS) {
        const G4 v = reinterpret_cast<const G4 *>(f)[i];
        return U4{{v.x, v.y, v.z, v.w}};
    }
    if (io == IO_PLAIN) {
        const G2 v = reinterpret_cast<const G2 *>(f)[i];
        return unit_embed64(v.x, v.y, emb);
    }
    U4 z = {{0, 0, 0, 0}};
    const u64 k = 2 * (u64)i;
    if (k >= o.n) return z;
    u32 e, g;
    if (io == IO_LCH) {
        if (k + 1 < o.n) {
            const uint2 v = *reinterpret_cast<const uint2 *>(o.lch + k);
            e = v.x;
            g = v.y;
        } else {
            e = o.lch[k];
            g = 0;
        }
    } else {
        e = chunk(o, k);
        g = chunk(o, k + 1);
    }
    return unit_embed32(e, g, emb);
}
GF2T_DEV void store_unit(U4 *f, u32 i, const U4 &u, int io, const Emb *une) {
    if (io == IO_UNITS) {
        reinterpret_cast<G4 *>(f)[i] = G4{u.w[0], u.w[1], u.w[2], u.w[3]};
        return;
    }
    u64 e, g;
    unit_unembed(u, une, e, g);
    reinterpret_cast<G2 *>(f)[i] = G2{e, g};
}
// copy a basis table (8 x 256 entries; 4 x 256 for chunks) to LDS
GF2T_DEV void load_basis(u64 *dst, const u64 (*src)[256], int bytes) {
    copy_lds(dst, src, (u32)bytes * 128);
}
GF2T_DEV u32 uniform32(u32 v) { return __builtin_amdgcn_readfirstlane(v); }

// One butterfly pass over the window of P (see BfPass): 2^RB units per
// thread, RB levels, an exchange through LDS, and so on.  A block takes
// every gridDim.x-th tile, so that the tables it copies to LDS (5 KB, and
// 8 or 16 KB of a basis table) serve several tiles of 16 KB.
template <int CLS, bool INV>
__global__ __launch_bounds__(256) void k_bfly(u64 *__restrict__ f_, u64 f_stride, const BfPass P,
                                              const Operands ops, int in, int out) {
    constexpr int R = 1 << RB;
    extern __shared__ __align__(16) unsigned char lds_raw[];
    MulLds &tab = *reinterpret_cast<MulLds *>(lds_raw);
    U4 *ex = reinterpret_cast<U4 *>(lds_raw + sizeof(MulLds));
    u64 *basis = reinterpret_cast<u64 *>(ex + (P.w > RB ? 1u << P.tb : 0u));
    U4 *f = reinterpret_cast<U4 *>(f_ + (u64)blockIdx.y * f_stride);
    Operand o{};
    if (in == IO_CHUNKS || in == IO_LCH) o = operand(ops, blockIdx.y);
    copy_lds(lds_raw, &g_tab, sizeof(MulLds) / 16);
    if (in != IO_UNITS) load_basis(basis, g_tab.emb, in == IO_PLAIN ? 8 : 4);
    if (out == IO_PLAIN) load_basis(basis, g_tab.une, 8);   // never both
    __syncthreads();
    const u32 tid = threadIdx.x;
    const int ns = bf_stages(P);
    const Emb *emb = reinterpret_cast<const Emb *>(basis);
    const u32 tiles = 1u << (P.m - 1 - P.tb);
    for (u32 blk = blockIdx.x; blk < tiles; blk += gridDim.x) {
        const BfTile T = bf_tile(P, blk);
        U4 x[R];
        int s = INV ? ns - 1 : 0;
#pragma unroll
        for (int r = 0; r < R; r++)
            x[r] = load_unit(f, bf_unit(P, T, bf_local(P, s, tid, r)), in, o, emb);
#pragma nounroll
        for (int k = 0;; k++) {
            TwEnt W[RB];
            bf_twiddles(P, T, s, tid, c_tw, W);
            fft_stage<CLS, INV>(x, bf_active(P, s), W, bf_zero(P, T, s), tab);
            if (k == ns - 1) break;
            __syncthreads();   // the last exchange is read
#pragma unroll
            for (int r = 0; r < R; r++) ex[bf_local(P, s, tid, r)] = x[r];
            s += INV ? -1 : 1;
            __syncthreads();
#pragma unroll
            for (int r = 0; r < R; r++) x[r] = ex[bf_local(P, s, tid, r)];
        }
#pragma unroll
        for (int r = 0; r < R; r++)
            store_unit(f, bf_unit(P, T, bf_local(P, s, tid, r)), x[r], out, emb);
    }
}

// ---- the low levels
constexpr u32 LO_UNITS = 64u << RB;              // per wave
// words of a wave's exchange plane, and of the two rows of units that the
// waves of a pair hand over
constexpr u32 LO_EXCH = 2 * 64 * 4;
static_assert(LO_EXCH >= (64u << RB) + (4u << RB), "a padded plane of one word per unit");

// (linear over disjoint bits, so a row's place is the lane's plus a constant)
GF2T_HD constexpr u32 lo_pad(u32 u) { return u + (u >> 4); }
// the wave's units from the layout of one stage to that of another, a word
// of each unit at a time through the wave's own plane in LDS
template <int FROM, int TO>
GF2T_DEV void lo_exchange(U4 *x, u32 lane, u32 *plane) {
    u32 *from = plane + lo_pad(lo_unit(FROM, lane, 0));
    const u32 *to = plane + lo_pad(lo_unit(TO, lane, 0));
#pragma unroll
    for (int p = 0; p < 4; p++) {
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int r = 0; r < (1 << RB); r++) from[lo_pad((u32)r << lo_pos(FROM))] = x[r].w[p];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int r = 0; r < (1 << RB); r++) x[r].w[p] = to[lo_pad((u32)r << lo_pos(TO))];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
}
template <int S, int CLS, bool INV>
GF2T_DEV void lo_stage(U4 *x, int m, u32 ubase, u32 lane, const MulLds &tab, const TwEnt *hi) {
    TwEnt W[RB], W0;
    lo_twiddles<S>(ubase, lane, c_tw, hi, W, W0);
    if (INV && S == lo_stages() - 1) fft_level0<CLS, true>(x, W0, tab);
    fft_stage<CLS, INV>(x, lo_active(m, S), W, false, tab);
    if (!INV && S == lo_stages() - 1) fft_level0<CLS, false>(x, W0, tab);
}
static_assert(lo_stages() == 4, "the stages are spelled out below");
template <int CA, int CB>
GF2T_DEV void lo_forward(U4 *x, int m, u32 ubase, u32 lane, const MulLds &tab, const TwEnt *hi,
                         u32 *plane) {
    lo_stage<0, CA, false>(x, m, ubase, lane, tab, hi);
    lo_exchange<0, 1>(x, lane, plane);
    lo_stage<1, CB, false>(x, m, ubase, lane, tab, hi);
    lo_exchange<1, 2>(x, lane, plane);
    lo_stage<2, CB, false>(x, m, ubase, lane, tab, hi);
    lo_exchange<2, 3>(x, lane, plane);
    lo_stage<3, CB, false>(x, m, ubase, lane, tab, hi);
}
template <int CA, int CB>
GF2T_DEV void lo_inverse(U4 *x, int m, u32 ubase, u32 lane, const MulLds &tab, const TwEnt *hi,
                         u32 *plane) {
    lo_stage<3, CB, true>(x, m, ubase, lane, tab, hi);
    lo_exchange<3, 2>(x, lane, plane);
    lo_stage<2, CB, true>(x, m, ubase, lane, tab, hi);
    lo_exchange<2, 1>(x, lane, plane);
    lo_stage<1, CB, true>(x, m, ubase, lane, tab, hi);
    lo_exchange<1, 0>(x, lane, plane);
    lo_stage<0, CA, true>(x, m, ubase, lane, tab, hi);
}
GF2T_DEV U4 unit_select(bool c, const U4 &a, const U4 &b) {
    return U4{{c ? a.w[0] : b.w[0], c ? a.w[1] : b.w[1], c ? a.w[2] : b.w[2],
               c ? a.w[3] : b.w[3]}};
}
enum { LO_FWD = 0, LO_INV = 1, LO_MUL = 2 };
// Levels 7..0 of a transform (LO_FWD, LO_INV), or, of two transforms, both
// forward, their product and the inverse of it in one pass (LO_MUL: f and
// g, into f).  A wave takes LO_UNITS consecutive units; LO_MUL pairs two
// waves, one per operand, which then multiply half of the units each, and
// the first inverts (one wave for both operands took 164 registers instead
// of about 100 and half as long again at sizes that do not fill the chip).
template <int CA, int CB, int DIR>
__global__ __launch_bounds__(256) void k_low(u64 *__restrict__ f_, u64 f_stride,
                                             const u64 *__restrict__ g_, int m,
                                             const Operands ops, u32 g_op, int in, int out) {
    constexpr int R = 1 << RB;
    constexpr int LAST = lo_stages() - 1;
    constexpr bool MUL = DIR == LO_MUL;
    extern __shared__ __align__(16) unsigned char lds_raw[];
    MulLds &tab = *reinterpret_cast<MulLds *>(lds_raw);
    const ProdLds &pt = *reinterpret_cast<const ProdLds *>(lds_raw + sizeof(MulLds));
    constexpr u32 TABS = sizeof(MulLds) + (MUL ? sizeof(ProdLds) : 0);
    TwEnt *hi = reinterpret_cast<TwEnt *>(lds_raw + TABS);
    const u32 wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    u32 *planes = reinterpret_cast<u32 *>(hi + 4);
    u32 *plane = planes + wave * LO_EXCH;
    u64 *basis = reinterpret_cast<u64 *>(planes + (blockDim.x >> 6) * LO_EXCH);
    const Emb *emb = reinterpret_cast<const Emb *>(basis);
    copy_lds(lds_raw, &g_tab, TABS / 16);
    if (threadIdx.x < 4) hi[threadIdx.x] = tw_of(g_tab.tw, threadIdx.x << 7);
    if (in != IO_UNITS) load_basis(basis, g_tab.emb, in == IO_PLAIN ? 8 : 4);
    __syncthreads();
    const u32 units = 1u << (m - 1);
    const u32 per = (blockDim.x >> 6) >> (MUL ? 1 : 0);   // runs of units per block
    const bool second = MUL && (wave & 1);                // the wave of operand g
    const u32 ubase = uniform32((blockIdx.x * per + (MUL ? wave >> 1 : wave)) * LO_UNITS);
    const bool act = ubase < units;                       // whole wave
    U4 *f = reinterpret_cast<U4 *>(f_ + (u64)blockIdx.y * f_stride);
    U4 x[R];
    if (act) {
        const U4 *src = second ? reinterpret_cast<const U4 *>(g_ + (u64)blockIdx.y * f_stride) : f;
        Operand o{};
        if (in == IO_CHUNKS || in == IO_LCH) o = operand(ops, blockIdx.y + (second ? g_op : 0));
#pragma unroll
        for (int r = 0; r < R; r++) {
            const u32 i = ubase + lo_unit(0, lane, r);
            x[r] = i < units ? load_unit(src, i, in, o, emb) : U4{{0, 0, 0, 0}};
        }
        if (DIR != LO_INV) lo_forward<CA, CB>(x, m, ubase, lane, tab, hi, plane);
        if (DIR == LO_FWD) lo_exchange<LAST, 0>(x, lane, plane);   // to contiguous stores
        if (DIR == LO_INV) lo_exchange<0, LAST>(x, lane, plane);
    }
    if (MUL) {
        // rows 0 and 1 are multiplied by the first wave of a pair, 2 and 3
        // by the second: each hands the other's rows over, then the second
        // its products, through the planes (a unit is four words)
        static_assert(R == 4 && LO_EXCH >= 2 * 64 * 4, "two rows fit a plane");
        U4 *mine = reinterpret_cast<U4 *>(plane);
        const U4 *other = reinterpret_cast<const U4 *>(planes + (wave ^ 1) * LO_EXCH);
        __syncthreads();
        mine[lane] = unit_select(second, x[0], x[2]);
        mine[64 + lane] = unit_select(second, x[1], x[3]);
        __syncthreads();
        U4 y0 = other[lane], y1 = other[64 + lane];
        U4 z0 = unit_select(second, x[2], x[0]), z1 = unit_select(second, x[3], x[1]);
        __syncthreads();
#pragma nounroll
        for (int k = 0; k < 2; k++) {
            const U4 v = unit_mul(z0, y0, pt.d32, pt.d5, pt.b32);
            z0 = z1;
            y0 = y1;
            z1 = v;
        }
        if (second) {
            mine[lane] = z0;
            mine[64 + lane] = z1;
        }
        __syncthreads();
        x[0] = z0;
        x[1] = z1;
        x[2] = other[lane];
        x[3] = other[64 + lane];
    }
    if (DIR != LO_FWD && act && !second)
        lo_inverse<CA, CB>(x, m, ubase, lane, tab, hi, plane);
    if (out == IO_PLAIN) {
        __syncthreads();
        load_basis(basis, g_tab.une, 8);
        __syncthreads();
    }
    if (act && !second) {
#pragma unroll
        for (int r = 0; r < R; r++) {
            const u32 i = ubase + lo_unit(0, lane, r);
            if (i < units) store_unit(f, i, x[r], out, emb);
        }
    }
}

// --------------------------------------------------- small products
// All chunk products of two operands, without a transform: c_k = sum of
// a_i b_(k-i), carry-less, i over the shorter operand.  A block takes
// SC_OUT outputs and SC_IN values of i, its four waves a quarter of them
// each, a lane two outputs; the products of one bit class (see clmul32)
// are XORed up as they come and the classes merged once at the end, so a
// 32 x 32 product costs 16 multiply-adds and 12 XORs.  Block (t, c) writes
// the part of the outputs [SC_OUT t, SC_OUT (t + 1)) that comes from the
// i in [SC_IN c, SC_IN (c + 1)) to part[c][.].  Bounded by the multiply-adds
// (a quarter of the VALU rate).
//
// From SC_KARA chunks on, two levels of Karatsuba's splitting by the
// chunks' index: of even, odd and all (summed) chunks, and of each again,
// nine products of a quarter of the length stand for sixteen.  The operand
// sums are formed as the chunks are read, and the products are put together
// by k_school_kara.  Two 132049-bit operands: 24 us, of which one product
// of all chunks took 27; 262,144 bits: 48 and 72 us; below SC_KARA chunks
// the nine are no faster (60,000 bits: 12.6 and 12.2 us).
constexpr u32 SC_OUT = 128, SC_IN = 128, SC_KARA = 1024;
struct SchoolShape {
    u32 na, nb;         // chunks (of a quarter where split), na <= nb
    u32 nout, nparts;   // na + nb - 1 outputs; parts
    u32 np;             // products: 1, or 9 where split
};
// of product p, whether the chunks r mod 4 are in its operands: p / 3 picks
// by the index's bit 0 (0: even, 1: odd, 2: both), p % 3 by its bit 1
GF2T_HD bool kara_picks(u32 p, u32 r) {
    const u32 u = p / 3, v = p % 3;
    return (u == 2 || u == (r & 1)) && (v == 2 || v == (r >> 1));
}
// chunk i of an operand of product p, 0 below the first and past the last;
// its loads do not wait for one another
GF2T_DEV u32 school_chunk(const Operand &o, u32 np, u32 p, int i) {
    if (np == 1) return i >= 0 ? chunk(o, (u64)i) : 0;
    u32 w[4], v = 0;
    const u32 n = (u32)o.n;
#pragma unroll
    for (u32 r = 0; r < 4; r++) {
        const u32 k = i >= 0 ? 4 * (u32)i + r : 0;
        w[r] = o.src[k < n ? k : n - 1];
    }
#pragma unroll
    for (u32 r = 0; r < 4; r++) {
        const u32 k = 4 * (u32)i + r;
        u32 x = w[r];
        x &= k == n - 1 ? o.mask : ~0u;
        x ^= k == 0 ? o.xor0 : 0u;
        v ^= i >= 0 && k < n && kara_picks(p, r) ? x : 0u;
    }
    return v;
}
// the parts that reach output tile t: c in [first, last]
GF2T_HD u32 school_first(const SchoolShape &s, u32 t) {
    const u32 k0 = t * SC_OUT;
    return k0 >= s.nb + SC_IN - 1 ? (k0 - s.nb + 1 - (SC_IN - 1) + SC_IN - 1) / SC_IN : 0;
}
GF2T_HD u32 school_last(const SchoolShape &s, u32 t) { return t < s.nparts - 1 ? t : s.nparts - 1; }

// products of any sizes without a transform: one of them, and a block for
// each of their tiles that has work (of the product's words: t its run of
// SP_WORDS)
struct SchoolJob {
    Operand a, b;   // a the shorter
    SchoolShape s;
    u64 *part, *out;
    u64 owords;
};
struct SchoolBlock {
    u32 job;
    unsigned short t, c;
};
// SC_JOBS: of a list of jobs, else of the operands y and b_op + y (swapped
// if y is the longer).  SC_MAT: the operands are a matrix m0..m3 and vector
// pairs (see gf2t_mat2n_host), product y = 4 pair + 2 o + h of entry 2 o + h
// and element h.  SC_FULL: a product split in nine, whose tiles are
// full but for a few (the tests below cost two 320,000-bit operands 2%).  The
// others skip what a tile has past their operands or outside its triangle: a
// slab of 4096 residues of 89 bits takes 23 us instead of 130, one of 20,000
// of 3071 bits 473 (620 by transforms).
enum { SC_SLACK = 0, SC_FULL = 1, SC_JOBS = 2, SC_MAT = 3 };
template <int FORM>
__global__ __launch_bounds__(256) void k_school(const Operands ops, u32 b_op, int swap,
                                                const SchoolShape shape, u64 *__restrict__ part,
                                                u64 part_stride, const SchoolJob *__restrict__ jobs,
                                                const SchoolBlock *__restrict__ blocks) {
    static_assert(SC_OUT == 128 && SC_IN == 128, "two outputs per lane, 32 values per wave, a b per thread");
    constexpr bool FULL = FORM == SC_FULL, JOBS = FORM == SC_JOBS;
    __shared__ u32 bs[SC_OUT + SC_IN];
    __shared__ u64 sum[4][SC_OUT];
    const SchoolBlock blk = JOBS ? blocks[blockIdx.x] : SchoolBlock{};
    const SchoolShape s = JOBS ? jobs[blk.job].s : shape;
    const u32 c = JOBS ? blk.c : blockIdx.y, t = JOBS ? blk.t : c + blockIdx.x;
    const u32 y = JOBS ? 0 : blockIdx.z / s.np, p = JOBS ? 0 : blockIdx.z % s.np;
    if (!JOBS && (c < school_first(s, t) || c > school_last(s, t))) return;   // whole block
    const u32 ya = FORM == SC_MAT ? y & 3 : y;
    const u32 yb = FORM == SC_MAT ? 4 + 2 * (y >> 2) + (y & 1) : y + b_op;
    const Operand oa = JOBS ? jobs[blk.job].a : operand(ops, swap ? yb : ya);
    const Operand ob = JOBS ? jobs[blk.job].b : operand(ops, swap ? ya : yb);
    if (JOBS) part = jobs[blk.job].part;
    const int k0 = (int)(t * SC_OUT), i0 = (int)(c * SC_IN);
    const int j0 = k0 - i0 - (int)(SC_IN - 1);   // b index of bs[0]
    const u32 wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int iw = i0 + (int)wave * 32;
    const u32 bv = school_chunk(ob, s.np, p, j0 + (int)threadIdx.x);
    const u32 av = lane < 32 ? school_chunk(oa, s.np, p, iw + (int)lane) : 0;
    bs[threadIdx.x] = bv;
    __syncthreads();
    const u32 m0 = 0x11111111u;
    u64 acc[2][4] = {};
    const u32 at = lane + (SC_IN - 1) - wave * 32;   // bs index of output `lane`, i = iw
    auto term = [&](int i, int o) {
        const u32 a = __builtin_amdgcn_readlane(av, i);
        const u64 a0 = a & m0, a1 = a & (m0 << 1), a2 = a & (m0 << 2), a3 = a & (m0 << 3);
        const u32 b = bs[at - i + 64 * o];
        const u64 b0 = b & m0, b1 = b & (m0 << 1), b2 = b & (m0 << 2), b3 = b & (m0 << 3);
        acc[o][0] = xor3(acc[o][0], a0 * b0 + a1 * b3, a2 * b2) ^ (a3 * b1);
        acc[o][1] = xor3(acc[o][1], a0 * b1 + a2 * b3, a1 * b0 + a3 * b2);
        acc[o][2] = xor3(acc[o][2], a0 * b2 + a3 * b3, a1 * b1) ^ (a2 * b0);
        acc[o][3] = xor3(xor3(acc[o][3], a0 * b3, a1 * b2), a2 * b1, a3 * b0);
    };
    // the wave's values that there are (an odd last one and a 0), and those
    // 64 of its outputs that any of them reaches
    const int i1 = FULL ? 0 : (int)uniform32((u32)iw);
    const int left = (int)s.na - i1, ni = FULL || left > 32 ? 32 : left;
    auto reached = [&](int k) { return FULL || (k + 63 >= i1 && k < i1 + ni - 1 + (int)s.nb); };
    if (reached(k0) && reached(k0 + 64)) {
        for (int i = 0; i < ni; i += 2) {
            term(i, 0);
            term(i, 1);
            term(i + 1, 0);
            term(i + 1, 1);
        }
    } else if (reached(k0)) {
        for (int i = 0; i < ni; i += 2) {
            term(i, 0);
            term(i + 1, 0);
        }
    } else if (reached(k0 + 64)) {
        for (int i = 0; i < ni; i += 2) {
            term(i, 1);
            term(i + 1, 1);
        }
    }
    const u64 q = 0x1111111111111111ULL;
#pragma unroll
    for (int o = 0; o < 2; o++)
        sum[wave][lane + 64 * o] =
            sel64(q, acc[o][0], sel64(q << 1, acc[o][1], sel64(q << 2, acc[o][2], acc[o][3])));
    __syncthreads();
    const u32 k = (u32)k0 + threadIdx.x;
    if (threadIdx.x < SC_OUT && k < s.nout)
        part[(u64)y * part_stride + (u64)(p * s.nparts + c) * s.nout + k] =
            xor3(sum[0][threadIdx.x], sum[1][threadIdx.x], sum[2][threadIdx.x]) ^
            sum[3][threadIdx.x];
}
// word k of the product: chunk coefficients 2k - 1, 2k and 2k + 1
struct SchoolWords {
    const u64 *part;
    SchoolShape s;
    GF2T_DEV u64 coef(u64 k) const {
        if (k >= s.nout) return 0;
        u64 v = 0;
        const u32 t = (u32)k / SC_OUT, hi = school_last(s, t);
        for (u32 c = school_first(s, t); c <= hi; c++) v ^= part[(u64)c * s.nout + k];
        return v;
    }
    GF2T_DEV u64 operator()(size_t w) const {
        const u64 k = 2 * (u64)w;
        u64 v = coef(k) ^ (coef(k + 1) << 32);
        if (w) v ^= coef(k - 1) >> 32;
        return v;
    }
};
// the words from w0 on of a product, or of the sum of SUMS: a block adds up
// the parts of 2 SP_WORDS + 1 chunk coefficients, four threads each, and
// writes SP_WORDS words
constexpr u32 SP_WORDS = 32;
template <int SUMS>
GF2T_DEV void school_product(const u64 *__restrict__ part, const SchoolShape &s, u32 w0,
                             u64 *__restrict__ out, size_t owords) {
    __shared__ u64 sum[4][2 * SP_WORDS + 1];   // coefficients k0 - 1 ..
    const u32 g = threadIdx.x & 3;
    for (u32 x = threadIdx.x >> 2; x < 2 * SP_WORDS + 1; x += 64) {
        u64 v = 0;
        const u64 k = 2 * (u64)w0 + x;   // coefficient k - 1
        if (k >= 1 && k - 1 < s.nout) {
            const u32 t = (u32)(k - 1) / SC_OUT, hi = school_last(s, t);
#pragma unroll
            for (u32 j = 0; j < SUMS; j++)
#pragma unroll 4
                for (u32 c = school_first(s, t) + g; c <= hi; c += 4)
                    v ^= part[(u64)(j * s.nparts + c) * s.nout + (k - 1)];
        }
        sum[g][x] = v;
    }
    __syncthreads();
    auto coef = [&](u32 x) { return xor3(sum[0][x], sum[1][x], sum[2][x]) ^ sum[3][x]; };
    const u32 x = threadIdx.x;
    if (x < SP_WORDS && w0 + x < owords)
        out[w0 + x] = coef(2 * x + 1) ^ (coef(2 * x + 2) << 32) ^ (coef(2 * x) >> 32);
}
__global__ __launch_bounds__(256) void k_school_product(const u64 *__restrict__ part,
                                                        const SchoolShape s,
                                                        u64 *__restrict__ out, size_t owords) {
    school_product<1>(part, s, blockIdx.x * SP_WORDS, out, owords);
}
// output y of a matrix-vector product, the sum of two (SC_MAT)
__global__ __launch_bounds__(256) void k_school_mat(const u64 *__restrict__ part,
                                                    const SchoolShape s, u64 *__restrict__ out,
                                                    size_t owords) {
    const u32 y = blockIdx.y;
    school_product<2>(part + (u64)y * 2 * s.nparts * s.nout, s, blockIdx.x * SP_WORDS,
                      out + y * owords, owords);
}
// of a job's blocks number t is its words' run of SP_WORDS
__global__ __launch_bounds__(256) void k_school_products(const SchoolJob *__restrict__ jobs,
                                                         const SchoolBlock *__restrict__ blocks) {
    const SchoolBlock b = blocks[blockIdx.x];
    const SchoolJob &j = jobs[b.job];
    school_product<1>(j.part, j.s, b.t * SP_WORDS, j.out, j.owords);
}
// The same from nine products: those of the index's bit 1 first,
//   e_2h = E_h + O_(h-1), e_(2h+1) = S_h + E_h + O_h
// (E, O, S: the products of even, odd and all), then those of bit 0 in the
// same way.  A block adds up the parts of the 17 coefficients of each that
// its words need.
__global__ __launch_bounds__(256) void k_school_kara(const u64 *__restrict__ part,
                                                     const SchoolShape s, u64 *__restrict__ out,
                                                     size_t owords) {
    constexpr int H = 2 * SP_WORDS / 4 + 1;
    __shared__ u64 sum[9][H];
    const u32 w0 = blockIdx.x * SP_WORDS;
    if (threadIdx.x < 9 * H) {
        const u32 p = threadIdx.x / H, x = threadIdx.x % H;
        const u32 h = w0 / 2 + x - 1;   // coefficient; none before the first
        u64 v = 0;
        if (w0 / 2 + x >= 1 && h < s.nout) {
            const u32 t = h / SC_OUT, hi = school_last(s, t);
#pragma unroll 4
            for (u32 c = school_first(s, t); c <= hi; c++)
                v ^= part[(u64)(p * s.nparts + c) * s.nout + h];
        }
        sum[p][x] = v;
    }
    __syncthreads();
    // coefficient w0 - 1 + l of the product of bit 0's choice u
    auto half = [&](int u, int l) -> u64 {
        const u64(*q)[H] = &sum[3 * u];
        if (l & 1) return q[0][(l + 1) / 2] ^ q[1][(l - 1) / 2];
        return xor3(q[2][l / 2], q[0][l / 2], q[1][l / 2]);
    };
    // coefficient 2 w0 - 1 + x
    auto coef = [&](int x) -> u64 {
        if (x & 1) return half(0, (x + 1) / 2) ^ half(1, (x - 1) / 2);
        return xor3(half(2, x / 2), half(0, x / 2), half(1, x / 2));
    };
    const int x = (int)threadIdx.x;
    if (x < (int)SP_WORDS && w0 + x < owords)
        out[w0 + x] = coef(2 * x + 1) ^ (coef(2 * x + 2) << 32) ^ (coef(2 * x) >> 32);
}
// the product folded mod x^r + x^s + 1 (s from svec where there is a batch)
__global__ __launch_bounds__(256) void k_school_fold(const u64 *__restrict__ part, u64 part_stride,
                                                     const SchoolShape s, u64 L,
                                                     u64 *__restrict__ out, size_t nw,
                                                     u64 o_stride, u64 r, u64 sv,
                                                     const u64 *__restrict__ svec) {
    const size_t w = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (w >= nw) return;
    out[(u64)blockIdx.y * o_stride + w] =
        fold_words(SchoolWords{part + (u64)blockIdx.y * part_stride, s}, L, r,
                   svec ? svec[blockIdx.y] : sv, w);
}

// overlap-add in gather form: output word w collects chunks 2w-1, 2w, 2w+1
// (blockIdx.y: batch element, F + y*f_stride -> out + y*o_stride)
__global__ void k_overlap_add(const u64 *__restrict__ F, size_t nchunks, u64 *__restrict__ out,
                              size_t owords, u64 f_stride, u64 o_stride) {
    size_t w = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (w >= owords) return;
    F += (u64)blockIdx.y * f_stride;
    out += (u64)blockIdx.y * o_stride;
    size_t k = 2 * w;
    u64 v = 0;
    if (k < nchunks) v ^= F[k];
    if (k + 1 < nchunks) v ^= F[k + 1] << 32;
    if (w && k - 1 < nchunks) v ^= F[k - 1] >> 32;
    out[w] = v;
}

// --------------------------------------------------------- basis (host)
u64 gf64_mul_host(u64 a, u64 b) { return gf64_mul(a, b); }

// y^2 + y = c: Gauss-Jordan on the 64x64 matrix of T(y) = y^2 + y; of the
// two roots (they differ by 1) return the one with bit 0 clear, which is
// the reference's choice (src/gf2_cantor_engine.h:78-110).
bool solve_T(u64 c, u64 &y) {
    u64 row[64];
    int rhs[64];
    for (int j = 0; j < 64; j++) { row[j] = 0; rhs[j] = (int)((c >> j) & 1); }
    for (int i = 0; i < 64; i++) {
        u64 ei = 1ULL << i, t = gf64_mul_host(ei, ei) ^ ei;
        for (int j = 0; j < 64; j++)
            if ((t >> j) & 1) row[j] |= ei;
    }
    int piv[64];
    for (int i = 0; i < 64; i++) piv[i] = -1;
    int rank = 0;
    for (int col = 63; col >= 0; col--) {
        int p = -1;
        for (int j = rank; j < 64; j++)
            if ((row[j] >> col) & 1) { p = j; break; }
        if (p < 0) continue;
        std::swap(row[p], row[rank]);
        std::swap(rhs[p], rhs[rank]);
        for (int j = 0; j < 64; j++)
            if (j != rank && ((row[j] >> col) & 1)) { row[j] ^= row[rank]; rhs[j] ^= rhs[rank]; }
        piv[col] = rank++;
    }
    for (int j = rank; j < 64; j++)
        if (rhs[j]) return false;
    u64 sol = 0;
    for (int col = 0; col < 64; col++)
        if (piv[col] >= 0 && rhs[piv[col]]) sol |= 1ULL << col;
    if (sol & 1) sol ^= 1;
    if ((gf64_mul_host(sol, sol) ^ sol) != c) return false;
    y = sol;
    return true;
}

struct BasisState {
    std::mutex mu;
    bool built = false;
    u64 b[64];
    int len = 0;
    int uploaded_dev = -1;
} g_basis;

void build_basis_host() {
    std::lock_guard<std::mutex> lk(g_basis.mu);
    if (g_basis.built) return;
    g_basis.b[0] = 1;
    g_basis.len = 1;
    while (g_basis.len < 64) {
        u64 y;
        if (!solve_T(g_basis.b[g_basis.len - 1], y)) break;
        g_basis.b[g_basis.len++] = y;
    }
    g_basis.built = true;
}

int ensure_basis() {
    build_basis_host();
    int dev = 0;
    GF2T_HIP(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lk(g_basis.mu);
    if (g_basis.uploaded_dev != dev) {
        static FftTables *tab = [] {
            FftTables *t = new FftTables;
            if (!cantor_host::build_tables(g_basis.b, *t)) {
                delete t;
                t = nullptr;
            }
            return t;
        }();
        if (!tab) {
            gf2t::set_error("fft: the Cantor basis does not give the subfield towers");
            return GF2T_EINTERNAL;
        }
        GF2T_HIP(hipMemcpyToSymbol(HIP_SYMBOL(g_tab), tab, sizeof(FftTables)));
        GF2T_HIP(hipMemcpyToSymbol(HIP_SYMBOL(c_tw), tab->tw, sizeof(tab->tw)));
        // the one kernel whose tile can pass 64 KiB of LDS (2^13 elements)
        for (const void *k : {(const void *)k_conv_tile64<false>, (const void *)k_conv_tile64<true>})
            GF2T_HIP(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, 72 * 1024));
        g_basis.uploaded_dev = dev;
    }
    return GF2T_OK;
}

}  // namespace

struct gf2t_fft_plan {
    int m, T;   // 2^m points, butterfly tiles of at most 2^T elements
};

namespace {
std::atomic<int> g_tile_bits[FFT_MAX_M + 1];   // 0: the default
std::atomic<int> g_fft_ept{2};
std::atomic<int> g_fft_low{FFT_LOW_BITS};

int tile_bits_for(int m) {
    int T = g_tile_bits[m].load(std::memory_order_relaxed);
    return T ? T : std::min(m < 6 ? 6 : m, FFT_TILE_BITS);
}
gf2t_fft_plan plan_for(int m) { return gf2t_fft_plan{m, tile_bits_for(m)}; }

// the conversion plans by size, built once
const cantor_host::ConvPlan &conv_plan32(int k) {
    static const std::vector<cantor_host::ConvPlan> v = [] {
        std::vector<cantor_host::ConvPlan> p;
        for (int j = 0; j <= FFT_MAX_M; j++)
            p.push_back(cantor_host::conv_plan(j, CONV_ONE_TILE, CONV_TILE32));
        return p;
    }();
    return v[k];
}
const cantor_host::ConvPlan &conv_plan64(int k) {
    static const std::vector<cantor_host::ConvPlan> v = [] {
        std::vector<cantor_host::ConvPlan> p;
        for (int j = 0; j <= FFT_MAX_M; j++)
            p.push_back(cantor_host::conv_plan(j, CONV_ONE_TILE, CONV_TILE64));
        return p;
    }();
    return v[k];
}
dim3 step_grid(const ConvStep &s, int k, unsigned nbatch, u32 &colblocks) {
    colblocks = (conv_full(s) + CONV_THREADS - 1) / CONV_THREADS;
    const u32 unit = 1u << s.ub;
    const u32 edges = unit < CONV_EDGE_RHO ? 1 : unit / CONV_EDGE_RHO;
    return dim3(colblocks + edges, 1u << (k - s.hb - s.K), nbatch);
}
size_t tile_lds(const ConvTile &t, size_t elem) {
    const size_t n = (size_t)1 << (t.c + t.w);
    return (n + n / 16) * elem;
}
dim3 tile_grid(const ConvTile &t, int k, unsigned nbatch) {
    const int T = t.c + t.w;
    return dim3(k > T ? 1u << (k - T) : 1u, nbatch);
}
dim3 tile_threads(const ConvTile &t) { return dim3(1u << (t.c + t.w - 4)); }

// basis conversion of nbatch operands of at most 2^k chunks, into their
// lch buffers; ran: whether anything was launched (k > 1)
int run_conv32(const Operands &ops, int k, unsigned nbatch, hipStream_t st, bool &ran) {
    const cantor_host::ConvPlan &P = conv_plan32(k);
    ran = !P.empty();
    int first = 1;
    for (const ConvStep &s : P.steps) {
        u32 cb;
        const dim3 g = step_grid(s, k, nbatch, cb);
        switch (s.K) {
        case 1: hipLaunchKernelGGL(k_conv_step32<1>, g, dim3(CONV_THREADS), 0, st, ops, s, cb, first); break;
        case 2: hipLaunchKernelGGL(k_conv_step32<2>, g, dim3(CONV_THREADS), 0, st, ops, s, cb, first); break;
        case 3: hipLaunchKernelGGL(k_conv_step32<3>, g, dim3(CONV_THREADS), 0, st, ops, s, cb, first); break;
        default: hipLaunchKernelGGL(k_conv_step32<4>, g, dim3(CONV_THREADS), 0, st, ops, s, cb, first); break;
        }
        first = 0;
    }
    for (const ConvTile &t : P.tiles) {
        hipLaunchKernelGGL(k_conv_tile32, tile_grid(t, k, nbatch), tile_threads(t), tile_lds(t, 4),
                           st, ops, t, first);
        first = 0;
    }
    GF2T_CHECK_LAUNCH("k_conv32");
    return GF2T_OK;
}
template <bool INV>
int run_conv64(u64 *f, u64 stride, int m, unsigned nbatch, hipStream_t st) {
    const cantor_host::ConvPlan &P = conv_plan64(m);
    auto step = [&](const ConvStep &s) {
        u32 cb;
        const dim3 g = step_grid(s, m, nbatch, cb);
        switch (s.K) {
        case 1: hipLaunchKernelGGL((k_conv_step64<1, INV>), g, dim3(CONV_THREADS), 0, st, f, stride, s, cb); break;
        case 2: hipLaunchKernelGGL((k_conv_step64<2, INV>), g, dim3(CONV_THREADS), 0, st, f, stride, s, cb); break;
        case 3: hipLaunchKernelGGL((k_conv_step64<3, INV>), g, dim3(CONV_THREADS), 0, st, f, stride, s, cb); break;
        default: hipLaunchKernelGGL((k_conv_step64<4, INV>), g, dim3(CONV_THREADS), 0, st, f, stride, s, cb); break;
        }
    };
    auto tile = [&](const ConvTile &t) {
        hipLaunchKernelGGL(k_conv_tile64<INV>, tile_grid(t, m, nbatch), tile_threads(t),
                           tile_lds(t, 8), st, f, stride, (u64)1 << m, t);
    };
    if (!INV) {
        for (const ConvStep &s : P.steps) step(s);
        for (const ConvTile &t : P.tiles) tile(t);
    } else {
        for (size_t i = P.tiles.size(); i--;) tile(P.tiles[i]);
        for (size_t i = P.steps.size(); i--;) step(P.steps[i]);
    }
    GF2T_CHECK_LAUNCH("k_conv64");
    return GF2T_OK;
}
constexpr u32 BF_BLOCKS = 2560;   // blocks of a butterfly launch: ten per CU
// butterfly passes above the low eight levels, all of nbatch transforms
// stride words apart
std::vector<BfPass> passes_for(const gf2t_fft_plan &pl, unsigned nbatch) {
    // tiles of at most 2^(T - 1) units (2^(8 + RB), as the eight levels of a
    // whole window always have), smaller until the launch fills the chip
    int tile = std::min(8 + RB, std::max(pl.T - 1, 6));
    while (tile > 6 + RB && ((((u64)1 << (pl.m - 1)) >> tile) * nbatch) < 1024) tile--;
    return cantor_host::bf_passes(pl.m, tile);
}
template <int CLS, bool INV>
void launch_bfly(u64 *f, u64 stride, const BfPass &P, const Operands &ops, int in, int out,
                 unsigned nbatch, hipStream_t st) {
    size_t lds = sizeof(MulLds) + (P.w > RB ? ((size_t)16 << P.tb) : 0);
    if (in == IO_PLAIN || out == IO_PLAIN) lds += 16384;
    else if (in != IO_UNITS) lds += 8192;
    const u32 tiles = 1u << (P.m - 1 - P.tb);
    hipLaunchKernelGGL((k_bfly<CLS, INV>), dim3(std::min(tiles, std::max(1u, BF_BLOCKS / nbatch)), nbatch),
                       dim3(1u << (P.tb - RB)), lds, st, f, stride, P, ops, in, out);
}
template <bool INV>
void run_bfly(u64 *f, u64 stride, const BfPass &P, const Operands &ops, int in, int out,
                 unsigned nbatch, hipStream_t st) {
    switch (cantor_host::bf_class(P)) {
    case 8: launch_bfly<8, INV>(f, stride, P, ops, in, out, nbatch, st); break;
    case 16: launch_bfly<16, INV>(f, stride, P, ops, in, out, nbatch, st); break;
    default: launch_bfly<32, INV>(f, stride, P, ops, in, out, nbatch, st); break;
    }
}
template <int DIR>
void run_low(u64 *f, u64 stride, const u64 *g, int m, const Operands &ops, u32 g_op, int in,
                int out, unsigned nbatch, hipStream_t st) {
    const u32 runs = std::max<u32>(1, (1u << (m - 1)) / LO_UNITS);
    const u32 pair = DIR == LO_MUL ? 2 : 1;
    // runs per block: more share the tables where the chip is full anyway
    const u64 waves = (u64)runs * nbatch * pair;
    const u32 rpb = waves >= 4096 ? 4 / pair : waves >= 1024 ? 2 / pair : 1;
    const u32 blocks = (runs + rpb - 1) / rpb, wpb = rpb * pair;
    size_t lds = sizeof(MulLds) + 4 * sizeof(TwEnt) + (DIR == LO_MUL ? sizeof(ProdLds) : 0) +
                 wpb * LO_EXCH * 4;
    if (in == IO_PLAIN || out == IO_PLAIN) lds += 16384;
    else if (in != IO_UNITS) lds += 8192;
    const dim3 gr(blocks, nbatch), th(64 * wpb);
    if (m <= 16)
        hipLaunchKernelGGL((k_low<16, 16, DIR>), gr, th, lds, st, f, stride, g, m, ops, g_op, in, out);
    else if (m <= 24 - RB)
        hipLaunchKernelGGL((k_low<16, 32, DIR>), gr, th, lds, st, f, stride, g, m, ops, g_op, in, out);
    else
        hipLaunchKernelGGL((k_low<32, 32, DIR>), gr, th, lds, st, f, stride, g, m, ops, g_op, in, out);
}
// Forward transforms of nbatch operands (at most 2^k chunks each) at f, f
// + stride, ... as units; low: the low levels too
int run_forward(const gf2t_fft_plan &pl, u64 *f, u64 stride, const Operands &ops, int k,
                unsigned nbatch, bool low, hipStream_t st, int &in) {
    bool ran;
    int rc = run_conv32(ops, k, nbatch, st, ran);
    if (rc) return rc;
    in = ran ? IO_LCH : IO_CHUNKS;
    for (const BfPass &P : passes_for(pl, nbatch)) {
        run_bfly<false>(f, stride, P, ops, in, IO_UNITS, nbatch, st);
        in = IO_UNITS;
    }
    if (low) {
        run_low<LO_FWD>(f, stride, nullptr, pl.m, ops, 0, in, IO_UNITS, nbatch, st);
        in = IO_UNITS;
    }
    GF2T_CHECK_LAUNCH("fft forward");
    return GF2T_OK;
}
// the rest of an inverse whose low levels are done (low: still to do), and
// the conversion back: coefficients in the polynomial basis
int run_inverse(const gf2t_fft_plan &pl, u64 *f, u64 stride, unsigned nbatch, bool low, int in,
                hipStream_t st) {
    const Operands none{};
    std::vector<BfPass> ps = passes_for(pl, nbatch);
    if (low) {
        run_low<LO_INV>(f, stride, nullptr, pl.m, none, 0, in, ps.empty() ? IO_PLAIN : IO_UNITS,
                        nbatch, st);
        in = IO_UNITS;
    }
    for (size_t i = ps.size(); i--;)
        run_bfly<true>(f, stride, ps[i], none, IO_UNITS, i ? IO_UNITS : IO_PLAIN, nbatch, st);
    GF2T_CHECK_LAUNCH("fft inverse");
    return run_conv64<true>(f, stride, pl.m, nbatch, st);
}
// Products of nbatch operand pairs (operands y and nbatch + y of ops, at
// most 2^k chunks): transforms at f + y stride and g + y stride, the
// product's coefficients modulo the vanishing polynomial of the 2^m
// points at f + y stride, in the polynomial basis.  g - f = nbatch stride.
// nbatch is at most MAX_PAIRS.
int run_product(const gf2t_fft_plan &pl, u64 *f, u64 stride, const Operands &ops, int k,
                unsigned nbatch, hipStream_t st) {
    int in;
    int rc = run_forward(pl, f, stride, ops, k, 2 * nbatch, false, st, in);
    if (rc) return rc;
    run_low<LO_MUL>(f, stride, f + (u64)nbatch * stride, pl.m, ops, nbatch, in,
                    pl.m <= 8 ? IO_PLAIN : IO_UNITS, nbatch, st);
    GF2T_CHECK_LAUNCH("k_low");
    return run_inverse(pl, f, stride, nbatch, false, IO_UNITS, st);
}

u32 last_mask(u64 bits) { return (bits & 31) ? (u32)((1ULL << (bits & 31)) - 1) : 0xFFFFFFFFu; }

// operand of `bits` bits, its converted chunks at lch
Operand operand_of(const u64 *src, u64 bits, void *lch, u32 xor0 = 0) {
    return Operand{(const u32 *)src, (u32 *)lch, (bits + 31) >> 5, last_mask(bits), xor0};
}
// the chunks [first, first + count) of operand o
Operand operand_range(Operand o, u64 first, u64 count) {
    if (first + count != o.n) o.mask = 0xFFFFFFFFu;
    if (first) o.xor0 = 0;
    o.src += first;
    o.n = count;
    return o;
}
int log2_ceil(u64 n) {
    int k = 0;
    while (((u64)1 << k) < n) k++;
    return k;
}
u64 round4(u64 n) { return (n + 3) & ~(u64)3; }

using cantor_host::fft_m_for;

}  // namespace

// gf2t_tune("fft_tile_<m>", T): tiles of at most 2^T elements (6..13) in the
// butterfly passes of fewer than eight levels of 2^m-point transforms from
// now on; 0 restores the default.
// Plans already made keep theirs.
int gf2t_fft_set_tile_bits(int m, int64_t T) {
    if (m < 1 || m > FFT_MAX_M || (T != 0 && (T < FFT_MIN_TILE_BITS || T > FFT_TILE_BITS))) {
        gf2t::set_error("gf2t_tune: fft_tile_<m> needs 1 <= m <= %d and T = 0 or %d..%d",
                        FFT_MAX_M, FFT_MIN_TILE_BITS, FFT_TILE_BITS);
        return GF2T_EINVAL;
    }
    g_tile_bits[m].store((int)T);
    return GF2T_OK;
}
int gf2t_fft_tile_bits(int m) { return (m >= 1 && m <= FFT_MAX_M) ? tile_bits_for(m) : 0; }
int gf2t_fft_set_ept(int64_t ept) {
    if (ept != 2 && ept != 4 && ept != 8 && ept != 16) {
        gf2t::set_error("gf2t_tune: fft_ept needs 2, 4, 8 or 16");
        return GF2T_EINVAL;
    }
    g_fft_ept.store((int)ept);
    return GF2T_OK;
}
int gf2t_fft_ept() { return g_fft_ept.load(); }
int gf2t_fft_set_low_bits(int64_t c) {
    if (c < 4 || c > 6) {
        gf2t::set_error("gf2t_tune: fft_low_bits needs 4, 5 or 6");
        return GF2T_EINVAL;
    }
    g_fft_low.store((int)c);
    return GF2T_OK;
}
int gf2t_fft_low_bits() { return g_fft_low.load(); }

extern "C" int gf2t_cantor_basis(uint64_t *hbasis, int *len) {
    build_basis_host();
    if (hbasis) std::memcpy(hbasis, g_basis.b, sizeof(g_basis.b));
    if (len) *len = g_basis.len;
    return GF2T_OK;
}

extern "C" int gf2t_fft_plan_create(int m, gf2t_fft_plan **plan) {
    if (!plan || m < 1 || m > FFT_MAX_M) {
        gf2t::set_error("gf2t_fft_plan_create: need 1 <= m <= %d", FFT_MAX_M);
        return GF2T_EINVAL;
    }
    build_basis_host();
    if (g_basis.len < m) {
        gf2t::set_error("gf2t_fft_plan_create: basis length %d < m", g_basis.len);
        return GF2T_EINTERNAL;
    }
    *plan = new gf2t_fft_plan(plan_for(m));
    return GF2T_OK;
}

extern "C" int gf2t_fft_plan_destroy(gf2t_fft_plan *plan) {
    delete plan;
    return GF2T_OK;
}

namespace {
template <bool INV>
int run_small(u64 *f, int m, hipStream_t st) {
    SmallFft A{};
    A.m = m;
    for (int k = 0; k < m - 1; k++) A.b[k] = g_basis.b[k + 1];
    if (m > 1) A.t = conv_plan64(m).tiles[0];
    hipLaunchKernelGGL(k_fft_small<INV>, dim3(1), dim3(m > 7 ? 1u << (m - 1) : 64u), 0, st, f, A);
    GF2T_CHECK_LAUNCH("k_fft_small");
    return GF2T_OK;
}
}  // namespace

extern "C" int gf2t_fft_plan_passes(const gf2t_fft_plan *plan, int *fwd_passes, int *inv_passes) {
    if (!plan) return GF2T_EINVAL;
    const size_t n = plan->m <= FFT_SMALL
                         ? 1 : conv_plan64(plan->m).launches() + passes_for(*plan, 1).size() + 1;
    if (fwd_passes) *fwd_passes = (int)n;
    if (inv_passes) *inv_passes = (int)n;
    return GF2T_OK;
}

extern "C" int gf2t_fft_fwd(const gf2t_fft_plan *plan, uint64_t *df, void *stream) {
    if (!plan || !df) return GF2T_EINVAL;
    int rc = ensure_basis();
    if (rc) return rc;
    hipStream_t st = (hipStream_t)stream;
    if (plan->m <= FFT_SMALL) return run_small<false>(df, plan->m, st);
    rc = run_conv64<false>(df, 0, plan->m, 1, st);
    if (rc) return rc;
    const Operands none{};
    int in = IO_PLAIN;
    for (const BfPass &P : passes_for(*plan, 1)) {
        run_bfly<false>(df, 0, P, none, in, IO_UNITS, 1, st);
        in = IO_UNITS;
    }
    run_low<LO_FWD>(df, 0, nullptr, plan->m, none, 0, in, IO_PLAIN, 1, st);
    GF2T_CHECK_LAUNCH("gf2t_fft_fwd");
    return GF2T_OK;
}

extern "C" int gf2t_fft_inv(const gf2t_fft_plan *plan, uint64_t *df, void *stream) {
    if (!plan || !df) return GF2T_EINVAL;
    int rc = ensure_basis();
    if (rc) return rc;
    if (plan->m <= FFT_SMALL) return run_small<true>(df, plan->m, (hipStream_t)stream);
    return run_inverse(*plan, df, 0, 1, true, IO_PLAIN, (hipStream_t)stream);
}

extern "C" size_t gf2t_mul_out_words(uint64_t abits, uint64_t bbits) {
    return words_of(abits + bbits) + 1;
}

namespace {
// Products of at most SC_WORK chunk pairs (and SC_OUTS outputs) are formed
// without a transform (k_school): 320,000 bits squared take 67 us so and
// 70 us by transforms, which at 360,000 are ahead, 71 to 78 us.
constexpr u64 SC_WORK = (u64)100 << 20, SC_OUTS = 65536;
constexpr u32 SC_FOLD_PARTS = 4;
// Chunk pairs of a slab of products of two parts up to which it takes no
// transforms either (4423 bits: 42 us against 51 for 512 residues, 72 against
// 60 for 1000; 8190 bits: 35 against 48 for 256, 59 against 52 for 512).
// Products of one part never take any (4090 bits: 15 against 34 us for one
// residue, 818 against 1000 for 32,767).
constexpr u64 SC_SLAB = 1 << 24;
bool school(u64 ca, u64 cb) { return ca && cb && ca + cb <= SC_OUTS && ca * cb <= SC_WORK; }
SchoolShape school_shape(u64 ca, u64 cb, bool split = true) {
    SchoolShape s;
    u64 na = std::min(ca, cb), nb = std::max(ca, cb);
    s.np = split && na >= SC_KARA ? 9 : 1;
    if (s.np == 9) {
        na = (na + 3) / 4;
        nb = (nb + 3) / 4;
    }
    s.na = (u32)na;
    s.nb = (u32)nb;
    s.nout = s.na + s.nb - 1;
    s.nparts = (s.na + SC_IN - 1) / SC_IN;
    return s;
}
// words of the parts, as a bound that grows with either operand also past
// the products that use it (a workspace for larger operands serves smaller
// ones): parts * outputs <= (na / SC_IN + 1)(na + nb), or a quarter of each
// nine times, with na nb <= SC_WORK
size_t school_words(u64 ca, u64 cb) {
    const u64 na = std::min(ca, cb), nb = std::max(ca, cb);
    const u64 most = 9 * ((2 * SC_WORK + 4 * SC_OUTS) / (4 * SC_IN) + SC_OUTS + 4) / 4;
    const u64 a = std::min<u64>(na, SC_OUTS), b = std::min<u64>(nb, SC_OUTS);
    const u64 one = std::min<u64>(a, SC_KARA - 1);
    u64 words = (one / SC_IN + 1) * (one + b);
    if (a >= SC_KARA) words = std::max(words, 9 * (a / (4 * SC_IN) + 1) * ((a + b) / 4 + 1));
    return (size_t)std::min(most, words);
}
int run_school(const Operands &ops, u32 b_op, bool swap, const SchoolShape &s, u64 *part,
               u64 part_stride, unsigned nbatch, hipStream_t st) {
    // part c reaches the outputs [SC_IN c, SC_IN (c + 1) + nb - 1): the tiles
    // from c on, as tiles and parts are of one length
    static_assert(SC_IN == SC_OUT, "tiles of a part");
    hipLaunchKernelGGL(s.np == 1 ? k_school<SC_SLACK> : k_school<SC_FULL>,
                       dim3((SC_IN - 1 + s.nb + SC_OUT - 1) / SC_OUT, s.nparts, nbatch * s.np),
                       dim3(256), 0, st, ops, b_op, swap ? 1 : 0, s, part, part_stride,
                       (const SchoolJob *)nullptr, (const SchoolBlock *)nullptr);
    GF2T_CHECK_LAUNCH("k_school");
    return GF2T_OK;
}
}  // namespace

extern "C" size_t gf2t_mul_workspace_bytes(uint64_t abits, uint64_t bbits) {
    u64 ca = (abits + 31) >> 5, cb = (bbits + 31) >> 5;
    if (!ca || !cb) return 0;
    int m = fft_m_for(ca + cb - 1);
    size_t n = (size_t)1 << m;
    return (std::max(2 * n, school_words(ca, cb)) + gf2t_mul_out_words(abits, bbits) + 8) *
           sizeof(u64);
}

namespace {
// p[0, n) = 0 with a kernel (no memset node when the caller captures a graph)
__global__ void k_zero_words(u64 *__restrict__ p, size_t n) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    size_t stride = (size_t)gridDim.x * blockDim.x;
    for (; i < n; i += stride) p[i] = 0;
}
int zero_words(u64 *p, size_t n, hipStream_t st) {
    hipLaunchKernelGGL(k_zero_words, dim3((unsigned)std::min<size_t>((n + 255) / 256, 4096)),
                       dim3(256), 0, st, p, n);
    GF2T_CHECK_LAUNCH("k_zero_words");
    return GF2T_OK;
}

// ---------------------------------------------------- wrapped products
// (see cantor_host::wrap_for)
using cantor_host::Wrap;
using cantor_host::wrap_for;
struct WrapArg {
    u64 n;          // 2^mp
    u64 e;          // top coefficients
    int noff;
    u32 off[15];    // 2^k for the proper bit-subsets k of mp
};
WrapArg wrap_arg(const Wrap &w) {
    WrapArg a{};
    a.n = (u64)1 << w.mp;
    a.e = w.e;
    for (int k = 0; k < w.mp; k++)
        if ((k & w.mp) == k) a.off[a.noff++] = 1u << k;
    return a;
}

// chunk coefficient k < n + e of the wrapped product: R = C mod V (2^mp
// coefficients), H = C_high; hit: the offsets to look at
GF2T_DEV u64 wrap_chunk(const u64 *__restrict__ R, const u64 *__restrict__ H, const WrapArg &w,
                        u32 hit, u64 k) {
    if (k >= w.n) return H[k - w.n];
    u64 v = R[k];
    for (u32 h = hit; h; h &= h - 1) {
        const u64 o = w.off[__builtin_ctz(h)];
        if (k >= o && k - o < w.e) v ^= H[k - o];
    }
    return v;
}

// overlap-add of a wrapped product (gather form, as k_overlap_add);
// blockIdx.y selects a batch element: R + y*r_stride, H + y*h_stride,
// out + y*o_stride
__global__ void k_overlap_add_wrap(const u64 *__restrict__ R, u64 r_stride,
                                   const u64 *__restrict__ H, u64 h_stride, const WrapArg w,
                                   size_t nchunks, u64 *__restrict__ out, size_t owords,
                                   u64 o_stride) {
    const size_t w0 = (size_t)blockIdx.x * blockDim.x, wd = w0 + threadIdx.x;
    // the offsets whose copy of C_high reaches the block's coefficients
    // (most blocks: none)
    const u64 k0 = w0 ? 2 * (u64)w0 - 1 : 0, k1 = 2 * (u64)(w0 + blockDim.x);
    u32 hit = 0;
    for (int j = 0; j < w.noff; j++)
        if (k1 > w.off[j] && k0 < w.off[j] + w.e) hit |= 1u << j;
    if (wd >= owords) return;
    R += (u64)blockIdx.y * r_stride;
    H += (u64)blockIdx.y * h_stride;
    out += (u64)blockIdx.y * o_stride;
    size_t k = 2 * wd;
    u64 v = 0;
    if (k < nchunks) v ^= wrap_chunk(R, H, w, hit, k);
    if (k + 1 < nchunks) v ^= wrap_chunk(R, H, w, hit, k + 1) << 32;
    if (wd && k - 1 < nchunks) v ^= wrap_chunk(R, H, w, hit, k - 1) >> 32;
    out[wd] = v;
}

int mul_core(const u64 *da, u64 abits, const u64 *db, u64 bbits, u64 *dprod, void *dwork,
             hipStream_t st) {
    u64 ca = (abits + 31) >> 5, cb = (bbits + 31) >> 5;
    size_t ow = gf2t_mul_out_words(abits, bbits);
    if (!ca || !cb) return zero_words(dprod, ow, st);
    int m = fft_m_for(ca + cb - 1);
    if (m > FFT_MAX_M) {
        gf2t::set_error("gf2t_mul: product needs 2^%d points (max 2^%d)", m, FFT_MAX_M);
        return GF2T_ERANGE;
    }
    int rc = ensure_basis();
    if (rc) return rc;
    if (school(ca, cb)) {
        Operands two{};
        two.op[0] = operand_of(da, abits, nullptr);
        two.op[1] = operand_of(db, bbits, nullptr);
        const SchoolShape s = school_shape(ca, cb);
        rc = run_school(two, 1, ca > cb, s, (u64 *)dwork, 0, 1, st);
        if (rc) return rc;
        hipLaunchKernelGGL(s.np == 1 ? k_school_product : k_school_kara,
                           dim3((unsigned)((ow + SP_WORDS - 1) / SP_WORDS)), dim3(256), 0, st,
                           (const u64 *)dwork, s, dprod, ow);
        GF2T_CHECK_LAUNCH("k_school_product");
        return GF2T_OK;
    }
    // the converted chunks of both operands, behind the two transforms
    // (where the product goes later, or the workspace's tail)
    const size_t n = (size_t)1 << m;
    u64 *FA = (u64 *)dwork;
    u32 *lch = (u32 *)(FA + 2 * n);
    Operands two{};
    two.op[0] = operand_of(da, abits, lch);
    two.op[1] = operand_of(db, bbits, lch + round4(ca));
    const int k = log2_ceil(std::max(ca, cb));
    const Wrap W = wrap_for(ca, cb);
    if (W.on) {
        // both operands at 2^mp points, their top e chunks at 2^ms points
        // (2^mp + 2^ms <= 2^m words each, inside the workspace of an
        // unwrapped product)
        const size_t np = (size_t)1 << W.mp, ns = (size_t)1 << W.ms;
        u64 *TA = FA + 2 * np;
        Operands top{};
        top.op[0] = operand_range(two.op[0], ca - W.e, W.e);
        top.op[1] = operand_range(two.op[1], cb - W.e, W.e);
        rc = run_product(plan_for(W.mp), FA, np, two, k, 1, st);
        if (rc) return rc;
        rc = run_product(plan_for(W.ms), TA, ns, top, log2_ceil(W.e), 1, st);
        if (rc) return rc;
        // C_high[u] = coefficient e - 1 + u of the top product
        hipLaunchKernelGGL(k_overlap_add_wrap, dim3((unsigned)((ow + 255) / 256)), dim3(256), 0,
                           st, FA, (u64)0, TA + (W.e - 1), (u64)0, wrap_arg(W),
                           (size_t)(ca + cb - 1), dprod, ow, (u64)0);
        GF2T_CHECK_LAUNCH("k_overlap_add_wrap");
        return GF2T_OK;
    }
    rc = run_product(plan_for(m), FA, n, two, k, 1, st);
    if (rc) return rc;
    hipLaunchKernelGGL(k_overlap_add, dim3((unsigned)((ow + 255) / 256)), dim3(256), 0, st, FA,
                       (size_t)(ca + cb - 1), dprod, ow, (u64)0, (u64)0);
    GF2T_CHECK_LAUNCH("k_overlap_add");
    return GF2T_OK;
}
}  // namespace

extern "C" int gf2t_mul(const uint64_t *da, uint64_t abits, const uint64_t *db, uint64_t bbits,
                        uint64_t *dout, void *dwork, void *stream) {
    if (!da || !db || !dout || (!dwork && abits && bbits)) {
        gf2t::set_error("gf2t_mul: null pointer");
        return GF2T_EINVAL;
    }
    return mul_core(da, abits, db, bbits, dout, dwork, (hipStream_t)stream);
}

extern "C" int gf2t_fold(const uint64_t *dsrc, uint64_t src_bits, uint64_t *dout, uint64_t r,
                         uint64_t s, void *stream);

namespace {
// the product in the workspace behind what mul_core uses of it, then its
// fold; both operands have chunks
int mulmod_core(const u64 *da, u64 abits, const u64 *db, u64 bbits, u64 r, u64 s, u64 *dout,
                u64 *dwork, hipStream_t st) {
    const u64 ca = (abits + 31) >> 5, cb = (bbits + 31) >> 5;
    if (school(ca, cb)) {
        const SchoolShape sh = school_shape(ca, cb);
        if (sh.np == 1 && sh.nparts <= SC_FOLD_PARTS) {   // few parts to add up: folded from them directly
            if (r >= (1ULL << 34)) {   // what gf2t_fold, passed by here, takes
                gf2t::set_error("gf2t_mulmod: need r < 2^34");
                return GF2T_EINVAL;
            }
            Operands two{};
            two.op[0] = operand_of(da, abits, nullptr);
            two.op[1] = operand_of(db, bbits, nullptr);
            int rc = run_school(two, 1, ca > cb, sh, dwork, 0, 1, st);
            if (rc) return rc;
            const size_t nw = words_of(r);
            hipLaunchKernelGGL(k_school_fold, dim3((unsigned)((nw + 255) / 256)), dim3(256), 0, st,
                               (const u64 *)dwork, (u64)0, sh, abits + bbits - 1, dout, nw,
                               (u64)0, r, s, (const u64 *)nullptr);
            GF2T_CHECK_LAUNCH("k_school_fold");
            return GF2T_OK;
        }
    }
    u64 *prod = dwork + std::max((size_t)2 << fft_m_for(ca + cb - 1), school_words(ca, cb));
    int rc = mul_core(da, abits, db, bbits, prod, dwork, st);
    if (rc) return rc;
    return gf2t_fold(prod, abits + bbits - 1, dout, r, s, st);
}
}  // namespace

extern "C" int gf2t_mulmod(const uint64_t *da, uint64_t abits, const uint64_t *db,
                           uint64_t bbits, uint64_t r, uint64_t s, uint64_t *dout, void *dwork,
                           void *stream) {
    if (!da || !db || !dout || !dwork) {
        gf2t::set_error("gf2t_mulmod: null pointer");
        return GF2T_EINVAL;
    }
    if (abits + bbits > 2 * r) {
        gf2t::set_error("gf2t_mulmod: product of %llu+%llu bits exceeds 2r-1",
                        (unsigned long long)abits, (unsigned long long)bbits);
        return GF2T_EINVAL;
    }
    if (!(r >= 3 && s >= 1 && 2 * s < r)) {
        gf2t::set_error("gf2t_mulmod: need 1 <= s, 2s < r");
        return GF2T_EINVAL;
    }
    u64 ca = (abits + 31) >> 5, cb = (bbits + 31) >> 5;
    if (!ca || !cb)   // a zero operand: the workspace may be empty, dout is 0
        return zero_words(dout, words_of(r), (hipStream_t)stream);
    return mulmod_core(da, abits, db, bbits, r, s, dout, (u64 *)dwork, (hipStream_t)stream);
}

// ------------------------------------------------ modmul without allocation
// gf2t_mulmod_noalloc: gf2t_mulmod with its workspace in a library-owned
// device array instead of a caller's buffer, for callers that cannot
// allocate.  The array holds the two 2^22-point transforms and the
// product (up to 2^27 bits): 80 MiB, which every GPU the library runs on
// keeps until the process ends.  The pack pass writes every transform
// element and the overlap-add every product word, so nothing in it needs
// clearing between calls.  Calls that overlap on one GPU share the array
// and race.
namespace {
constexpr int NA_MAX_M = 22;
constexpr size_t NA_FFT_WORDS = (size_t)1 << NA_MAX_M;
constexpr size_t NA_PROD_WORDS = ((size_t)1 << 21) + 2;   // gf2t_mul_out_words(a, b), a+b <= 2^27+64
constexpr size_t NA_WORDS = 2 * NA_FFT_WORDS + NA_PROD_WORDS + 30;
constexpr int NA_MAX_DEVICES = 64;
}  // namespace

static __device__ __align__(256) u64 scratch[NA_WORDS];

namespace {
std::mutex g_scratch_mu;
// device address of `scratch` on each device, from hipGetSymbolAddress
// (the name itself is only a host-side stand-in)
u64 *g_scratch_ptr[NA_MAX_DEVICES] = {};

}  // namespace

// Once per device, with that device current (gf2t_init calls it; the
// entry point calls it on its first use on a device otherwise): record
// the scratch array's device address, upload the Cantor basis and build
// the transform plans the entry point can need, so that its calls
// allocate nothing.
int gf2t_noalloc_setup() {
    int dev = 0;
    GF2T_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= NA_MAX_DEVICES) {
        gf2t::set_error("gf2t_noalloc_setup: device %d beyond %d", dev, NA_MAX_DEVICES);
        return GF2T_ERANGE;
    }
    {
        std::lock_guard<std::mutex> lk(g_scratch_mu);
        if (!g_scratch_ptr[dev]) {
            void *p = nullptr;
            GF2T_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
            g_scratch_ptr[dev] = (u64 *)p;
        }
    }
    conv_plan32(0);
    conv_plan64(0);
    return ensure_basis();
}

extern "C" int gf2t_mulmod_noalloc(const uint64_t *da, uint64_t abits, const uint64_t *db,
                                   uint64_t bbits, uint64_t r, uint64_t s, uint64_t *dout,
                                   void *stream) {
    if (!da || !db || !dout) {
        gf2t::set_error("gf2t_mulmod_noalloc: null pointer");
        return GF2T_EINVAL;
    }
    if (!(r >= 3 && s >= 1 && 2 * s < r) || abits + bbits > 2 * r) {
        gf2t::set_error("gf2t_mulmod_noalloc: need 1 <= s, 2s < r and a product of at most "
                        "2r-1 bits (r=%llu s=%llu, %llu+%llu bits)", (unsigned long long)r,
                        (unsigned long long)s, (unsigned long long)abits,
                        (unsigned long long)bbits);
        return GF2T_EINVAL;
    }
    const u64 ca = (abits + 31) >> 5, cb = (bbits + 31) >> 5;
    if (ca && cb && ca + cb - 1 > NA_FFT_WORDS) {
        gf2t::set_error("gf2t_mulmod_noalloc: a %llu x %llu-bit product needs more than the "
                        "2^%d transform points its scratch holds (at most %llu 32-bit chunks "
                        "in both operands together); use gf2t_mulmod with a workspace",
                        (unsigned long long)abits, (unsigned long long)bbits, NA_MAX_M,
                        (unsigned long long)(NA_FFT_WORDS + 1));
        return GF2T_ERANGE;
    }
    int dev = 0;
    GF2T_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= NA_MAX_DEVICES) {
        gf2t::set_error("gf2t_mulmod_noalloc: device %d beyond %d", dev, NA_MAX_DEVICES);
        return GF2T_ERANGE;
    }
    u64 *ptr;
    {
        std::lock_guard<std::mutex> lk(g_scratch_mu);
        ptr = g_scratch_ptr[dev];
    }
    if (!ptr) {
        int rc = gf2t_noalloc_setup();
        if (rc) return rc;
        std::lock_guard<std::mutex> lk(g_scratch_mu);
        ptr = g_scratch_ptr[dev];
    }
    hipStream_t st = (hipStream_t)stream;
    if (!ca || !cb) return zero_words(dout, words_of(r), st);   // a zero operand
    return mulmod_core(da, abits, db, bbits, r, s, dout, ptr, st);
}

// ------------------------------------------------- variable-size batch
// gf2t_mulmod_batch: products of different sizes, each folded mod
// x^r + x^s_j + 1.  The smaller sizes are formed without transforms, all in
// one launch; of the others the pairs of one size share a chain of launches;
// the overlap-adds and folds of all pairs are one launch each.
namespace {
struct PairSeg {       // one pair's part of a flat grouped launch over elements
    const u64 *fa;
    u64 *prod;
    u64 *out;
    u64 nch, ow, pw, L, s, start;   // start: the pair's first element in the launch
};

GF2T_DEV int find_seg(const PairSeg *__restrict__ sg, int np, u64 i) {
    int lo = 0, hi = np - 1;
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (sg[mid].start <= i) lo = mid; else hi = mid - 1;
    }
    return lo;
}

// phase 0: overlap-add FA into prod; 1: fold prod into out.  total = sum
// of the pairs' element counts for the phase.  A block takes `run`
// consecutive elements and finds the first one's pair once; the pairs after
// it are few (a search per element took two thirds of the time).  Runs of up
// to 2048 elements, shorter where that fills the chip: 200 pairs of 18 words
// were two blocks that took their 114 pairs one after another, 529 us in all.
u32 pairs_run(u64 total) { return (u32)std::max<u64>(8, std::min<u64>(2048, total / 1024)); }
__global__ __launch_bounds__(256) void k_pairs_grouped(const PairSeg *__restrict__ sg, int np,
                                                       u64 total, u32 run, int phase, u64 r) {
    const u64 i0 = (u64)blockIdx.x * run, i1 = i0 + run < total ? i0 + run : total;
    for (int p = find_seg(sg, np, i0); p < np && sg[p].start < i1; p++) {
        const PairSeg S = sg[p];
        const u64 end = p + 1 < np && sg[p + 1].start < i1 ? sg[p + 1].start : i1;
        for (u64 i = (S.start > i0 ? S.start : i0) + threadIdx.x; i < end; i += 256) {
            const u64 k = i - S.start;
            if (phase == 0) {
                const u64 c = 2 * k;
                u64 v = 0;
                if (c < S.nch) v ^= S.fa[c];
                if (c + 1 < S.nch) v ^= S.fa[c + 1] << 32;
                if (k && c - 1 < S.nch) v ^= S.fa[c - 1] >> 32;
                S.prod[k] = v;
            } else {
                S.out[k] = fold_word(S.prod, S.pw, S.L, r, S.s, k);
            }
        }
    }
}

// Pairs of one transform size run as one chain of launches, their A
// transforms side by side and the B transforms behind them.
struct BatchLayout {
    std::vector<cantor_host::SizeGroup> groups;
    std::vector<size_t> fa, prod;   // word offsets of each pair's A transform (or parts) and product
    std::vector<int> m;
    std::vector<char> school;
    size_t desc_off = 0, words = 0;
};

// The words grow with each pair's operands, and with the number of pairs:
// every pair has its transforms' space, whatever its route, and the parts of
// those that take none lie in theirs together and 2 / SC_IN words more for
// each chunk pair: parts * outputs <= (ca / SC_IN + 1)(ca + cb) for ca <= cb.
BatchLayout batch_layout(int n, const uint64_t *abits, const uint64_t *bbits) {
    BatchLayout L;
    L.fa.resize(n);
    std::vector<u64> ca(n), cb(n);
    for (int j = 0; j < n; j++) {
        ca[j] = (abits[j] + 31) >> 5;
        cb[j] = (bbits[j] + 31) >> 5;
        L.m.push_back((ca[j] && cb[j]) ? fft_m_for(ca[j] + cb[j] - 1) : 0);
    }
    L.school = cantor_host::direct_pairs(L.m, ca, cb);
    std::vector<int> m = L.m;
    size_t off = 0, space = 0, blocks = 0, direct = 0;
    for (int j = 0; j < n; j++) {
        if (!m[j]) continue;
        space += (size_t)2 << m[j];
        direct = std::min(cantor_host::DIRECT_PAIRS,
                          direct + std::min<size_t>(cantor_host::DIRECT_PAIRS, ca[j] * cb[j]));
        blocks += 3 * (ca[j] + cb[j]) / SC_IN + 4 + (ca[j] + cb[j]) / (2 * SP_WORDS) + 2;
        if (L.school[j]) m[j] = 0;
    }
    L.groups = cantor_host::size_groups(m);
    for (const cantor_host::SizeGroup &g : L.groups) {
        for (size_t i = 0; i < g.pairs.size(); i++) L.fa[g.pairs[i]] = off + (i << g.m);
        off += 2 * g.pairs.size() << g.m;
    }
    for (int j = 0; j < n; j++) {
        if (!L.school[j]) continue;
        const SchoolShape s = school_shape(ca[j], cb[j], false);
        L.fa[j] = off;
        off += (size_t)s.nparts * s.nout;
    }
    off = (space + 2 * direct / SC_IN + 31) & ~(size_t)31;
    for (int j = 0; j < n; j++) {
        L.prod.push_back(off);
        // the product, and before it both operands' converted chunks
        off += (gf2t_mul_out_words(abits[j], bbits[j]) + 4 + 31) & ~(size_t)31;
    }
    L.desc_off = off;
    blocks += direct / (SC_IN * SC_IN);
    const size_t desc = (size_t)n * 2 * (sizeof(Operand) + sizeof(PairSeg)) +
                        (size_t)n * sizeof(SchoolJob) + blocks * sizeof(SchoolBlock) + 256;
    L.words = off + (desc + 7) / 8 + 32;
    return L;
}
}  // namespace

extern "C" size_t gf2t_mulmod_batch_workspace_bytes(int n, const uint64_t *abits,
                                                   const uint64_t *bbits) {
    if (n <= 0 || !abits || !bbits) return 0;
    return batch_layout(n, abits, bbits).words * 8;
}

extern "C" int gf2t_mulmod_batch(int n, const uint64_t *const *da, const uint64_t *abits,
                                 const uint64_t *const *db, const uint64_t *bbits, uint64_t r,
                                 const uint64_t *s, uint64_t *const *dout, void *dwork,
                                 void *stream) {
    if (n < 0 || (n > 0 && (!da || !abits || !db || !bbits || !s || !dout || !dwork))) {
        gf2t::set_error("gf2t_mulmod_batch: bad arguments");
        return GF2T_EINVAL;
    }
    if (n == 0) return GF2T_OK;
    for (int j = 0; j < n; j++) {
        if (!da[j] || !db[j] || !dout[j] || !(r >= 3 && s[j] >= 1 && 2 * s[j] < r) ||
            abits[j] + bbits[j] > 2 * r) {
            gf2t::set_error("gf2t_mulmod_batch: pair %d: bad pointers, s, or a product over "
                            "2r-1 bits", j);
            return GF2T_EINVAL;
        }
        u64 ca = (abits[j] + 31) >> 5, cb = (bbits[j] + 31) >> 5;
        if (ca && cb && fft_m_for(ca + cb - 1) > FFT_MAX_M) {
            gf2t::set_error("gf2t_mulmod_batch: pair %d needs more than 2^%d points", j,
                            FFT_MAX_M);
            return GF2T_ERANGE;
        }
    }
    int rc = ensure_basis();
    if (rc) return rc;
    hipStream_t st = (hipStream_t)stream;
    const BatchLayout L = batch_layout(n, abits, bbits);
    u64 *W = (u64 *)dwork;
    // products without a transform, and the operands of the others, group
    // by group: the A's, then the B's
    std::vector<SchoolJob> jobs;
    std::vector<SchoolBlock> blocks;
    for (int j = 0; j < n; j++) {
        if (!L.school[j]) continue;
        const u64 ca = (abits[j] + 31) >> 5, cb = (bbits[j] + 31) >> 5;
        SchoolJob q{operand_of(da[j], abits[j], nullptr), operand_of(db[j], bbits[j], nullptr),
                    school_shape(ca, cb, false), W + L.fa[j], W + L.prod[j],
                    gf2t_mul_out_words(abits[j], bbits[j])};
        if (ca > cb) std::swap(q.a, q.b);
        for (u32 t = 0; t * SC_OUT < q.s.nout; t++)
            for (u32 c = school_first(q.s, t); c <= school_last(q.s, t); c++)
                blocks.push_back(SchoolBlock{(u32)jobs.size(), (unsigned short)t, (unsigned short)c});
        jobs.push_back(q);
    }
    const size_t nblocks = blocks.size();   // and then those of the products
    for (u32 j = 0; j < jobs.size(); j++)
        for (u32 t = 0; t * SP_WORDS < jobs[j].owords; t++)
            blocks.push_back(SchoolBlock{j, (unsigned short)t, 0});
    std::vector<Operand> opv;
    for (const cantor_host::SizeGroup &g : L.groups)
        for (int o = 0; o < 2; o++)
            for (int j : g.pairs) {
                u32 *lch = (u32 *)(W + L.prod[j]);
                opv.push_back(o ? operand_of(db[j], bbits[j],
                                             lch + round4((abits[j] + 31) >> 5))
                                : operand_of(da[j], abits[j], lch));
            }
    std::vector<PairSeg> seg[2];
    u64 total[2] = {0, 0};
    int nz = 0;
    for (int j = 0; j < n; j++) {
        const size_t nw = words_of(r);
        if (!L.m[j]) {   // a zero operand: the residue is 0
            rc = zero_words(dout[j], nw, st);
            if (rc) return rc;
            nz++;
            continue;
        }
        const u64 ca = (abits[j] + 31) >> 5, cb = (bbits[j] + 31) >> 5;
        const u64 ow = gf2t_mul_out_words(abits[j], bbits[j]);
        PairSeg p{};
        p.fa = W + L.fa[j];
        p.prod = W + L.prod[j];
        p.out = dout[j];
        p.nch = ca + cb - 1;
        p.ow = ow;
        p.pw = ow;
        p.L = abits[j] + bbits[j] - 1;
        p.s = s[j];
        const u64 cnt[2] = {ow, (u64)nw};
        for (int ph = L.school[j] ? 1 : 0; ph < 2; ph++) {
            p.start = total[ph];
            total[ph] += cnt[ph];
            seg[ph].push_back(p);
        }
    }
    if (nz == n) return GF2T_OK;
    // descriptors: the jobs and their blocks, the operands, then the two
    // segment tables
    std::vector<unsigned char> host;
    auto put = [&](const void *v, size_t bytes) {
        const size_t at = host.size();
        host.resize(at + bytes);
        if (bytes) std::memcpy(host.data() + at, v, bytes);
        return at;
    };
    const size_t oj = put(jobs.data(), jobs.size() * sizeof(SchoolJob));
    const size_t ok = put(blocks.data(), blocks.size() * sizeof(SchoolBlock));
    const size_t oo = put(opv.data(), opv.size() * sizeof(Operand));
    const size_t os[2] = {put(seg[0].data(), seg[0].size() * sizeof(PairSeg)),
                          put(seg[1].data(), seg[1].size() * sizeof(PairSeg))};
    unsigned char *dd = (unsigned char *)(W + L.desc_off);
    dd = (unsigned char *)(((uintptr_t)dd + 255) & ~(uintptr_t)255);
    GF2T_HIP(hipMemcpyAsync(dd, host.data(), host.size(), hipMemcpyHostToDevice, st));
    GF2T_HIP(hipStreamSynchronize(st));   // `host` is a pageable local buffer
    const Operand *dop = (const Operand *)(dd + oo);
    if (!blocks.empty()) {
        const SchoolJob *dj = (const SchoolJob *)(dd + oj);
        const SchoolBlock *db = (const SchoolBlock *)(dd + ok);
        hipLaunchKernelGGL(k_school<SC_JOBS>, dim3((unsigned)nblocks), dim3(256), 0, st, Operands{},
                           0u, 0, SchoolShape{}, (u64 *)nullptr, (u64)0, dj, db);
        hipLaunchKernelGGL(k_school_products, dim3((unsigned)(blocks.size() - nblocks)), dim3(256), 0,
                           st, dj, db + nblocks);
        GF2T_CHECK_LAUNCH("k_school_products");
    }
    size_t first = 0;
    for (const cantor_host::SizeGroup &g : L.groups) {
        const unsigned cnt = (unsigned)g.pairs.size();
        u64 most = 1;
        for (int j : g.pairs)
            most = std::max(most, std::max((abits[j] + 31) >> 5, (bbits[j] + 31) >> 5));
        Operands ops{};
        ops.list = dop + first;
        rc = run_product(plan_for(g.m), W + L.fa[g.pairs[0]], (u64)1 << g.m, ops, log2_ceil(most), cnt, st);
        if (rc) return rc;
        first += 2 * cnt;
    }
    for (int ph = 0; ph < 2; ph++) {
        if (!total[ph]) continue;
        const u32 run = pairs_run(total[ph]);
        hipLaunchKernelGGL(k_pairs_grouped, dim3((unsigned)((total[ph] + run - 1) / run)), dim3(256),
                           0, st, (const PairSeg *)(dd + os[ph]), (int)seg[ph].size(), total[ph], run,
                           ph, (u64)r);
    }
    GF2T_CHECK_LAUNCH("gf2t_mulmod_batch");
    return GF2T_OK;
}

// ------------------------------------------------------------------ slabs
namespace {
__global__ void k_fold_slab(const u64 *__restrict__ p, size_t pw, u64 p_stride, u64 L,
                            u64 *__restrict__ out, u64 o_stride, size_t nw, u64 r,
                            const u64 *__restrict__ svec) {
    size_t w = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (w >= nw) return;
    const u64 s = svec[blockIdx.y];
    p += (u64)blockIdx.y * p_stride;
    out += (u64)blockIdx.y * o_stride;
    out[w] = fold_word(p, pw, L, r, s, w);
}
}  // namespace

extern "C" size_t gf2t_mulmod_slab_workspace_bytes(uint64_t r, int n) {
    u64 ca = (r + 31) >> 5;
    int m = fft_m_for(2 * ca - 1);
    size_t per = 2 * ((size_t)1 << m) + 2 * words_of(r) + 2;
    return per * (size_t)(n > 0 ? n : 0) * sizeof(u64);
}

extern "C" int gf2t_mulmod_slab(const uint64_t *da, size_t apitch, const uint64_t *db,
                                size_t bpitch, int b_add_x, uint64_t r, const uint64_t *ds,
                                uint64_t *dout, size_t opitch, int n, void *dwork, void *stream) {
    if (!da || !db || !dout || !ds || !dwork || n < 0 || r < 3) {
        gf2t::set_error("gf2t_mulmod_slab: bad arguments");
        return GF2T_EINVAL;
    }
    if (n == 0) return GF2T_OK;
    size_t nw = words_of(r);
    if (apitch < nw || bpitch < nw || opitch < nw || n > 65535) {
        gf2t::set_error("gf2t_mulmod_slab: pitch below nw or more than 65535 residues");
        return GF2T_EINVAL;
    }
    hipStream_t st = (hipStream_t)stream;
    int rc = ensure_basis();
    if (rc) return rc;
    u64 ca = (r + 31) >> 5;
    int m = fft_m_for(2 * ca - 1);
    if (m > FFT_MAX_M) { gf2t::set_error("gf2t_mulmod_slab: r too large"); return GF2T_ERANGE; }
    const size_t N = (size_t)1 << m;
    u64 *FA = (u64 *)dwork, *prod = FA + 2 * N * n;
    const size_t ppitch = 2 * nw + 2;
    // operands y < n: the a's, then the b's; their converted chunks where
    // the products go later (2 ca chunks in the 4 nw + 4 of a residue)
    Operands ops{};
    ops.group = (u32)n;
    ops.lstride = 2 * ppitch;
    ops.sstride[0] = 2 * apitch;
    ops.sstride[1] = 2 * bpitch;
    ops.op[0] = operand_of(da, r, prod);
    ops.op[1] = operand_of(db, r, (u32 *)prod + 2 * nw + 2, b_add_x ? 2u : 0u);
    const u64 ow = 2 * nw;   // product of two r-bit operands: 2r-1 bits
    const SchoolShape sh = school_shape(ca, ca);
    if (sh.np == 1 && (sh.nparts == 1 || (sh.nparts == 2 && n * ca * ca <= SC_SLAB))) {   // the parts fit the transforms' space
        rc = run_school(ops, (u32)n, false, sh, FA, 2 * N, (unsigned)n, st);
        if (rc) return rc;
        hipLaunchKernelGGL(k_school_fold, dim3((unsigned)((nw + 255) / 256), n), dim3(256), 0, st,
                           FA, (u64)(2 * N), sh, 2 * r - 1, dout, nw, (u64)opitch, r, (u64)0, ds);
        GF2T_CHECK_LAUNCH("k_school_fold");
        return GF2T_OK;
    }
    const int k = log2_ceil(ca);
    const Wrap W = wrap_for(ca, ca, (u64)n);
    // MAX_PAIRS residues at a time, through the same transforms' space
    for (unsigned i0 = 0; i0 < (unsigned)n; i0 += cantor_host::MAX_PAIRS) {
        const unsigned cnt = std::min((unsigned)n - i0, cantor_host::MAX_PAIRS);
        Operands part = ops;
        part.group = cnt;
        for (int g = 0; g < 2; g++) {
            part.op[g].src += i0 * ops.sstride[g];
            part.op[g].lch += i0 * ops.lstride;
        }
        u64 *pr = prod + i0 * ppitch;
        if (W.on) {
            // the wrapped product (see wrap_for): 2^mp-point transforms of
            // both operands and 2^ms-point transforms of their top e chunks,
            // laid out inside the 2 N words a residue of an unwrapped product
            // uses
            const size_t np = (size_t)1 << W.mp, ns = (size_t)1 << W.ms;
            u64 *TA = FA + 2 * np * cnt;
            rc = run_product(plan_for(W.mp), FA, np, part, k, cnt, st);
            if (rc) return rc;
            // top chunks [ca - e, ca); chunk 0 (where b_add_x adds x) is not among them
            Operands top = part;
            for (int g = 0; g < 2; g++) top.op[g] = operand_range(part.op[g], ca - W.e, W.e);
            rc = run_product(plan_for(W.ms), TA, ns, top, log2_ceil(W.e), cnt, st);
            if (rc) return rc;
            hipLaunchKernelGGL(k_overlap_add_wrap, dim3((unsigned)((ow + 255) / 256), cnt),
                               dim3(256), 0, st, FA, (u64)np, TA + (W.e - 1), (u64)ns, wrap_arg(W),
                               (size_t)(2 * ca - 1), pr, (size_t)ow, (u64)ppitch);
        } else {
            rc = run_product(plan_for(m), FA, N, part, k, cnt, st);
            if (rc) return rc;
            hipLaunchKernelGGL(k_overlap_add, dim3((unsigned)((ow + 255) / 256), cnt), dim3(256), 0,
                               st, FA, (size_t)(2 * ca - 1), pr, (size_t)ow, (u64)N, (u64)ppitch);
        }
    }
    hipLaunchKernelGGL(k_fold_slab, dim3((unsigned)((nw + 255) / 256), n), dim3(256), 0, st, prod,
                       (size_t)ow, (u64)ppitch, 2 * r - 1, dout, (u64)opitch, nw, r, ds);
    GF2T_CHECK_LAUNCH("gf2t_mulmod_slab");
    return GF2T_OK;
}

// --------------------------------------------- host-buffer product service
// The device side of the reference's GpuMulHook (TsGpuMul, src/tsfactor.cu:
// 467-607; interface src/gf2_gcd.h:155-172): host vectors in and out, one
// mutex-guarded context per process with a private stream and device
// buffers grown on demand (never shrunk).
namespace {

// A pool of contexts, each with its own non-blocking stream, device
// buffer and pinned host staging buffer, so products requested by
// different host threads (the gcds of different s values) run
// concurrently on the device.  Operands are copied into the pinned
// buffer and go to the device in one transfer; results come back the
// same way.
constexpr int HM_CONTEXTS = 16;
// products whose operands and results together take at most this many
// words go through pinned host memory directly (gf2t_tune "hm_zc_words")
std::atomic<long long> g_hm_zc_words{65536};
struct HostMulCtx {
    hipStream_t st = nullptr;
    u64 *dbuf = nullptr;
    size_t dcap = 0;   // words
    u64 *hbuf = nullptr;
    size_t hcap = 0;   // words
    bool busy = false;
};
struct HostMulPool {
    std::mutex mu;
    std::condition_variable cv;
    HostMulCtx ctx[HM_CONTEXTS];
} g_hm;

// RAII: a free context for the duration of one product
struct HmLease {
    HostMulCtx *c = nullptr;
    HmLease() {
        std::unique_lock<std::mutex> lk(g_hm.mu);
        for (;;) {
            for (auto &x : g_hm.ctx)
                if (!x.busy) { x.busy = true; c = &x; return; }
            g_hm.cv.wait(lk);
        }
    }
    ~HmLease() {
        {
            std::lock_guard<std::mutex> lk(g_hm.mu);
            c->busy = false;
        }
        g_hm.cv.notify_one();
    }
};

int hm_reserve(HostMulCtx &c, size_t words, size_t host_words) {
    if (!c.st) GF2T_HIP(hipStreamCreateWithFlags(&c.st, hipStreamNonBlocking));
    if (words > c.dcap) {
        if (c.dbuf) GF2T_HIP(hipFree(c.dbuf));
        c.dbuf = nullptr;
        c.dcap = 0;
        size_t want = words + words / 4;
        if (hipMalloc(&c.dbuf, want * 8) != hipSuccess) {
            (void)hipGetLastError();
            gf2t::set_error("gf2t host product service: cannot allocate %zu bytes", want * 8);
            return GF2T_ENOMEM;
        }
        c.dcap = want;
    }
    if (host_words > c.hcap) {
        if (c.hbuf) GF2T_HIP(hipHostFree(c.hbuf));
        c.hbuf = nullptr;
        c.hcap = 0;
        size_t want = host_words + host_words / 4;
        if (hipHostMalloc((void **)&c.hbuf, want * 8, hipHostMallocDefault) != hipSuccess) {
            (void)hipGetLastError();
            gf2t::set_error("gf2t host product service: cannot allocate %zu pinned bytes",
                            want * 8);
            return GF2T_ENOMEM;
        }
        c.hcap = want;
    }
    return GF2T_OK;
}

}  // namespace

int gf2t_hm_set_zc_words(int64_t words) {
    if (words < 0) {
        gf2t::set_error("gf2t_tune: hm_zc_words must be >= 0");
        return GF2T_EINVAL;
    }
    g_hm_zc_words.store(words);
    return GF2T_OK;
}
int64_t gf2t_hm_zc_words() { return g_hm_zc_words.load(); }

extern "C" int gf2t_mul_host(const uint64_t *ha, uint64_t abits, const uint64_t *hb,
                             uint64_t bbits, uint64_t *hout) {
    if ((!ha && abits) || (!hb && bbits) || !hout) {
        gf2t::set_error("gf2t_mul_host: null pointer");
        return GF2T_EINVAL;
    }
    size_t ow = gf2t_mul_out_words(abits, bbits);
    if (!abits || !bbits) {
        std::memset(hout, 0, ow * 8);
        return GF2T_OK;
    }
    HmLease lease;
    HostMulCtx &hc = *lease.c;
    const size_t aw = words_of(abits), bw = words_of(bbits);
    const size_t ww = (gf2t_mul_workspace_bytes(abits, bbits) + 7) / 8;
    int rc = hm_reserve(hc, aw + bw + ow + ww + 64, std::max(aw + bw, ow));
    if (rc) return rc;
    u64 *da = hc.dbuf, *db = da + aw, *dout = db + bw, *dw = dout + ow;
    dw = (u64 *)(((uintptr_t)dw + 255) & ~(uintptr_t)255);
    hipStream_t st = hc.st;
    std::memcpy(hc.hbuf, ha, aw * 8);
    std::memcpy(hc.hbuf + aw, hb, bw * 8);
    GF2T_HIP(hipMemcpyAsync(da, hc.hbuf, (aw + bw) * 8, hipMemcpyHostToDevice, st));
    rc = mul_core(da, abits, db, bbits, dout, dw, st);
    if (rc) return rc;
    GF2T_HIP(hipMemcpyAsync(hc.hbuf, dout, ow * 8, hipMemcpyDeviceToHost, st));
    GF2T_HIP(hipStreamSynchronize(st));
    std::memcpy(hout, hc.hbuf, ow * 8);
    return GF2T_OK;
}

namespace {
// Pair p of a batched matrix-vector product: its two transforms (at F + (4
// + 2p) n and F + (5 + 2p) n) become (m0 a + m1 b, m2 a + m3 b), the
// matrix transforms at F .. F + 3n left as they are.  A thread per unit.
__global__ __launch_bounds__(256) void k_mat2n_pointwise(u64 *__restrict__ F, size_t n,
                                                         int npairs) {
    __shared__ __align__(16) ProdLds pt;
    copy_lds(&pt, g_tab.d32, sizeof(ProdLds) / 16);
    __syncthreads();
    const size_t units = n / 2;
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    const Operand none{};
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < units; i += stride) {
        Half32 M[4], C[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const U4 u = load_unit((const U4 *)(F + k * n), (u32)i, IO_UNITS, none, nullptr);
            M[k] = unit_to32(u, pt.d32);
            C[k] = unit_c5(u, pt.d5);
        }
        for (int p = 0; p < npairs; p++) {
            U4 *fa = (U4 *)(F + (4 + 2 * (size_t)p) * n), *fb = (U4 *)(F + (5 + 2 * (size_t)p) * n);
            const Half32 a = unit_to32(load_unit(fa, (u32)i, IO_UNITS, none, nullptr), pt.d32);
            const Half32 b = unit_to32(load_unit(fb, (u32)i, IO_UNITS, none, nullptr), pt.d32);
#pragma unroll
            for (int o = 0; o < 2; o++) {
                Acc64 E{0, 0}, G{0, 0};
                acc_mul(E, a.v[0], a.v[1], M[2 * o].v[0], M[2 * o].v[1], C[2 * o].v[1]);
                acc_mul(E, b.v[0], b.v[1], M[2 * o + 1].v[0], M[2 * o + 1].v[1], C[2 * o + 1].v[1]);
                acc_mul(G, a.v[2], a.v[3], M[2 * o].v[2], M[2 * o].v[3], C[2 * o].v[3]);
                acc_mul(G, b.v[2], b.v[3], M[2 * o + 1].v[2], M[2 * o + 1].v[3], C[2 * o + 1].v[3]);
                store_unit(o ? fb : fa, (u32)i, unit_back(E, G, pt.b32), IO_UNITS, nullptr);
            }
        }
    }
}
}  // namespace

// Matrix-vector products of up to MAT_PAIRS chunk pairs are formed without
// transforms, whose chain of eight launches (five below 2^9 points) is as
// long however few points it has: two pairs of 64 bits take 18 us and 37 by
// transforms, of 16,000 bits 26 and 87, of 65,000 bits (2^25) 66 and 96.  One
// product at a time is faster so up to 2^26 (one pair of 131,000 bits: 95 and
// 101), but 15 full-size gcds at once, whose products share the chip, take
// 4.45 s with that line and 4.2 with this one (4.39 by transforms alone).
namespace { constexpr u64 MAT_PAIRS = (u64)1 << 25; }

extern "C" int gf2t_mat2n_host(const uint64_t *const hm[4], const uint64_t mbits[4], int npairs,
                               const uint64_t *const *hv, const uint64_t *vbits,
                               uint64_t *const *hout, size_t outw) {
    if (!hm || !mbits || !hv || !vbits || !hout || npairs < 1 || npairs > (PACK_LIST - 4) / 2) {
        gf2t::set_error("gf2t_mat2n_host: bad arguments (1 <= npairs <= %d)", (PACK_LIST - 4) / 2);
        return GF2T_EINVAL;
    }
    const int nv = 2 * npairs;
    u64 mb = 0, vb = 0;
    for (int i = 0; i < 4; i++) {
        if (!hm[i] && mbits[i]) { gf2t::set_error("gf2t_mat2n_host: null entry"); return GF2T_EINVAL; }
        mb = std::max<u64>(mb, mbits[i]);
    }
    for (int i = 0; i < nv; i++) {
        if ((!hv[i] && vbits[i]) || !hout[i]) {
            gf2t::set_error("gf2t_mat2n_host: null operand");
            return GF2T_EINVAL;
        }
        vb = std::max<u64>(vb, vbits[i]);
    }
    if (outw < gf2t_mul_out_words(mb, vb)) {
        gf2t::set_error("gf2t_mat2n_host: outw %zu below %zu", outw, gf2t_mul_out_words(mb, vb));
        return GF2T_EINVAL;
    }
    if (!mb || !vb) {
        for (int i = 0; i < nv; i++) std::memset(hout[i], 0, outw * 8);
        return GF2T_OK;
    }
    u64 cm = (mb + 31) >> 5, cv = (vb + 31) >> 5;
    int m = fft_m_for(cm + cv - 1);
    if (m > FFT_MAX_M) { gf2t::set_error("gf2t_mat2n_host: product too large"); return GF2T_ERANGE; }
    int rc = ensure_basis();
    if (rc) return rc;
    HmLease lease;
    HostMulCtx &hc = *lease.c;
    const gf2t_fft_plan plan = plan_for(m);
    const int nt = 4 + nv;                    // transforms: matrix, then the vectors
    size_t n = (size_t)1 << m, ow = gf2t_mul_out_words(mb, vb);
    const u64 *src[PACK_LIST];
    u64 bits[PACK_LIST];
    size_t in_w[PACK_LIST], stage = 0, lchw = 0;   // words
    for (int i = 0; i < nt; i++) {
        src[i] = i < 4 ? hm[i] : hv[i - 4];
        bits[i] = i < 4 ? mbits[i] : vbits[i - 4];
        in_w[i] = words_of(bits[i]);
        stage += (in_w[i] + 3) & ~(size_t)3;
    }
    lchw = stage;   // the converted chunks of every operand
    // the transforms, or two products' parts for each output
    const SchoolShape sh = school_shape(cm, cv, false);
    const bool direct = cm + cv <= SC_OUTS && 4 * npairs * cm * cv <= MAT_PAIRS;
    const size_t space = direct ? (size_t)2 * nv * sh.nparts * sh.nout : nt * n;
    rc = hm_reserve(hc, space + nv * ow + stage + lchw + 64, std::max(stage, nv * ow));
    if (rc) return rc;
    hipStream_t st = hc.st;
    u64 *F = hc.dbuf;                         // nt transforms, n words apart
    u64 *dout = F + space, *dstage = dout + nv * ow;
    // the operands, 32-byte aligned, in one pinned buffer and one copy
    Operands pk{};
    u64 *lch = dstage + stage;
    size_t off = 0;
    for (int i = 0; i < nt; i++) {
        if (in_w[i]) std::memcpy(hc.hbuf + off, src[i], in_w[i] * 8);
        pk.op[i] = operand_of(dstage + off, bits[i], lch + off);   // n = 0 for a zero operand
        off += (in_w[i] + 3) & ~(size_t)3;
    }
    // small products read their operands from the pinned staging buffer
    // and write their results back into it (the GPU reaches pinned host
    // memory directly), instead of a copy each way
    const bool zc = off + nv * ow <= (size_t)g_hm_zc_words.load(std::memory_order_relaxed);
    if (zc) {
        size_t o2 = 0;
        for (int i = 0; i < nt; i++) {
            pk.op[i].src = (const u32 *)(hc.hbuf + o2);
            o2 += (in_w[i] + 3) & ~(size_t)3;
        }
        dout = hc.hbuf;
    } else if (off) {
        GF2T_HIP(hipMemcpyAsync(dstage, hc.hbuf, off * 8, hipMemcpyHostToDevice, st));
    }
    if (direct) {
        hipLaunchKernelGGL(k_school<SC_MAT>, dim3((SC_IN - 1 + sh.nb + SC_OUT - 1) / SC_OUT, sh.nparts, 2 * nv),
                           dim3(256), 0, st, pk, 0u, cm > cv ? 1 : 0, sh, F,
                           (u64)sh.nparts * sh.nout, (const SchoolJob *)nullptr,
                           (const SchoolBlock *)nullptr);
        hipLaunchKernelGGL(k_school_mat, dim3((unsigned)((ow + SP_WORDS - 1) / SP_WORDS), nv),
                           dim3(256), 0, st, F, sh, dout, ow);
    } else {
        int in;
        rc = run_forward(plan, F, n, pk, log2_ceil(std::max(cm, cv)), (unsigned)nt, true, st, in);
        if (rc) return rc;
        unsigned blocks = (unsigned)std::min<size_t>((n / 2 + 255) / 256, 2048);
        hipLaunchKernelGGL(k_mat2n_pointwise, dim3(blocks), dim3(256), 0, st, F, n, npairs);
        rc = run_inverse(plan, F + 4 * n, n, (unsigned)nv, true, IO_UNITS, st);
        if (rc) return rc;
        size_t nch = (size_t)(cm + cv - 1);
        hipLaunchKernelGGL(k_overlap_add, dim3((unsigned)((ow + 255) / 256), nv), dim3(256), 0, st,
                           F + 4 * n, nch, dout, ow, (u64)n, (u64)ow);
    }
    GF2T_CHECK_LAUNCH("gf2t_mat2n_host");
    if (!zc) GF2T_HIP(hipMemcpyAsync(hc.hbuf, dout, nv * ow * 8, hipMemcpyDeviceToHost, st));
    GF2T_HIP(hipStreamSynchronize(st));
    for (int i = 0; i < nv; i++) {
        std::memcpy(hout[i], hc.hbuf + (size_t)i * ow, ow * 8);
        if (outw > ow) std::memset(hout[i] + ow, 0, (outw - ow) * 8);
    }
    return GF2T_OK;
}

extern "C" int gf2t_mat2_host(const uint64_t *const hm[4], const uint64_t mbits[4],
                              const uint64_t *ha, uint64_t abits, const uint64_t *hb,
                              uint64_t bbits, uint64_t *hoa, uint64_t *hob, size_t outw) {
    const uint64_t *hv[2] = {ha, hb};
    const uint64_t vbits[2] = {abits, bbits};
    uint64_t *hout[2] = {hoa, hob};
    if (!hoa || !hob) {
        gf2t::set_error("gf2t_mat2_host: null pointer");
        return GF2T_EINVAL;
    }
    return gf2t_mat2n_host(hm, mbits, 1, hv, vbits, hout, outw);
}
