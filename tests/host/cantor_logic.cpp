// Host emulation of the Cantor transform's kernels (cantor.hpp): the same
// tables, index maps and arithmetic, thread by thread, for CPU checks
// against the oracle.  Test code only.
#include <stdlib.h>
#include <string.h>
#include <vector>
#include "cantor.hpp"

static FftTables T;

struct Tab {
    Mul8 operator()(u32 off) const {
        if (off > 255 * 16 || off % 16) abort();
        const u32 *e = T.mulA[off / 16];
        return Mul8{e[0], e[1], e[2], e[3], T.mulB[off / 16]};
    }
};

template <class E>
static void step(std::vector<E> &f, const ConvStep &s, int k, bool inv) {
    const int R = 1 << s.K;
    const size_t row = (size_t)1 << s.hb, blk = row << s.K;
    std::vector<char> seen(f.size(), 0);
    auto at = [&](size_t b, int r, size_t col) -> E & {
        const size_t i = b + r * row + col;
        if (col >= row || i >= f.size()) abort();
        return f[i];
    };
    for (size_t b = 0; b < f.size(); b += blk) {
        for (u32 t = 0; t < conv_full(s); t++) {
            E x[16];
            for (int r = 0; r < R; r++) {
                x[r] = at(b, r, conv_col(s, t, r));
                seen[b + r * row + conv_col(s, t, r)]++;
            }
            for (int j = 0; j < s.K; j++) {
                const int e = inv ? j : s.K - 1 - j;
                for (int r = 0; r < R; r++)
                    if ((r >> e) & 1) x[r ^ (1 << e)] ^= x[r];
            }
            for (int r = 0; r < R; r++) at(b, r, conv_col(s, t, r)) = x[r];
        }
        for (u32 rho = 0; rho < (1u << s.ub); rho++) {
            std::vector<E> x(R * R);
            for (int r = 0; r < R; r++)
                for (int q = 0; q < R; q++) {
                    x[r * R + q] = at(b, r, conv_edge(s, r, q, rho));
                    seen[b + r * row + conv_edge(s, r, q, rho)]++;
                }
            for (int j = 0; j < s.K; j++) {
                const int e = inv ? j : s.K - 1 - j;
                for (u32 idx = 0; idx < (u32)(R * R / 2); idx++)
                    conv_edge_pair([&](u32 i) -> E & { return x.at(i); }, s.K, e, inv, idx);
            }
            for (int r = 0; r < R; r++)
                for (int q = 0; q < R; q++) at(b, r, conv_edge(s, r, q, rho)) = x[r * R + q];
        }
    }
    for (char c : seen)
        if (c != 1) abort();
    (void)k;
}
template <class E, bool INV>
static void tile(std::vector<E> &f, const ConvTile &t, size_t n) {
    const int T = t.c + t.w;
    const u32 sz = 1u << T, threads = sz >> 4;
    for (u32 blk = 0; blk == 0 || (size_t)blk < n >> T; blk++) {
        std::vector<E> x(sz, 0);
        const u64 base = tile_base(t, blk);
        for (u32 l = 0; l < sz; l++)
            if (base + tile_mem(t, l) < n) x[l] = f.at(base + tile_mem(t, l));
        for (int i = 0; i < t.n; i++) {
            const ConvStep &s = t.st[INV ? t.n - 1 - i : i];
            std::vector<int> owner(sz, -1);   // no two threads touch one coefficient
            for (u32 q = 0; q < threads; q++)
                conv_tile_stage<INV, E>(
                    [&](u32 l) -> E & {
                        if (s.K != 1 && owner.at(l) >= 0 && owner[l] != (int)q) abort();
                        owner.at(l) = (int)q;
                        return x[l];
                    },
                    q, threads, s);
        }
        for (u32 l = 0; l < sz; l++)
            if (base + tile_mem(t, l) < n) f.at(base + tile_mem(t, l)) = x[l];
            else if (x[l]) abort();
    }
}
template <class E>
static void convert(std::vector<E> &f, int k, int one, int tb, bool inv) {
    const cantor_host::ConvPlan P = cantor_host::conv_plan(k, one, tb);
    if (!inv) {
        for (auto &s : P.steps) step(f, s, k, false);
        for (auto &t : P.tiles) tile<E, false>(f, t, f.size());
    } else {
        for (size_t i = P.tiles.size(); i--;) tile<E, true>(f, P.tiles[i], f.size());
        for (size_t i = P.steps.size(); i--;) step(f, P.steps[i], k, true);
    }
}

template <int CLS>
static void pass(std::vector<U4> &f, const BfPass &P, bool inv) {
    const u32 threads = 1u << (P.tb - RB);
    for (size_t blk = 0; blk < f.size() >> P.tb; blk++) {
        const BfTile T0 = bf_tile(P, (u32)blk), &t = T0;
        std::vector<U4> x((size_t)1 << P.tb);
        for (u32 l = 0; l < x.size(); l++) x[l] = f.at(bf_unit(P, t, l));
        const int ns = bf_stages(P);
        for (int k = 0; k < ns; k++) {
            const int s = inv ? ns - 1 - k : k;
            for (u32 tid = 0; tid < threads; tid++) {
                U4 y[1 << RB];
                TwEnt W[RB];
                for (int r = 0; r < (1 << RB); r++) y[r] = x.at(bf_local(P, s, tid, r));
                bf_twiddles(P, t, s, tid, T.tw, W);
                const bool zero = bf_zero(P, T0, s);
                if (inv) fft_stage<CLS, true>(y, bf_active(P, s), W, zero, Tab());
                else fft_stage<CLS, false>(y, bf_active(P, s), W, zero, Tab());
                for (int r = 0; r < (1 << RB); r++) x.at(bf_local(P, s, tid, r)) = y[r];
            }
        }
        for (u32 l = 0; l < x.size(); l++) f.at(bf_unit(P, t, l)) = x[l];
    }
}
template <int CA, int CB>
static void low(std::vector<U4> &f, int m, bool inv) {
    const u32 N = 64u << RB;
    TwEnt hi[4];
    for (u32 i = 0; i < 4; i++) hi[i] = tw_of(T.tw, i << 7);
    for (u32 base = 0; base < f.size(); base += N) {
        std::vector<U4> x(N);
        for (u32 l = 0; l < N; l++) {
            if (base + l < f.size()) x[l] = f[base + l];
            else memset(&x[l], 0, sizeof(U4));
        }
        const int ns = lo_stages();
        for (int k = 0; k < ns; k++) {
            const int s = inv ? ns - 1 - k : k;
            for (u32 lane = 0; lane < 64; lane++) {
                U4 y[1 << RB];
                TwEnt W[RB], W0{};
                for (int r = 0; r < (1 << RB); r++) y[r] = x.at(lo_unit(s, lane, r));
                static_assert(lo_stages() == 4, "stages");
                if (s == 0) lo_twiddles<0>(base, lane, T.tw, hi, W, W0);
                if (s == 1) lo_twiddles<1>(base, lane, T.tw, hi, W, W0);
                if (s == 2) lo_twiddles<2>(base, lane, T.tw, hi, W, W0);
                if (s == 3) lo_twiddles<3>(base, lane, T.tw, hi, W, W0);
                const int act = lo_active(m, s);
                if (inv) {
                    if (s == ns - 1) fft_level0<CB, true>(y, W0, Tab());
                    if (s) fft_stage<CB, true>(y, act, W, false, Tab());
                    else fft_stage<CA, true>(y, act, W, false, Tab());
                } else {
                    if (s) fft_stage<CB, false>(y, act, W, false, Tab());
                    else fft_stage<CA, false>(y, act, W, false, Tab());
                    if (s == ns - 1) fft_level0<CB, false>(y, W0, Tab());
                }
                for (int r = 0; r < (1 << RB); r++) x.at(lo_unit(s, lane, r)) = y[r];
            }
        }
        for (u32 l = 0; l < N && base + l < f.size(); l++) f[base + l] = x[l];
    }
}
static void butterflies(std::vector<U4> &f, int m, int tb, bool inv) {
    const std::vector<BfPass> ps = cantor_host::bf_passes(m, tb);
    auto lo = [&] {
        if (m <= 16) low<16, 16>(f, m, inv);
        else if (m <= 24 - RB) low<16, 32>(f, m, inv);
        else low<32, 32>(f, m, inv);
    };
    if (inv) lo();
    for (size_t i = 0; i < ps.size(); i++) {
        const BfPass &P = ps[inv ? ps.size() - 1 - i : i];
        const int c = cantor_host::bf_class(P);
        if (c == 8) pass<8>(f, P, inv);
        else if (c == 16) pass<16>(f, P, inv);
        else pass<32>(f, P, inv);
    }
    if (!inv) lo();
}

extern "C" {
int cl_init(const u64 *basis) { return cantor_host::build_tables(basis, T) ? 0 : 1; }
// transform of 2^m elements, as gf2t_fft_fwd / gf2t_fft_inv run it
void cl_fft(u64 *f, int m, int inv, int one, int tb, int bf) {
    const size_t n = (size_t)1 << m;
    std::vector<u64> v(f, f + n);
    if (!inv) convert(v, m, one, tb, false);
    std::vector<U4> u(n / 2);
    for (size_t i = 0; i < n / 2; i++) u[i] = unit_embed64(v[2 * i], v[2 * i + 1], T.emb);
    butterflies(u, m, bf, inv != 0);
    for (size_t i = 0; i < n / 2; i++) unit_unembed(u[i], T.une, v[2 * i], v[2 * i + 1]);
    if (inv) convert(v, m, one, tb, true);
    memcpy(f, v.data(), n * 8);
}
// chunk products: a, b of na, nb 32-bit chunks, 2^m points >= na + nb - 1;
// out: 2^m 64-bit coefficients
void cl_product(const u32 *a, size_t na, const u32 *b, size_t nb, int m, u64 *out, int one, int tb,
                int bf) {
    const size_t n = (size_t)1 << m;
    std::vector<U4> F[2];
    for (int o = 0; o < 2; o++) {
        const u32 *s = o ? b : a;
        const size_t c = o ? nb : na;
        int k = 0;
        while (((size_t)1 << k) < c) k++;
        std::vector<u32> v((size_t)1 << k, 0);
        for (size_t i = 0; i < c; i++) v[i] = s[i];
        convert(v, k, one, tb, false);
        for (size_t i = c; i < v.size(); i++)
            if (v[i]) abort();   // the conversion keeps the degree
        v.resize(n, 0);
        F[o].resize(n / 2);
        for (size_t i = 0; i < n / 2; i++) F[o][i] = unit_embed32(v[2 * i], v[2 * i + 1], T.emb);
        butterflies(F[o], m, bf, false);
    }
    for (size_t i = 0; i < n / 2; i++) F[0][i] = unit_mul(F[0][i], F[1][i], T.d32, T.d5, T.b32);
    butterflies(F[0], m, bf, true);
    std::vector<u64> v(n);
    for (size_t i = 0; i < n / 2; i++) unit_unembed(F[0][i], T.une, v[2 * i], v[2 * i + 1]);
    convert(v, m, one, tb, true);
    memcpy(out, v.data(), n * 8);
}
}
