// Single tiles of the Cantor transform's butterfly windows (cantor.hpp)
// against GF(2^64) products, for CPU checks at sizes whose whole transform
// would take too long.  Test code only.
#include <random>
#include <stdlib.h>
#include "cantor.hpp"

static FftTables T;
struct Tab {
    Mul8 operator()(u32 off) const {
        if (off > 255 * 16 || off % 16) abort();
        const u32 *e = T.mulA[off / 16];
        return Mul8{e[0], e[1], e[2], e[3], T.mulB[off / 16]};
    }
};
template <int CLS>
static void tile(std::vector<U4> &x, const BfPass &P, const BfTile &t, bool inv) {
    const int ns = bf_stages(P);
    for (int k = 0; k < ns; k++) {
        const int s = inv ? ns - 1 - k : k;
        for (u32 tid = 0; tid < 1u << (P.tb - RB); tid++) {
            U4 y[1 << RB];
            TwEnt W[RB];
            for (int r = 0; r < (1 << RB); r++) y[r] = x.at(bf_local(P, s, tid, r));
            bf_twiddles(P, t, s, tid, T.tw, W);
            if (inv) fft_stage<CLS, true>(y, bf_active(P, s), W, bf_zero(P, t, s), Tab());
            else fft_stage<CLS, false>(y, bf_active(P, s), W, bf_zero(P, t, s), Tab());
            for (int r = 0; r < (1 << RB); r++) x.at(bf_local(P, s, tid, r)) = y[r];
        }
    }
}
extern "C" {
// tile blk of window number `pass` of 2^m points; -1: no such window, 0:
// equal, 1: not; cls: the window's class
int cw_check(const u64 *b, int m, int tile_bits, int pass, u64 blk, int inv, int *cls) {
    static const bool ok = cantor_host::build_tables(b, T);
    const std::vector<BfPass> ps = cantor_host::bf_passes(m, tile_bits);
    if (!ok || pass >= (int)ps.size()) return -1;
    const BfPass &P = ps[pass];
    *cls = cantor_host::bf_class(P);
    const BfTile t = bf_tile(P, (u32)(blk & (((u64)1 << (m - 1 - P.tb)) - 1)));
    const u32 n = 1u << P.tb;
    std::mt19937_64 rng(blk);
    std::vector<u64> e(2 * n);
    for (u64 &v : e) v = rng();
    std::vector<U4> x(n);
    for (u32 l = 0; l < n; l++) x[l] = unit_embed64(e[2 * l], e[2 * l + 1], T.emb);
    if (*cls == 8) tile<8>(x, P, t, inv != 0);
    else if (*cls == 16) tile<16>(x, P, t, inv != 0);
    else tile<32>(x, P, t, inv != 0);
    // the same levels on the elements, by their indexes
    std::vector<u64> at(2 * n);
    for (u32 l = 0; l < n; l++)
        for (u32 h = 0; h < 2; h++) at[2 * l + h] = 2 * (u64)bf_unit(P, t, l) + h;
    for (int k = 0; k < P.w; k++) {
        const int L = inv ? P.a + k : P.a + P.w - 1 - k;
        const u32 step = 2u << (P.tb - P.w + L - P.a);   // of the partner in the tile
        for (u32 i = 0; i < 2 * n; i++) {
            if ((at[i] >> L) & 1) continue;
            if (at[i + step] != (at[i] | (u64)1 << L)) abort();
            u64 w = 0;
            for (int j = 0; j + L + 1 < m; j++)
                if ((at[i] >> (L + 1 + j)) & 1) w ^= b[j + 1];
            if (inv) e[i + step] ^= e[i];
            e[i] ^= gf64_mul(w, e[i + step]);
            if (!inv) e[i + step] ^= e[i];
        }
    }
    for (u32 l = 0; l < n; l++) {
        u64 f, g;
        unit_unembed(x[l], T.une, f, g);
        if (f != e[2 * l] || g != e[2 * l + 1]) return 1;
    }
    return 0;
}
}
