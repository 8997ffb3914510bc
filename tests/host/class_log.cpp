// Host build of the class logarithms (csrc/class_log.hpp) for
// tests/test_class_log.py: the sieve's passes over the same functions the
// kernels call, one class after another.
#include "../../mersenne_trinomial_amd/csrc/class_log.hpp"

extern "C" {

int cl_lyndon(u32 j, int d) { return lyndon_word(j, d, aperiodic_rotations(d)); }
int cl_prefix(u32 w, int n) { return lyndon_prefix(w, n); }
int cl_is_lyndon32(u32 j, int d, u32 M) { return is_lyndon32(j, d, M); }
int cl_maps(u64 q, int d, u32 *map) { return class_host::class_maps(q, d, map); }
u64 cl_minpoly(u32 beta, int d, const u32 *map) {
    return minpoly_seq(trace_sequence(beta, map + CL_RED, map + CL_DUAL, d), d);
}
u64 cl_minpoly_bm(u32 beta, u64 q, int d, u32 tmask) { return minpoly_bm(beta, q, d, tmask); }

// T over the n classes j (elements el = g^j), as k_class_log fills it
void cl_fill(const u32 *j, const u32 *el, u64 n, int d, const u32 *map, u32 *T) {
    for (u64 i = 0; i < n; i++) {
        int k;
        const u32 m = least_rotation(periodic64(map8(map + CL_NORM, el[i]), d), k);
        T[class_index(m, d)] = rotl_d(j[i], k, d);
    }
}
// log of y from T; prod: an unreduced product equal to y modulo q
u32 cl_log(u64 prod, int d, const u32 *map, const u32 *T) {
    int k;
    const u32 m = least_rotation(periodic64(map8(map + CL_NORM, prod), d), k);
    return rotl_d(T[class_index(m, d)], d - k, d);
}
// s == v / j modulo n by the units of eight classes at once, as k_zech:
// out n (0: none), s
void cl_progressions(const u32 *j_, const u32 *v_, int d, const u32 *primes, int np, u32 *n_out,
                     u32 *s_out) {
    const u32 M = (u32)(((u64)1 << d) - 1);
    SievePrime pr[8];
    for (int i = 0; i < np; i++) pr[i] = class_host::sieve_prime(primes[i], M);
    u32 j[8], v[8], un[8], nn[8], pre[8];
    for (int i = 0; i < 8; i++) {
        j[i] = j_[i];
        v[i] = v_[i];
    }
    const u32 ok = progressions(v, j, nn, un, M, pr, np);
    for (int i = 0; i < 8; i++) pre[i] = i ? mulmod_mersenne(pre[i - 1], un[i], d, M) : un[i];
    u32 inv = inv32(pre[7], M);
    for (int i = 7; i >= 0; i--) {
        const u32 iv = i ? mulmod_mersenne(inv, pre[i - 1], d, M) : inv;
        inv = mulmod_mersenne(inv, un[i], d, M);
        u32 s0 = mulmod_mersenne(iv, v[i], d, M);
        if (nn[i] != M) s0 %= nn[i];
        n_out[i] = (ok >> i) & 1 ? nn[i] : 0;
        s_out[i] = s0;
    }
}
}
