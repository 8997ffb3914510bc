// The host rules of the products' launches (cantor.hpp), for CPU checks.
// Test code only.
#include <algorithm>
#include "cantor.hpp"

extern "C" {
unsigned pr_max_pairs() { return cantor_host::MAX_PAIRS; }
// group[j], place[j]: of pair j (-1: none); size[g]: transform size of group g
int pr_groups(const int *m, int n, int *group, int *place, int *size) {
    const auto v = cantor_host::size_groups(std::vector<int>(m, m + n));
    for (int j = 0; j < n; j++) group[j] = place[j] = -1;
    for (size_t g = 0; g < v.size(); g++) {
        size[g] = v[g].m;
        for (size_t i = 0; i < v[g].pairs.size(); i++) {
            group[v[g].pairs[i]] = (int)g;
            place[v[g].pairs[i]] = (int)i;
        }
    }
    return (int)v.size();
}
// v[j]: pair j is formed without transforms
void pr_direct(const int *m, const u64 *ca, const u64 *cb, int n, char *v) {
    const auto d = cantor_host::direct_pairs(std::vector<int>(m, m + n), std::vector<u64>(ca, ca + n),
                                             std::vector<u64>(cb, cb + n));
    std::copy(d.begin(), d.end(), v);
}
u64 pr_direct_pairs() { return cantor_host::DIRECT_PAIRS; }
// whether products of ca x cb chunks wrap, and the sizes
int pr_wrap(u64 ca, u64 cb, u64 nbatch, int *mp, int *ms, u64 *e) {
    const auto w = cantor_host::wrap_for(ca, cb, nbatch);
    *mp = w.mp;
    *ms = w.ms;
    *e = w.e;
    return w.on;
}
}
