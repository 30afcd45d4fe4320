// CPU build driver, for the sanitizer build: a sorted join whose buckets hold more
// than 1024 spread build keys each (work-groups of 1024 threads, one s_payload
// interval per key), with s_payloads over the whole int32 range; or, with an
// argument, one of many buckets of few rows and a key of 4000.
#include <algorithm>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <tuple>
#include <vector>

#include "qo.h"

#define CK(x)                                                                     \
    do {                                                                          \
        int rc_ = (x);                                                            \
        if (rc_ != QO_OK) {                                                       \
            fprintf(stderr, "%s:%d %s -> %d (%s)\n", __FILE__, __LINE__, #x, rc_, \
                    qo_last_error());                                             \
            exit(1);                                                              \
        }                                                                         \
    } while (0)

static int32_t *dev(const std::vector<int32_t> &h) {
    void *p = nullptr;
    CK(qo_malloc(&p, h.size() * 4));
    CK(qo_memcpy_h2d(p, h.data(), h.size() * 4));
    return static_cast<int32_t *>(p);
}

int main(int argc, char **) {
    const bool hot = argc > 1;
    CK(qo_init(0));
    // One key holds 3000 rows, so buckets need the larger work-groups; 500 rows are
    // spread over 10,000 keys 3355 apart, so a bucket of some 500 rows holds a
    // thousand keys and more.  The rest of S does not pass the filter.
    const size_t nr = hot ? 6000 : 10000, ns = 20000, hot_rows = hot ? 4000 : 3000, rows = hot ? ns : 3500;
    std::vector<int32_t> rk(nr), rp(nr), sk(ns), sp(ns), sf(ns);
    for (size_t i = 0; i < nr; ++i) {
        rk[i] = (int32_t)(i * 3355) - 15000000;
        rp[i] = (int32_t)i;
    }
    uint32_t x = 12345;
    auto rnd = [&] { return x = x * 1664525u + 1013904223u; };
    std::vector<std::tuple<int32_t, int32_t, int32_t>> want;
    for (size_t i = 0; i < ns; ++i) {
        const size_t at = i * 7919 % ns, r = i < hot_rows ? 77 : (rnd() >> 8) % nr;
        sk[at] = rk[r];
        sp[at] = i == 0 ? INT32_MIN : i == 1 ? INT32_MAX : (int32_t)rnd();
        sf[at] = i < rows ? 1 : 2;
        if (i < rows) want.emplace_back(rk[r], sp[at], rp[r]);
    }
    std::sort(want.begin(), want.end());
    const size_t tb = qo_join_table_bytes(nr);
    void *table = nullptr;
    CK(qo_malloc(&table, tb));
    const std::vector<int32_t> zero(ns, 0);
    int32_t *drk = dev(rk), *drp = dev(rp), *dsk = dev(sk), *dsp = dev(sp), *dsf = dev(sf), *o[3] = {dev(zero), dev(zero), dev(zero)};
    uint64_t m = 0;
    CK(qo_hj_filter_sort(table, tb, drk, drp, nr, dsk, dsp, dsf, ns, 0, 1, o[0], o[1], o[2], ns, &m, nullptr));
    bool ok = m == want.size();
    for (size_t i = 0; ok && i < m; ++i) ok = want[i] == std::make_tuple(o[0][i], o[2][i], o[1][i]);
    for (void *p : {table, (void *)drk, (void *)drp, (void *)dsk, (void *)dsp, (void *)dsf,
                    (void *)o[0], (void *)o[1], (void *)o[2]})
        CK(qo_free(p));
    CK(qo_release_workspaces());
    printf("%llu rows %s\n%s\n", (unsigned long long)m, ok ? "in order" : "wrong", ok ? "PASS" : "FAIL");
    return ok ? 0 : 1;
}
