// CPU build driver: a group-by whose workspace was sized before another thread
// changed the tune table (more blocks per CU, larger tables, partitioned) writes
// nothing past that workspace, and its rows are right.
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <vector>

#include "qo.h"
#include "qo_internal.hpp"

#define CK(x)                                                                     \
    do {                                                                          \
        int rc_ = (x);                                                            \
        if (rc_ != QO_OK) {                                                       \
            fprintf(stderr, "%s:%d %s -> %d (%s)\n", __FILE__, __LINE__, #x, rc_, \
                    qo_last_error());                                             \
            exit(1);                                                              \
        }                                                                         \
    } while (0)

template <class T>
static T *dev(size_t n) {
    void *p = nullptr;
    CK(qo_malloc(&p, n * sizeof(T)));
    return static_cast<T *>(p);
}

int main() {
    CK(qo_init(0));
    const size_t n = 200000, guard = 64 << 20;
    int fails = 0;
    for (const size_t groups : {size_t(1024), size_t(3000)})
    for (const bool part : {false, true}) {
        std::vector<int32_t> k(n), v(n);
        for (size_t i = 0; i < n; ++i) {
            k[i] = (int32_t)((i * 2654435761u >> 7) % groups);
            v[i] = (int32_t)(i % 1000) - 500;
        }
        int32_t *dk = dev<int32_t>(n), *dv = dev<int32_t>(n);
        CK(qo_memcpy_h2d(dk, k.data(), 4 * n));
        CK(qo_memcpy_h2d(dv, v.data(), 4 * n));
        int32_t *okey = dev<int32_t>(groups), *omin = dev<int32_t>(groups), *omax = dev<int32_t>(groups);
        int64_t *ocount = dev<int64_t>(groups), *osum = dev<int64_t>(groups);
        uint64_t *num = dev<uint64_t>(1);
        CK(qo_tune_reset());
        CK(qo_tune_set(3, 17, 1024, 2048, 1));
        const qo::GroupbyCall call = qo::groupby_call(groups, n);
        const size_t bytes = qo::groupby_ws_bytes(call);
        unsigned char *ws = dev<unsigned char>(bytes + guard);
        memset(ws + bytes, 0xA5, guard);  // device memory of the CPU build is host memory
        if (part) CK(qo_tune_set(6, 17, 512, 64, 1));
        else CK(qo_tune_set(3, 17, 1024, 4096, 8));
        CK(qo::launch_groupby(call, dk, dv, okey, ocount, osum, omin, omax, num, ws, hipStreamPerThread));
        CK(qo_device_sync());
        size_t damaged = 0;
        for (size_t i = 0; i < guard; ++i) damaged += ws[bytes + i] != 0xA5;
        std::map<int32_t, std::pair<int64_t, int64_t>> want;
        for (size_t i = 0; i < n; ++i) {
            want[k[i]].first += 1;
            want[k[i]].second += v[i];
        }
        bool ok = *num == want.size();
        size_t g = 0;
        for (const auto &w : want) {
            ok = ok && okey[g] == w.first && ocount[g] == w.second.first && osum[g] == w.second.second;
            ++g;
        }
        printf("%zu groups: %zu bytes damaged, rows %s\n", groups, damaged, ok ? "right" : "wrong");
        fails += damaged != 0 || !ok;
        for (void *p : {(void *)dk, (void *)dv, (void *)okey, (void *)omin, (void *)omax, (void *)ocount, (void *)osum,
                        (void *)num, (void *)ws})
            CK(qo_free(p));
    }
    printf(fails ? "FAIL\n" : "PASS\n");
    return fails ? 1 : 0;
}
