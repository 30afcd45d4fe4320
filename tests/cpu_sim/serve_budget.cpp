// CPU build driver: served group-bys under a device-memory budget.  A request
// needs the budget of its outputs, global table and sort (under 1.5 MB here), not
// that of the block tables a merge launch would like beside them; with a small
// and with a large budget its result is that of the request alone.
#include <cstdint>
#include <cstdio>
#include <cstdlib>
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

int main() {
    CK(qo_init(0));
    const uint64_t n = 200000, G = 1000;
    int32_t *col[3];
    for (int32_t *&c : col) {
        void *p = nullptr;
        CK(qo_malloc(&p, n * 4));
        c = static_cast<int32_t *>(p);
    }
    CK(qo_gen_uniform_u32((uint32_t *)col[0], n, 1, 2, 0, G, nullptr));
    CK(qo_gen_uniform_u32((uint32_t *)col[1], n, 1, 3, 0, 1u << 16, nullptr));
    CK(qo_gen_uniform_u32((uint32_t *)col[2], n, 1, 4, 0, 1000, nullptr));
    CK(qo_device_sync());
    int bad = 0;
    for (const double mb : {1.5, 8.0, 200.0}) {
        qo_server_config cfg{(uint64_t)(mb * 1e6), 1, 4, 0, 600000.0};
        qo_server *sv = nullptr;
        CK(qo_server_create(&cfg, &sv));
        const qo_table_desc d{nullptr, nullptr, col[0], col[1], col[2], n, G};
        int id = 0;
        CK(qo_server_add_table(sv, &d, &id));
        std::vector<qo_request> reqs;
        for (const int hi : {99, 999, 499, 0}) {
            const qo_request r{QO_Q_GROUPBY, id, -1, 0, hi};
            uint64_t rid = 0;
            CK(qo_server_submit(sv, &r, &rid));
            reqs.push_back(r);
        }
        CK(qo_server_run(sv));
        std::vector<qo_result> res(reqs.size());
        const int got = qo_server_poll(sv, res.data(), (int)res.size(), 0);
        int same = 0;
        for (int i = 0; i < got; ++i) {
            qo_result alone{};
            CK(qo_server_run_plain(sv, &reqs[(res[i].id - 1) % reqs.size()], &alone));
            same += res[i].status == QO_OK && res[i].count == alone.count && res[i].checksum == alone.checksum;
        }
        printf("%.1f MB: %d of %zu served as alone\n", mb, same, reqs.size());
        bad += same != (int)reqs.size();
        CK(qo_server_destroy(sv));
    }
    printf(bad ? "FAIL\n" : "PASS\n");
    return bad ? 1 : 0;
}
