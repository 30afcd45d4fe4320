// Sorted join of a batch's small queries: the key-order split of join_sorted.hip
// for many queries in the same launches, planned on the device.
//
// A query of up to 512 buckets is split once by key value and every bucket is
// joined in LDS and written in final order by one work-group, without a hash
// table and without sort passes.  Everything that depends on the columns' values
// (key range, expected rows, bucket width) is measured in the launch itself, so a
// captured batch can be replayed on refreshed columns:
//  * k_bj_scan: build key range per query; 1024 sampled S tuples per query;
//  * k_bj_plan: bucket width per query;
//  * k_bj_split: S (filter fused) and R tiles of all queries to their buckets;
//  * k_bj_list: the buckets in use;
//  * k_bj_finish: one work-group per bucket (sj_bucket), whose rows go behind those
//    of the query's buckets before it, by a look-back;
//  * k_bj_end: queries that a bucket overflowed or that repeat a build key are
//    left to the generic stages of the batch, which otherwise return at once.
// 512 queries of 4K to 64K build rows (99 M S tuples): 1.07 ms, 3.96 ms with the
// generic stages alone.
#include <algorithm>
#include <cmath>

#include "qo_batch.hpp"
#include "qo_sorted.hpp"

namespace qo {

constexpr int kBjThreads = 512;  // finishing work-groups: 3072 S tuples, 1024 build keys
using BjLds = SjLds<false, kBjThreads>;
constexpr int kBjMaxBits = 9;
constexpr uint32_t kBjMaxBuckets = 1u << kBjMaxBits;
constexpr uint32_t kBjRows = BjLds::kRows, kBjKeys = BjLds::kSlots;
constexpr uint32_t kBjWantRows = kBjRows * 3 / 4, kBjWantKeys = kBjKeys * 3 / 4;
constexpr uint32_t kBjSamples = 1024;
static_assert(kBjSamples == 2 * kSplitThreads, "two samples per thread");

// Blocks [0, nrt): smallest and largest key of a build tile.  Blocks from nrt
// on: the samples of one query.
__global__ __launch_bounds__(kSplitThreads) void k_bj_scan(const SjBQuery *__restrict__ qs, SjBState *state,
                                                           const uint2 *__restrict__ rtiles, uint32_t nrt) {
    __shared__ uint32_t s_v[4];
    if (threadIdx.x < 4) s_v[threadIdx.x] = 0;
    __syncthreads();
    if (blockIdx.x < nrt) {
        const uint2 t = rtiles[blockIdx.x];
        const SjBQuery &Q = qs[t.x];
        const uint64_t r0 = (uint64_t)t.y * kSplitTile;
        const uint32_t m = (uint32_t)(Q.nr - r0 < kSplitTile ? Q.nr - r0 : kSplitTile);
        constexpr uint32_t kPer = kSplitTile / kSplitThreads;
        uint32_t lo = 0, hi = 0;  // largest ~key and key, both biased
        uint32_t k[kPer];
#pragma unroll
        for (uint32_t j = 0; j < kPer; ++j) {
            const uint32_t i = j * kSplitThreads + threadIdx.x;
            k[j] = (uint32_t)ld_stream(Q.rkey + r0 + (i < m ? i : 0u)) ^ 0x80000000u;
        }
#pragma unroll
        for (uint32_t j = 0; j < kPer; ++j) {
            lo = max(lo, ~k[j]);
            hi = max(hi, k[j]);
        }
        lo = wave_max(lo);
        hi = wave_max(hi);
        if (lane_id() == 0) {
            atomicMax(&s_v[0], lo);
            atomicMax(&s_v[1], hi);
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            atomicMax(&state[t.x].rmin_inv, s_v[0]);
            atomicMax(&state[t.x].rmax, s_v[1]);
        }
        return;
    }
    const uint32_t q = blockIdx.x - nrt;
    const SjBQuery &Q = qs[q];
    if (!Q.on || Q.ns == 0) return;  // whole block
    // Both samples' loads are issued before either is looked at.
    uint32_t pass = 0, lo = 0, hi = 0, pay[2];
    int32_t f[2];
    bool in[2];
    // Samples come in groups of 8 neighbours, one group per cell of S: 1024 single
    // ones per query touched eight times the memory pages (scan of 512 queries
    // 68 us).
    constexpr uint32_t kGroup = 8, kCells = kBjSamples / kGroup;
    const uint32_t cell = (uint32_t)(Q.ns / kCells);  // ns < 2^32 here
#pragma unroll
    for (uint32_t u = 0; u < 2; ++u) {
        const uint32_t i = u * kSplitThreads + threadIdx.x;
        const uint32_t c = i / kGroup;
        const uint64_t at = Q.ns >= kBjSamples ? (uint64_t)c * cell + hash32(c) % (cell - (kGroup - 1)) + i % kGroup : i;
        in[u] = at < Q.ns;
        pay[u] = in[u] ? (uint32_t)Q.spay[at] : 0u;
        f[u] = in[u] && Q.sfilt ? Q.sfilt[at] : Q.flo;
    }
#pragma unroll
    for (uint32_t u = 0; u < 2; ++u) {
        if (!in[u] || (Q.sfilt && (f[u] < Q.flo || f[u] > Q.fhi))) continue;
        const uint32_t p = pay[u] ^ 0x80000000u;
        ++pass;
        lo = max(lo, ~p);
        hi = max(hi, p);
    }
    pass = wave_sum(pass);
    lo = wave_max(lo);
    hi = wave_max(hi);
    if (lane_id() == 0) {
        atomicAdd(&s_v[0], pass);
        atomicMax(&s_v[1], lo);
        atomicMax(&s_v[2], hi);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        state[q].pass = s_v[0];
        state[q].pmin_inv = s_v[1];
        state[q].pmax = s_v[2];
    }
}

// Bucket width of a query: the widest whose expected rows and build keys fit a
// work-group with a quarter to spare, in at most the query's buckets.  A bucket
// holds no more than all of them, however far its width goes past the keys' span.
QO_DEV void bj_plan_query(const SjBQuery &Q, SjBState &s) {
    if (!Q.on || Q.nr == 0 || Q.ns == 0) return;  // no buckets, no rows
    const uint32_t kmin = ~s.rmin_inv, last = s.rmax - kmin;
    const float span = (float)last + 1.0f, pass = (float)s.pass;
    const float per = Q.ns >= kBjSamples ? (float)Q.ns / kBjSamples : 1.0f;
    const float rows = fminf((float)Q.ns, per * (pass + 4.0f * sqrtf(pass) + 4.0f));
    int sh = 0;
    for (; sh < 31; ++sh) {
        const float w = fminf(1.0f, (float)(uint64_t(2) << sh) / span);
        const bool fits = rows * w <= (float)kBjWantRows && (float)Q.nr * w <= (float)kBjWantKeys;
        if ((last >> sh) == 0 || (!fits && (last >> sh) < Q.nbmax)) break;
    }
    s.kmin = kmin ^ 0x80000000u;
    s.last = last;
    s.sh = (uint32_t)sh;
    s.nb = (last >> sh) + 1u;
    s.pay_bits = 32u - (uint32_t)__clz((int)((s.pmax - ~s.pmin_inv) | 1u));
    const float w = fminf(1.0f, (float)(uint64_t(1) << sh) / span);
    if (s.nb > Q.nbmax || rows * w > 0.9f * kBjRows || (float)Q.nr * w > 0.95f * kBjKeys) {
        s.overflow = 1u;  // the generic stages run it
        s.nb = 0;
    }
}

// words[0] := buckets in use; the buckets of kBjChunk queries are listed together.
constexpr int kBjChunk = 256;
__global__ __launch_bounds__(kBjChunk) void k_bj_plan(const SjBQuery *__restrict__ qs, SjBState *state, int nq,
                                                 uint32_t *words) {
    __shared__ uint32_t s_w[4];
    __shared__ uint32_t s_base;
    const int q = blockIdx.x * kBjChunk + threadIdx.x;
    uint32_t nb = 0;
    if (q < nq) {
        bj_plan_query(qs[q], state[q]);
        nb = state[q].nb;
    }
    const uint32_t ex = block_excl_scan256(nb, s_w);
    if (threadIdx.x == kBjChunk - 1) s_base = atomicAdd(&words[0], ex + nb);
    __syncthreads();
    if (q < nq) state[q].from = s_base;
}

// Lists the buckets of query blockIdx.x with their sizes: first the first bucket of
// each of the chunk's queries, then the second ones, and so on, so that few buckets
// of a query are being finished at the same time.
static_assert(kBjMaxBuckets == 512, "one bucket per thread");
__global__ __launch_bounds__(512) void k_bj_list(const SjBQuery *__restrict__ qs, const SjBState *state,
                                                 int nq, const uint32_t *sctr, const uint32_t *rctr, SjBucket *list) {
    __shared__ uint32_t s_nb[kBjChunk];
    const uint32_t q = blockIdx.x, f = threadIdx.x, q0 = q - q % kBjChunk;
    if (f < (uint32_t)kBjChunk) s_nb[f] = q0 + f < (uint32_t)nq ? state[q0 + f].nb : 0u;
    __syncthreads();
    const SjBState &st = state[q];
    if (f >= st.nb) return;
    uint32_t at = st.from;
    const uint32_t m = min((uint32_t)kBjChunk, (uint32_t)nq - q0);
#pragma unroll 8
    for (uint32_t i = 0; i < m; ++i) at += min(s_nb[i], f) + (q0 + i < q && s_nb[i] > f ? 1u : 0u);
    const size_t c = (size_t)(qs[q].bucket0 + f) * kCtrStride;
    list[at] = SjBucket{q, f, min(sctr[c], kBjRows), min(rctr[c], kBjKeys)};
}

// Blocks [0, nst): S tiles; from nst on: build tiles.
__global__ __launch_bounds__(kSplitThreads) void k_bj_split(const SjBQuery *__restrict__ qs, SjBState *state,
                                                            const uint2 *__restrict__ stiles, uint32_t nst,
                                                            const uint2 *__restrict__ rtiles, uint64_t *sbuckets,
                                                            uint32_t *sctr, uint64_t *rbuckets, uint32_t *rctr) {
    __shared__ SplitLdsT<kBjMaxBuckets> sh;
    const bool build = blockIdx.x >= nst;
    const uint2 t = build ? rtiles[blockIdx.x - nst] : stiles[blockIdx.x];
    const SjBQuery &Q = qs[t.x];
    SjBState &st = state[t.x];
    // nb does not change during this launch (overflow does, so it is not looked
    // at: a block's waves could see different values).
    if (st.nb == 0) return;
    int32_t key[kSplitJ][4], pay[kSplitJ][4];
    uint32_t pass[kSplitJ];
    if (build)
        load_s_tile<kSplitJ, false, kSplitThreads>(Q.rkey, Q.rpay, nullptr, Q.nr, 0, 0, Q.rvec != 0, t.y, key, pay, pass);
    else if (Q.sfilt)
        load_s_tile<kSplitJ, true, kSplitThreads>(Q.skey, Q.spay, Q.sfilt, Q.ns, Q.flo, Q.fhi, Q.svec != 0, t.y, key,
                                                  pay, pass);
    else
        load_s_tile<kSplitJ, false, kSplitThreads>(Q.skey, Q.spay, nullptr, Q.ns, 0, 0, Q.svec != 0, t.y, key, pay, pass);
    const KeySpan span{st.kmin, st.last};
#pragma unroll
    for (int j = 0; j < kSplitJ; ++j)
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            uint32_t d;
            if (!span(key[j][k], d)) pass[j] &= ~(1u << k);
        }
    uint32_t parts = 1;
    while (parts < st.nb) parts *= 2;
    split_block<kSplitJ>(key, pay, pass, span, (int)st.sh, parts, Q.bucket0, build ? rbuckets : sbuckets,
                         FixedLayout{build ? kBjKeys : kBjRows}, build ? rctr : sctr, sh, FlagOverflow{&st.overflow});
}

// lookback over at most kBjMaxBuckets tiles from `near`, the words of the 64 before
// f as read some time before.  With many queries an inclusive prefix is among them;
// with few the words of all predecessors are read together (a query's buckets then
// run at the same time, and a load per 64 of them is a chain of up to eight).
constexpr int kBjWords = kBjMaxBuckets / kWave;
QO_DEV uint64_t bj_word(const uint64_t *status, uint32_t f, int k) {
    const int idx = (int)f - 1 - k * kWave - (int)lane_id();
    return idx >= 0 ? ld_agent(&status[idx]) : kFlagInc;
}
QO_DEV uint64_t bj_lookback(uint64_t *status, uint32_t f, uint32_t aggregate, DevCtl *ctl, uint64_t near) {
    const unsigned lane = lane_id();
    uint64_t excl = 0;
    if (f > 0) {
        const uint32_t limit = ctl->spin_limit;
        for (uint32_t sleeps = 0;;) {  // wave-uniform: the branches depend on ballots only
            uint64_t w[kBjWords];
            uint64_t sum = 0;
            bool done = false, empty = false;
            auto add = [&](uint64_t word) {
                const uint64_t inc = ballot(word >> 62 == 2);
                const unsigned first = inc ? (unsigned)__builtin_ctzll(inc) : 64u;
                const uint64_t relevant = first >= 63 ? ~uint64_t(0) : ((uint64_t(2) << first) - 1);
                empty = (ballot(word >> 62 == 0) & relevant) != 0;
                if (lane <= first) sum += word & kValMask;
                done = inc != 0;
            };
            add(near);
            if (!done && !empty) {
#pragma unroll
                for (int k = 1; k < kBjWords; ++k) w[k] = bj_word(status, f, k);
#pragma unroll
                for (int k = 1; k < kBjWords; ++k)
                    if (!done && !empty) add(w[k]);
            }
            if (!empty) {
                excl = wave_sum(sum);
                break;
            }
            if (++sleeps > limit) {
                if (lane == 0) atomicOr(&ctl->error, kDevErrLookback);
                return 0;
            }
            __builtin_amdgcn_s_sleep(1);
            near = bj_word(status, f, 0);
        }
    }
    if (lane == 0) st_agent(&status[f], kFlagInc | (excl + aggregate));
    return excl;
}

// A bucket's rows go behind the rows of the query's buckets before it.
struct BjChained {
    SjBState *st;
    uint64_t *status;  // of the query's buckets
    uint32_t f;
    DevCtl *ctl;
    QO_DEV void begin(uint32_t total) const {
        // Successors need not wait for the placement.
        if (threadIdx.x == 0) st_agent(&status[f], (f ? kFlagAgg : kFlagInc) | total);
    }
    using Asked = uint64_t;
    QO_DEV void ask(Asked &a) const { a = bj_word(status, f, 0); }
    QO_DEV uint64_t position(uint32_t total, Asked a) const {
        const uint64_t e = bj_lookback(status, f, total, ctl, a);
        if (f == st->nb - 1 && lane_id() == 0) st->rows = e + total;
        return e;
    }
    QO_DEV void repeated() const { st->repeated = 1u; }
};

// One listed bucket, taken by ticket: a query's buckets are listed in order, so
// every predecessor in the look-back is already running or done.  465 us for 512
// queries, 37 of them the tickets (a counter per query, read after the list, 30
// more).  With the buckets listed query by query, so that a query's were all being
// finished at once, and the look-back's words read where they are needed 513.  Rows
// at positions that assume every tuple matches took 363, and left rows behind the
// result where one did not.
__global__ __launch_bounds__(kBjThreads, 8) void k_bj_finish(const SjBQuery *__restrict__ qs, SjBState *state,
                                                             const SjBucket *__restrict__ list,
                                                             uint32_t *words,
                                                             const uint64_t *sbuckets, const uint64_t *rbuckets,
                                                             uint64_t *status, DevCtl *ctl) {
    __shared__ BjLds s;
    if (blockIdx.x >= words[0]) return;
    if (threadIdx.x == 0) s.tile = atomicAdd(&words[1], 1u);
    sj_clear(s);
    __syncthreads();
    const SjBucket e = list[s.tile];
    const SjBQuery &Q = qs[e.q];
    SjBState &st = state[e.q];
    if (st.overflow) return;  // block-uniform: this launch does not set it
    const size_t b = Q.bucket0 + e.f;
    const PayloadBins pbins{~st.pmin_inv, (int)st.pay_bits};
    const SoaEmit emit{Q.okey, Q.orpay, Q.ospay, Q.out_cap};
    sj_bucket(s, sbuckets + b * kBjRows, e.n, rbuckets + b * kBjKeys, e.nr, static_cast<const uint64_t *>(nullptr),
              st.kmin + (e.f << st.sh), (int)st.sh, pbins, emit, BjChained{&st, status + Q.bucket0, e.f, ctl});
}

// Queries that the generic stages still have to run: skip[q] = 0, *any = 1.
__global__ void k_bj_end(const SjBQuery *__restrict__ qs, const SjBState *state, int nq, uint32_t *skip, uint32_t *any) {
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= nq) return;
    const bool done = qs[q].on && !state[q].overflow && !state[q].repeated;
    skip[q] = done;
    if (!done) *any = 1u;
}

// Match counts of the whole batch.
__global__ void k_bj_counts(const SjBState *state, const uint32_t *skip, const unsigned long long *generic, int nq,
                            unsigned long long *counts) {
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q < nq) counts[q] = skip && skip[q] ? state[q].rows : generic[q];
}

void bj_plan_init(const qo_join_query *queries, int nq, const std::vector<char> &generic, SjBatchPlan &p) {
    p = SjBatchPlan{};
    p.q.assign(nq, SjBQuery{});
    p.all_on = true;
    for (int i = 0; i < nq; ++i) {
        const qo_join_query &u = queries[i];
        SjBQuery &q = p.q[i];
        q.rkey = u.rkey; q.rpay = u.rpay; q.skey = u.skey; q.spay = u.spay; q.sfilt = u.sfilt;
        q.nr = u.nr; q.ns = u.ns; q.flo = u.flo; q.fhi = u.fhi;
        q.okey = u.okey; q.orpay = u.orpay; q.ospay = u.ospay; q.out_cap = u.out_capacity;
        q.svec = (((uintptr_t)u.skey | (uintptr_t)u.spay | (uintptr_t)u.sfilt) & 15u) == 0;
        q.rvec = (((uintptr_t)u.rkey | (uintptr_t)u.rpay) & 15u) == 0;
        q.bucket0 = p.buckets;
        // The power-of-two width leaves a bucket at least half of what it may hold;
        // a query that fits one bucket gets two, for keys that span more than 2^31.
        const uint64_t want = 2 * std::max<uint64_t>({1, (u.ns + kBjWantRows - 1) / kBjWantRows,
                                                       (u.nr + kBjWantKeys - 1) / kBjWantKeys}) + 1;
        q.nbmax = want == 3 ? 2u : (uint32_t)std::min<uint64_t>(kBjMaxBuckets, want);
        q.on = !generic[i] && u.ns <= (uint64_t)kBjMaxBuckets * kBjWantRows && u.nr <= (uint64_t)kBjMaxBuckets * kBjWantKeys;
        if (!q.on) {
            q.nbmax = 0;
            p.all_on = false;
            continue;
        }
        p.any_on = true;
        p.buckets += q.nbmax;
        for (uint64_t t = 0; t * kSplitTile < u.ns; ++t) p.stiles.push_back(uint2{(uint32_t)i, (uint32_t)t});
        for (uint64_t t = 0; t * kSplitTile < u.nr; ++t) p.rtiles.push_back(uint2{(uint32_t)i, (uint32_t)t});
    }
}

void bj_plan_carve(SjBatchPlan &p, Carver &cv) {
    if (!p.any_on) return;
    const size_t nq = p.q.size();
    p.d_q = cv.take<SjBQuery>(nq);
    p.d_stiles = cv.take<uint2>(p.stiles.size() + 1);
    p.d_rtiles = cv.take<uint2>(p.rtiles.size() + 1);
    p.list = cv.take<SjBucket>(p.buckets + 1);
    p.skip = cv.take<uint32_t>(nq);
    // Cleared by every launch: state, counters, look-back words.
    p.state = cv.take<SjBState>(nq);
    const size_t from = cv.off - nq * sizeof(SjBState);
    p.sctr = cv.take<uint32_t>((size_t)p.buckets * kCtrStride);
    p.rctr = cv.take<uint32_t>((size_t)p.buckets * kCtrStride);
    p.status = cv.take<uint64_t>(p.buckets);
    p.words = cv.take<uint32_t>(2);
    p.clear_words = (cv.off - from) / 4;
    p.sbuckets = cv.take<uint64_t>((size_t)p.buckets * kBjRows);
    p.rbuckets = cv.take<uint64_t>((size_t)p.buckets * kBjKeys);
}

int bj_plan_upload(const SjBatchPlan &p, hipStream_t st) {
    if (!p.any_on) return QO_OK;
    auto up = [&](void *dst, const void *src, size_t bytes) {
        return bytes ? hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, st) : hipSuccess;
    };
    QO_HIP(up(p.d_q, p.q.data(), p.q.size() * sizeof(SjBQuery)));
    QO_HIP(up(p.d_stiles, p.stiles.data(), p.stiles.size() * sizeof(uint2)));
    QO_HIP(up(p.d_rtiles, p.rtiles.data(), p.rtiles.size() * sizeof(uint2)));
    return QO_OK;
}

int bj_plan_launch(const SjBatchPlan &p, uint32_t *any, hipStream_t st) {
    const int nq = (int)p.q.size();
    const uint32_t nst = (uint32_t)p.stiles.size(), nrt = (uint32_t)p.rtiles.size();
    const unsigned qg = (unsigned)(nq + 255) / 256;
    QO_TRY(launch_fill_u32(p.state, 0, p.clear_words, st));
    k_bj_scan<<<nrt + (unsigned)nq, kSplitThreads, 0, st>>>(p.d_q, p.state, p.d_rtiles, nrt);
    QO_LAUNCHED();
    k_bj_plan<<<qg, 256, 0, st>>>(p.d_q, p.state, nq, p.words);
    QO_LAUNCHED();
    if (nst + nrt) {
        k_bj_split<<<nst + nrt, kSplitThreads, 0, st>>>(p.d_q, p.state, p.d_stiles, nst, p.d_rtiles, p.sbuckets, p.sctr,
                                                        p.rbuckets, p.rctr);
        QO_LAUNCHED();
        k_bj_list<<<(unsigned)nq, 512, 0, st>>>(p.d_q, p.state, nq, p.sctr, p.rctr, p.list);
        QO_LAUNCHED();
        // One block per bucket a query may use (two to four times those in use; 2048
        // blocks that walk the list took a tenth longer).
        k_bj_finish<<<p.buckets, kBjThreads, 0, st>>>(p.d_q, p.state, p.list, p.words, p.sbuckets, p.rbuckets,
                                                      p.status, dev_ctl());
        QO_LAUNCHED();
    }
    k_bj_end<<<qg, 256, 0, st>>>(p.d_q, p.state, nq, p.skip, any);
    QO_LAUNCHED();
    return QO_OK;
}

int bj_counts_launch(const SjBatchPlan &p, const unsigned long long *generic, int nq, unsigned long long *counts,
                     hipStream_t st) {
    k_bj_counts<<<(unsigned)(nq + 255) / 256, 256, 0, st>>>(p.any_on ? p.state : nullptr, p.any_on ? p.skip : nullptr,
                                                            generic, nq, counts);
    QO_LAUNCHED();
    return QO_OK;
}

}  // namespace qo
