// Sorted filtered join by key order (qo_hj_filter_sort, unique build keys).
//
// The generic path probes in arrival order and then sorts the joined rows with
// radix passes, each of which reads and writes all of them.  Here S is split by
// key value instead of by hash: bucket f holds the S tuples (and the build
// tuples) with key - kmin in [f << sh, (f + 1) << sh), small enough that one
// work-group joins it in LDS and writes its rows in their final order, so the
// rows move twice (one split, or two) before they are written once.
//
//  * k_sj_sample: 16384 S tuples give the host the expected number of rows, how
//    evenly their keys spread over the build range and the hottest key.
//  * k_sj_split1 / k_sj_split2: S (filter fused; keys outside the build range
//    dropped) into up to 256 buckets, each again into up to 256.
//  * k_sj_finish: per bucket, looks every tuple up, counts the matches per
//    (build key, s_payload interval) in LDS, scans the counts, places the rows
//    and ranks each in its bin's run.
// A key-range table (dense keys) serves the lookup directly: the bucket's slots
// are a contiguous table slice and the slot is the key's rank.  For other keys
// the build tuples are split the same way and ordered in LDS by bins of the
// bucket's key interval.  A bucket that overflows (skew that the sample did not
// show) sets a flag; nothing is written then and the generic path runs.
//
// Only rows of the result are written: where a bucket's rows start is known
// beforehand when every tuple in the build range must have a match (the build
// keys are the whole range), and comes from a look-back over the buckets'
// matches otherwise.  More rows than the outputs hold: none is written.
//
// Whole calls, generic path -> this one: 2^28 S rows, half selected, 2^24 dense
// build keys 5.64 -> 2.44 ms (split 0.96, second split 0.55, finish 0.67, build
// 0.2); 12,000,008 S rows, half selected, 1,500,001 spread 31-bit keys 684 ->
// 349 us; 16384 S rows, half selected, 4096 spread keys 204 -> 75 us (the
// table built by one work-group).
#include <algorithm>
#include <cmath>
#include <cstddef>
#include <cstring>

#include "qo_internal.hpp"
#include "qo_join.hpp"
#include "qo_sorted.hpp"

namespace qo {

constexpr uint32_t kSjSamples = 16384;
constexpr uint32_t kSjBins = 256;
constexpr int kSjHotBits = 16;
constexpr int kSjHotRounds = 8;

// What the host plans from: the table's state and the sample's counts.
struct SjInfo {
    uint32_t mode, dups;   // dups: repeated keys or (-1, -1) build tuples
    int32_t rmin, rmax;
    uint32_t pass;         // sampled tuples that pass the filter inside the build range
    uint32_t hot;          // most samples with one key (to the collisions of kSjHotBits hash bits)
    uint32_t pmin, pmax;   // ~smallest and largest sampled s_payload, both as value ^ 2^31
    uint32_t bin[kSjBins];
};

QO_DEV int span_bin_shift(uint32_t last) { return last < kSjBins ? 0 : 24 - __clz((int)last); }

// Thread i samples tuple i of an even grid over S, jittered inside its cell.
// `keys` counts the samples by key hash (zeroed, like *info, beforehand).
constexpr int kSjSampleThreads = 1024;  // few blocks: their counts meet in same-address atomics
template <bool HAS_FILTER>
__global__ __launch_bounds__(kSjSampleThreads) void k_sj_sample(const JoinHeader *__restrict__ hdr, const int32_t *__restrict__ skey,
                                                   const int32_t *__restrict__ spay,
                                                   const int32_t *__restrict__ sfilt, size_t ns, int32_t flo,
                                                   int32_t fhi, SjInfo *info, uint32_t *keys) {
    __shared__ uint32_t s_bin[kSjBins];
    __shared__ uint32_t s_pass, s_hot, s_pmin, s_pmax;
    if (threadIdx.x < kSjBins) s_bin[threadIdx.x] = 0;
    if (threadIdx.x == 0) s_pass = s_hot = s_pmin = s_pmax = 0;
    const uint32_t i = blockIdx.x * kSjSampleThreads + threadIdx.x;
    const uint64_t cell = ns >= kSjSamples ? ns / kSjSamples : 1;
    const uint64_t at = ns >= kSjSamples ? (uint64_t)i * cell + hash32(i) % cell : i;
    const uint32_t last = (uint32_t)hdr->rmax - (uint32_t)hdr->rmin;
    const KeySpan span{(uint32_t)hdr->rmin, last};
    bool in = at < ns;
    const int32_t key = in ? skey[at] : 0;
    const int32_t filt = HAS_FILTER && in ? sfilt[at] : 0;
    const uint32_t pay = in ? (uint32_t)spay[at] ^ 0x80000000u : 0u;
    uint32_t d = 0;
    in = in && span(key, d) && (!HAS_FILTER || (filt >= flo && filt <= fhi));
    __syncthreads();
    const uint64_t m = ballot(in);
    // Samples of one key meet at one address, where 16384 take 0.2 ms: a few keys
    // of the wave are counted there once, which a hot one is unlikely to escape.
    uint32_t hot = in ? 1u : 0u;  // samples this lane counts
    uint64_t open = m;
#pragma unroll
    for (int r = 0; r < kSjHotRounds; ++r) {
        // Another part of the wave each time: hot keys may come in any pattern.
        const uint64_t from = open >> (r * (kWave / kSjHotRounds)) << (r * (kWave / kSjHotRounds));
        if (from == 0) continue;
        const int leader = __builtin_ctzll(from);
        const uint64_t same = ballot(key == __shfl(key, leader, kWave)) & open;
        if ((same >> lane_id()) & 1u) hot = (int)lane_id() == leader ? popc(same) : 0u;
        open &= ~same;
    }
    if (hot) hot += atomicAdd(&keys[hash32((uint32_t)key) >> (32 - kSjHotBits)], hot);
    if (in) atomicAdd(&s_bin[(d >> span_bin_shift(last)) & (kSjBins - 1)], 1u);
    hot = wave_max(hot);
    const uint32_t pmin = wave_max(in ? ~pay : 0u), pmax = wave_max(in ? pay : 0u);
    if (lane_id() == 0 && m) {
        atomicAdd(&s_pass, popc(m));
        atomicMax(&s_hot, hot);
        atomicMax(&s_pmin, pmin);
        atomicMax(&s_pmax, pmax);
    }
    __syncthreads();
    if (threadIdx.x < kSjBins && s_bin[threadIdx.x]) atomicAdd(&info->bin[threadIdx.x], s_bin[threadIdx.x]);
    if (threadIdx.x == 0 && s_pass) {
        atomicAdd(&info->pass, s_pass);
        atomicMax(&info->hot, s_hot);
        atomicMax(&info->pmin, s_pmin);
        atomicMax(&info->pmax, s_pmax);
    }
    if (i == 0) {
        info->mode = hdr->mode;
        info->dups = hdr->has_dups | hdr->sentinel_count | hdr->overflow;
        info->rmin = hdr->rmin;
        info->rmax = hdr->rmax;
    }
}

// *flag of a sorted join (a split's overflowing bucket stores kSjOverflow): with
// one of the first two the finish writes nothing; the finish sets kSjWait when its
// look-back gave up.
constexpr uint32_t kSjOverflow = 1u, kSjFull = 2u, kSjWait = 4u;
constexpr int kSjPartBits = 8;
using SjSplitLds = SplitLdsT<1u << kSjPartBits>;

// Columns -> `parts` buckets of (key - kmin) >> shift.
// The table the plan counts on, which was not built yet when it was made: off with
// repeated keys, (-1, -1) build tuples or a table of the other kind.
struct SjGate {
    const JoinHeader *hdr;
    uint32_t mode;
    QO_DEV bool off() const {
        return (hdr->has_dups | hdr->sentinel_count | hdr->overflow) != 0 || hdr->mode != mode;
    }
};

template <bool HAS_FILTER, class Layout>
__global__ __launch_bounds__(kSplitThreads) void k_sj_split1(const int32_t *__restrict__ kcol,
                                                             const int32_t *__restrict__ pcol,
                                                             const int32_t *__restrict__ fcol, size_t n, int32_t flo,
                                                             int32_t fhi, bool vec, KeySpan span, int shift,
                                                             uint32_t parts, uint64_t *__restrict__ bucket, Layout out,
                                                             uint32_t *ctr, FlagOverflow overflow, SjGate gate) {
    __shared__ SjSplitLds sh;
    if (gate.off()) return;  // the whole grid
    int32_t key[kSplitJ][4], pay[kSplitJ][4];
    uint32_t pass[kSplitJ];
    load_s_tile<kSplitJ, HAS_FILTER, kSplitThreads>(kcol, pcol, fcol, n, flo, fhi, vec, blockIdx.x, key, pay, pass);
#pragma unroll
    for (int j = 0; j < kSplitJ; ++j)
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            uint32_t d;
            if (!span(key[j][k], d)) pass[j] &= ~(1u << k);
        }
    split_block<kSplitJ>(key, pay, pass, span, shift, parts, 0, bucket, out, ctr, sh, overflow);
}

// Bucket b of the first split (its XCD regions) -> fine buckets (b << b2) +
// part.  Block order as in the L2 probe: work-group i runs on XCD i % 8, which
// walks its own buckets one after another, so that one L2 completes the lines
// of a fine bucket's runs.
__global__ __launch_bounds__(kSplitThreads) void k_sj_split2(const uint64_t *__restrict__ in, uint64_t incap,
                                                             const uint32_t *inctr, uint32_t nb1, uint32_t tpr,
                                                             KeySpan span, int shift, int b2,
                                                             uint64_t *__restrict__ bucket, FixedLayout out,
                                                             uint32_t *ctr, FlagOverflow overflow, SjGate gate) {
    __shared__ SjSplitLds sh;
    if (gate.off()) return;  // the whole grid
    const uint32_t x = blockIdx.x & 7u, q = blockIdx.x >> 3;
    const uint32_t per = kXcdRegions * tpr;
    const uint32_t b = (q / per) * 8u + x, rem = q % per;
    if (b >= nb1) return;
    const uint32_t reg = b * kXcdRegions + rem / tpr;
    uint64_t n = inctr[reg * kCtrStride];
    if (n > incap) n = incap;
    const uint64_t e0 = (uint64_t)(rem % tpr) * kSplitTile;
    if (e0 >= n) return;  // whole block: no barrier has been reached
    const uint32_t m = (uint32_t)(n - e0 < kSplitTile ? n - e0 : kSplitTile);
    int32_t key[kSplitJ][4], pay[kSplitJ][4];
    uint32_t pass[kSplitJ];
    load_pairs<kSplitJ, kSplitThreads>(in + (size_t)reg * incap + e0, m, key, pay, pass);
    split_block<kSplitJ>(key, pay, pass, span, shift, 1u << b2, b << b2, bucket, out, ctr, sh, overflow);
}

// off[f]: where the rows of bucket f start when every S tuple of a bucket has
// a match (off[nb]: their number, also in *d_count; more than `cap` sets kSjFull).
// Block b scans the 2^b2 buckets of first-split bucket b behind the totals of the
// first-split buckets before it (A: nsub regions each).
__global__ __launch_bounds__(256) void k_sj_offsets(SjBuckets A, uint32_t nsub, SjBuckets S, uint32_t nb, int b2,
                                                    uint32_t *__restrict__ off, uint64_t *d_count, uint64_t cap,
                                                    uint32_t *flag) {
    __shared__ uint32_t s_w[4];
    __shared__ uint32_t s_before;
    if (threadIdx.x == 0) s_before = 0;
    __syncthreads();
    uint32_t before = 0;
    if (threadIdx.x < blockIdx.x)  // at most 256 first-split buckets
        for (uint32_t r = 0; r < nsub; ++r) before += A.count(threadIdx.x * nsub + r);
    before = wave_sum(before);
    if (lane_id() == 0 && before) atomicAdd(&s_before, before);
    const uint32_t per = b2 ? 1u << b2 : nb, f0 = blockIdx.x * per;  // per <= 256
    const uint32_t f = f0 + threadIdx.x;
    const uint32_t c = threadIdx.x < per && f < nb ? S.count(f) : 0u;
    const uint32_t ex = block_excl_scan256(c, s_w);
    __syncthreads();
    if (threadIdx.x < per && f < nb) {
        off[f] = s_before + ex;
        if (f == nb - 1) {
            off[nb] = s_before + ex + c;
            *d_count = s_before + ex + c;
            if (s_before + ex + c > cap) atomicOr(flag, kSjFull);
        }
    }
}

// Where a bucket's rows go.  Known: at off[f], when every tuple has a match.
// Chained: behind the rows of the buckets before it, by a look-back in ticket
// order.
struct SjKnown {
    uint32_t at;
    QO_DEV void begin(uint32_t) const {}
    struct Asked {};
    QO_DEV void ask(Asked &) const {}
    QO_DEV uint64_t position(uint32_t, Asked) const { return at; }
    QO_DEV void repeated() const {}  // the table build saw to that
};
struct SjChained {
    uint64_t *status;
    uint32_t f, nb;
    uint64_t *d_count;
    DevCtl *ctl;
    uint32_t *flag;
    QO_DEV void begin(uint32_t total) const {
        // Successors need not wait for the placement.
        if (threadIdx.x == 0) st_agent(&status[f], (f ? kFlagAgg : kFlagInc) | total);
    }
    struct Asked {};
    QO_DEV void ask(Asked &) const {}
    QO_DEV uint64_t position(uint32_t total, Asked) const {
        const uint64_t e = lookback(status, f, total, ctl, flag, kSjWait);
        if (f == nb - 1 && lane_id() == 0) *d_count = e + total;
        return e;
    }
    QO_DEV void repeated() const {}
};

// Bound by vector instructions and by the latency between its barriers, then by
// HBM (2^28 rows: 2.8 GB in 0.64 ms).  What was measured at that size: rows
// ranked within whole key runs (mean 8 rows, but a wave waits for its longest)
// 0.84 ms, 185 vector instructions per row; within (key, s_payload interval)
// bins 0.64 ms.  Work-groups of 1024 threads with ticket and look-back 1.04 ms.
template <bool DENSE, int NT, bool ALL>
__global__ __launch_bounds__(NT, 8) void k_sj_finish(SjBuckets S, SjBuckets R, uint32_t nb, int sh, KeySpan span,
                                                     PayloadBins pbins, const uint64_t *__restrict__ slots,
                                                     SoaEmit emit, uint32_t *flag, const uint32_t *__restrict__ off,
                                                     uint64_t *status, uint32_t *ticket, uint64_t *d_count,
                                                     DevCtl *ctl, SjGate gate) {
    __shared__ SjLds<DENSE, NT> s;
    // In the ALL form the flag and the bucket's place are three scalar loads in
    // flight together, and the tuples' loads wait for them only.
    const uint32_t fl = *flag;
    const uint32_t o0 = ALL ? off[blockIdx.x] : 0u, o1 = ALL ? off[blockIdx.x + 1] : 0u;
    if ((fl & (kSjOverflow | kSjFull)) || gate.off()) return;  // the whole grid
    if (!ALL && threadIdx.x == 0) s.tile = atomicAdd(ticket, 1u);
    sj_clear(s);
    __syncthreads();
    const uint32_t f = ALL ? blockIdx.x : s.tile;
    if (f >= nb) return;  // whole block; one block per bucket, so never taken
    const uint32_t n = ALL ? o1 - o0 : S.count(f);
    const uint32_t nr = DENSE ? 0u : R.count(f), base_d = f << sh;  // offset of the bucket's first key
    const uint64_t *src = S.bucket + (size_t)f * S.cap;
    const uint64_t *rsrc = DENSE ? nullptr : R.bucket + (size_t)f * R.cap;
    const uint64_t *slice = DENSE ? slots + base_d : nullptr;
    if (ALL)
        sj_bucket(s, src, n, rsrc, nr, slice, span.kmin + base_d, sh, pbins, emit, SjKnown{o0});
    else
        sj_bucket(s, src, n, rsrc, nr, slice, span.kmin + base_d, sh, pbins, emit,
                  SjChained{status, f, nb, d_count, ctl, flag});
}

// ---------------------------------------------------------------------------
// Host plan.
// ---------------------------------------------------------------------------
struct SjSide {            // one input's buckets
    uint64_t capA = 0;     // pairs per region of the first split (two splits only)
    uint64_t capB = 0;     // pairs per fine bucket
};
struct SjPlan {
    bool on = false, dense = false;
    bool all = false;      // every S tuple in the build range has a match
    int nt = 0;            // threads of the finishing work-groups
    KeySpan span{};
    PayloadBins pay{};
    int sh = 0, b2 = 0;    // bucket = offset >> sh; b2 > 0: two splits, first by offset >> (sh + b2)
    uint32_t nb = 0, nb1 = 0, parts1 = 0;
    SjSide s, r;
};

// Fewer S tuples than this are probed and sorted by the generic path, whose
// small sort is one launch.  At the line, 16383 S rows that way and 16384 this way,
// us: 64 build keys spread 157 and 113, dense 141 and 96; 4096 spread 233 and 112,
// dense 138 and 97.  (What breaks even lies below and was not looked for: those rows
// fewer keep the path they had.)
constexpr size_t kSjMinRows = size_t(1) << 14;
constexpr uint64_t kSjMaxBuckets = 1u << (2 * kSjPartBits);

// What the sample says about S: expected rows, and the most of them in an
// aligned interval of 2^shift key offsets.
struct SjSpread {
    const SjInfo &info;
    double rows, per, hot, span;  // per: tuples a sample stands for; hot: rows of the hottest key
    int bsh;                      // a bin of the sample covers 2^bsh offsets
    bool even;
    SjSpread(const SjInfo &in, uint32_t last, size_t ns) : info(in) {
        per = (double)ns / (double)std::min<size_t>(ns, kSjSamples);
        rows = std::min((double)ns, per * (in.pass + 4.0 * std::sqrt((double)in.pass)));
        // A key seen up to 6 times in the sample may be chance (or a collision); the
        // largest of many counts lies above its own mean.
        hot = in.hot <= 6 ? 0.0 : per * (in.hot - std::sqrt((double)in.hot));
        span = (double)last + 1.0;
        bsh = last < kSjBins ? 0 : 24 - __builtin_clz(last);
        // Even: no bin far above the mean of the bins in use, as far as the sample can tell.
        const double mean = (double)in.pass / ((last >> bsh) + 1);
        const uint32_t top = *std::max_element(in.bin, in.bin + kSjBins);
        even = top <= 1.5 * mean + 6.0 * std::sqrt(mean) + 4.0;
    }
    double expected() const { return per * info.pass; }
    double most(int shift) const {
        const double part = std::min(1.0, std::ldexp(1.0, shift) / span);
        if (even) return rows * part + hot;
        // Uneven: the fullest group of bins, or the fullest bin's share.
        const uint32_t group = shift > bsh ? 1u << std::min(8, shift - bsh) : 1u;
        uint32_t top = 0;
        for (uint32_t b = 0; b < kSjBins; b += group) {
            uint32_t c = 0;
            for (uint32_t u = 0; u < group; ++u) c += info.bin[b + u];
            top = std::max(top, c);
        }
        const double m = per * (top + 2.0 * std::sqrt((double)top));
        return shift >= bsh ? m : m * std::ldexp(1.0, shift - bsh) + hot;
    }
};

// A fine bucket has room for all the rows a work-group takes, so that a hot key of
// some thousand rows still fits; where fewer than 256 are expected in one (then S
// is small, and its sample shows such a key), for eight times those and 1024 beside
// the fullest one's (`top`).  `most`: rows expected in the fullest bucket of the
// first split.
static SjSide sj_side(const SjPlan &p, double most, double top, double mean, uint32_t limit) {
    SjSide o;
    o.capB = std::min<uint64_t>(limit, ((uint64_t)(top + 8.0 * mean) + 1024 + 31) / 32 * 32);
    if (p.b2) o.capA = ((uint64_t)(most / kXcdRegions * 1.25 + 8.0 * std::sqrt(most)) + kSplitTile + 31) / 32 * 32;
    return o;
}

// Buckets for work-groups of nt threads: the widest whose rows (and build
// keys) fit with room to spare, and narrow enough to give a small join a few
// work-groups per CU.
static bool sj_buckets(SjPlan &p, int nt, const SjSpread &s, size_t nr) {
    const double limit = (double)sj_items(p.dense, nt) * nt;
    const double want = std::min(0.75 * limit, std::max(512.0, s.rows / 512.0));
    p.nt = nt;
    p.sh = 0;
    while (p.sh < 31) {
        const double w = std::ldexp(1.0, p.sh + 1);
        if (s.rows * w / s.span > want || w / 2 >= s.span) break;  // 2^sh <= the smallest power of two >= span
        if (s.most(p.sh + 1) > 0.9 * limit) break;
        if (p.dense ? w > 2.0 * nt : (double)nr * w / s.span > 1.5 * nt) break;
        ++p.sh;
    }
    const uint64_t nb = ((uint64_t)p.span.last >> p.sh) + 1;
    // Of uneven keys no more buckets than a few per 1000 rows: most would be empty.
    // Even ones can need many for the build keys alone: a slice of the table each, or
    // (spread keys) their share of R, which is split as well.  Half of S selected,
    // this path and the generic one in us: 2^24 dense keys with 2^18 S rows 408, 396,
    // 2^20 418, 487; 2^20 spread keys with 2^14 rows 305, 333, 2^22 401, 366; 2^24
    // spread with 2^22 rows 876, 829, with 2^24 969, 1131.
    if (nb > kSjMaxBuckets || s.most(p.sh) > 0.9 * limit || (!s.even && nb > 1024 + s.rows / 256)) return false;
    if (p.dense ? (double)nb > 8192.0 + s.rows / 16.0 : (double)nr > 1048576.0 + 4.0 * s.rows) return false;
    p.nb = (uint32_t)nb;
    int bits = 0;
    while ((1u << bits) < p.nb) ++bits;
    p.b2 = bits <= kSjPartBits ? 0 : bits / 2;
    p.nb1 = ((p.nb - 1) >> p.b2) + 1;
    p.parts1 = 1;
    while (p.parts1 < p.nb1) p.parts1 *= 2;
    p.s = sj_side(p, s.most(p.sh + p.b2), s.most(p.sh), s.rows / p.nb, (uint32_t)limit);
    if (!p.dense) {
        const double even = (double)nr * std::min(1.0, std::ldexp(1.0, p.sh + p.b2) / s.span);
        p.r = sj_side(p, s.even ? even : std::min((double)nr, 4.0 * even), 0.0, (double)nr / p.nb, 2u * (uint32_t)nt);
    }
    return true;
}

static SjPlan sj_plan(const SjInfo &info, size_t nr, size_t ns, size_t out_capacity) {
    SjPlan p;
    if (info.dups || info.rmin > info.rmax || info.pass == 0) return p;
    const uint32_t last = (uint32_t)info.rmax - (uint32_t)info.rmin;
    const SjSpread s(info, last, ns);
    p.dense = info.mode == kJoinKeyRange;
    p.all = p.dense && (uint64_t)last + 1 == nr;  // distinct keys that fill their range
    // Outputs without room for every tuple in range may still hold the rows: only
    // the generic path counts them before any is written.
    if (!p.all && s.expected() > (double)out_capacity) return p;
    p.span = KeySpan{(uint32_t)info.rmin, last};
    p.pay = PayloadBins{~info.pmin, 32 - __builtin_clz((info.pmax - ~info.pmin) | 1u)};
    p.on = sj_buckets(p, 512, s, nr) || sj_buckets(p, 1024, s, nr);
    return p;
}

struct SjSideBufs {
    uint32_t *ctrA = nullptr, *ctrB = nullptr;
    uint64_t *a = nullptr, *b = nullptr;
};
struct SjBufs {
    uint64_t *res = nullptr;  // [0] rows, [1] overflow flag
    uint32_t *ticket = nullptr, *off = nullptr;
    uint64_t *status = nullptr;
    SjSideBufs s, r;
    size_t clear_words = 0;   // from res on: zeroed before the splits
};

static SjBufs sj_carve(const SjPlan &p, Carver &cv) {
    SjBufs b;
    const size_t fine = (size_t)p.nb1 << p.b2;
    b.res = cv.take<uint64_t>(2);
    const size_t from = cv.off - 16;
    b.ticket = cv.take<uint32_t>(1);
    b.status = cv.take<uint64_t>(p.nb);
    auto counters = [&](SjSideBufs &o) {
        o.ctrB = cv.take<uint32_t>(fine * kCtrStride);
        if (p.b2) o.ctrA = cv.take<uint32_t>((size_t)p.parts1 * kXcdRegions * kCtrStride);
    };
    counters(b.s);
    if (!p.dense) counters(b.r);
    b.clear_words = (cv.off - from) / 4;
    b.off = cv.take<uint32_t>(p.nb + 1);
    auto data = [&](SjSideBufs &o, const SjSide &side) {
        if (p.b2) o.a = cv.take<uint64_t>((size_t)p.nb1 * kXcdRegions * side.capA);
        o.b = cv.take<uint64_t>(fine * side.capB);
    };
    data(b.s, p.s);
    if (!p.dense) data(b.r, p.r);
    return b;
}

template <bool HAS_FILTER>
static int sj_split(const SjPlan &p, const SjSide &side, const SjSideBufs &b, uint32_t *flag, const int32_t *key,
                    const int32_t *pay, const int32_t *filt, size_t n, int32_t flo, int32_t fhi, const SjGate &gate,
                    hipStream_t st) {
    const bool vec = (((uintptr_t)key | (uintptr_t)pay | (HAS_FILTER ? (uintptr_t)filt : 0)) & 15u) == 0;
    const size_t tiles = (n + kSplitTile - 1) / kSplitTile;
    QO_REQUIRE(tiles < 0x7FFFFFFFull, "join input too large");
    const FlagOverflow ovf{flag};
    if (!p.b2) {
        k_sj_split1<HAS_FILTER><<<(unsigned)tiles, kSplitThreads, 0, st>>>(
            key, pay, filt, n, flo, fhi, vec, p.span, p.sh, p.parts1, b.b, FixedLayout{side.capB}, b.ctrB, ovf,
            gate);
        QO_LAUNCHED();
        return QO_OK;
    }
    k_sj_split1<HAS_FILTER><<<(unsigned)tiles, kSplitThreads, 0, st>>>(key, pay, filt, n, flo, fhi, vec, p.span,
                                                                      p.sh + p.b2, p.parts1, b.a, XcdLayout{side.capA},
                                                                      b.ctrA, ovf, gate);
    QO_LAUNCHED();
    const uint32_t tpr = (uint32_t)((side.capA + kSplitTile - 1) / kSplitTile);
    const uint64_t grid = (uint64_t)((p.nb1 + 7) / 8) * 8 * kXcdRegions * tpr;
    QO_REQUIRE(grid < 0x7FFFFFFFull, "join input too large");
    k_sj_split2<<<(unsigned)grid, kSplitThreads, 0, st>>>(b.a, side.capA, b.ctrA, p.nb1, tpr, p.span, p.sh, p.b2, b.b,
                                                          FixedLayout{side.capB}, b.ctrB, ovf, gate);
    QO_LAUNCHED();
    return QO_OK;
}

constexpr size_t kSjSampleWords = sizeof(SjInfo) / 4 + (size_t(1) << kSjHotBits);
// The stream's host words: the sample's counts, then the first words of the
// built table's header, then the result.
constexpr size_t kSjHostHeader = 2048, kSjHostResult = 3072;
static_assert(sizeof(SjInfo) <= kSjHostHeader && kSjHostResult + 16 <= kHostWordsBytes, "host words");
constexpr size_t kSjHeaderBytes = offsetof(JoinHeader, nr);

bool SortedJoin::wanted() const {
    return nr != 0 && ns >= kSjMinRows && ns < 0xFFFFFFFFull && tune_get(TUNE_JOIN_PART, ns).param == PART_AUTO;
}

size_t SortedJoin::sample_ws_bytes() { return kSjSampleWords * 4; }

int SortedJoin::sample(void *ws) {
    QO_TRY(host_words(st, &host));
    const JoinHeader *hdr = static_cast<const JoinHeader *>(table);
    SjInfo *d_info = static_cast<SjInfo *>(ws);
    uint32_t *d_keys = reinterpret_cast<uint32_t *>(d_info + 1);
    QO_TRY(launch_fill_u32(d_info, 0, kSjSampleWords, st));
    constexpr unsigned grid = kSjSamples / kSjSampleThreads;
    if (sfilt) k_sj_sample<true><<<grid, kSjSampleThreads, 0, st>>>(hdr, skey, spay, sfilt, ns, flo, fhi, d_info, d_keys);
    else k_sj_sample<false><<<grid, kSjSampleThreads, 0, st>>>(hdr, skey, spay, sfilt, ns, flo, fhi, d_info, d_keys);
    QO_LAUNCHED();
    QO_HIP(hipMemcpyAsync(host.ptr, d_info, sizeof(SjInfo), hipMemcpyDeviceToHost, st));
    QO_HIP(hipEventRecord(host.ev[0], st));
    return QO_OK;
}

int SortedJoin::built() {
    QO_HIP(hipMemcpyAsync(static_cast<char *>(host.ptr) + kSjHostHeader, table, kSjHeaderBytes, hipMemcpyDeviceToHost, st));
    QO_HIP(hipEventRecord(host.ev[1], st));
    return QO_OK;
}

int SortedJoin::run(bool table_known, uint64_t *rows, bool *done) {
    *done = false;
    QO_HIP(hipEventSynchronize(host.ev[0]));
    SjInfo info;
    memcpy(&info, host.ptr, sizeof(info));
    const SjPlan p = sj_plan(info, nr, ns, out_capacity);
    if (!p.on) return QO_OK;
    const JoinHeader *hdr = static_cast<const JoinHeader *>(table);
    const SjGate gate{hdr, info.mode};
    int status = QO_OK;
    Carver size(nullptr);
    sj_carve(p, size);
    void *ws = workspace(st, size.off + 256, &status);
    if (!ws) {  // no room for the buckets: the generic path may need less
        (void)hipGetLastError();
        return QO_OK;
    }
    Carver cv(ws);
    const SjBufs b = sj_carve(p, cv);
    uint32_t *flag = reinterpret_cast<uint32_t *>(b.res + 1);
    QO_TRY(launch_fill_u32(b.res, 0, b.clear_words, st));
    if (sfilt) QO_TRY(sj_split<true>(p, p.s, b.s, flag, skey, spay, sfilt, ns, flo, fhi, gate, st));
    else QO_TRY(sj_split<false>(p, p.s, b.s, flag, skey, spay, nullptr, ns, 0, 0, gate, st));
    if (!p.dense) QO_TRY(sj_split<false>(p, p.r, b.r, flag, rkey, rpay, nullptr, nr, 0, 0, gate, st));
    const SoaEmit out{okey, orpay, ospay, out_capacity};
    const SjBuckets sb{b.s.b, p.s.capB, b.s.ctrB}, rb{b.r.b, p.r.capB, b.r.ctrB};
    const uint64_t *slots = reinterpret_cast<const uint64_t *>(hdr + 1);
    if (p.all || ns > out_capacity) {
        k_sj_offsets<<<p.b2 ? p.nb1 : 1u, 256, 0, st>>>(SjBuckets{nullptr, p.s.capA, b.s.ctrA}, kXcdRegions, sb, p.nb,
                                                        p.b2, b.off, b.res, out_capacity, flag);
        QO_LAUNCHED();
    }
#define QO_SJ_FINISH(D, T, A)                                                                                       \
    k_sj_finish<D, T, A><<<p.nb, T, 0, st>>>(sb, rb, p.nb, p.sh, p.span, p.pay, slots, out, flag, b.off, b.status, b.ticket, \
                                             b.res, dev_ctl(), gate)
    if (p.all) {
        if (p.nt == 512) QO_SJ_FINISH(true, 512, true);
        else QO_SJ_FINISH(true, 1024, true);
    } else if (p.dense) {
        if (p.nt == 512) QO_SJ_FINISH(true, 512, false);
        else QO_SJ_FINISH(true, 1024, false);
    } else {
        if (p.nt == 512) QO_SJ_FINISH(false, 512, false);
        else QO_SJ_FINISH(false, 1024, false);
    }
#undef QO_SJ_FINISH
    QO_LAUNCHED();
    const uint64_t *res = reinterpret_cast<const uint64_t *>(static_cast<const char *>(host.ptr) + kSjHostResult);
    QO_HIP(hipMemcpyAsync(const_cast<uint64_t *>(res), b.res, 16, hipMemcpyDeviceToHost, st));
    if (!table_known) {
        // Off on the device too then, and the caller's probe is queued without a gap.
        QO_HIP(hipEventSynchronize(host.ev[1]));
        JoinHeader h;
        memcpy(&h, static_cast<const char *>(host.ptr) + kSjHostHeader, kSjHeaderBytes);
        if ((h.has_dups | h.sentinel_count | h.overflow) || h.mode != info.mode) return QO_OK;
    }
    QO_HIP(hipStreamSynchronize(st));
    // Nothing was written then.  kSjFull: the rows are too many if every tuple counted has a match.
    const uint32_t f = (uint32_t)res[1];
    if (f & kSjWait) {
        QO_TRY(check_device_error());
        return set_error(QO_ERR_DEVICE_WAIT, "a device-side wait of the join ran out of its bound");
    }
    if ((f & kSjOverflow) || (f && !p.all)) return QO_OK;
    *rows = res[0];
    *done = true;
    return QO_OK;
}

}  // namespace qo
