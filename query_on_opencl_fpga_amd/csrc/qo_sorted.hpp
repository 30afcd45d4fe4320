// Device work of the sorted join: one bucket of S tuples joined with its build
// keys in LDS and written in (key, s_payload) order, by one work-group.  Shared
// by the single sorted join and the batch.
#pragma once
#include "qo_internal.hpp"
#include "qo_join.hpp"
#include "qo_split.hpp"

namespace qo {

// Offset of a key in the build keys' span (monotone in the signed key).
struct KeySpan {
    uint32_t kmin, last;  // smallest build key, largest - smallest
    QO_DEV bool operator()(int32_t key, uint32_t &d) const {
        d = (uint32_t)key - kmin;
        return d <= last;
    }
};

struct FlagOverflow {
    uint32_t *flag;
    QO_DEV void operator()(uint64_t) const { *flag = 1u; }  // kSjOverflow
};

constexpr uint32_t kSjRankRun = 256;  // longest run whose rows are ranked one against another
// S tuples per thread: six, and for the larger work-groups, which take the joins
// with a hot key, as many as leave room for two of them per CU.
constexpr int sj_items(bool dense, int nt) { return nt <= 512 ? 6 : dense ? 8 : 7; }

// Interval of the s_payload's range, by which a build key's matches are
// counted: 2^sb intervals of [pmin, pmin + 2^bits), monotone in the s_payload
// (values outside the sampled range fall into the first or last one).
struct PayloadBins {
    uint32_t pmin;  // value ^ 2^31
    int bits;
    QO_DEV uint32_t operator()(uint32_t pay, int sb) const {
        const uint32_t x = pay ^ 0x80000000u;
        if (sb == 0 || x < pmin) return 0u;  // bits - sb < 32 from here on
        return min((x - pmin) >> (bits > sb ? bits - sb : 0), (1u << sb) - 1u);
    }
};

// A bucket's work-group has NT threads: at most kRows S tuples and kSlots
// build keys (dense: key slots), two per thread.  Rows are counted in kBins
// (build key, s_payload interval) bins, so that a run left to be ranked is a row
// or two long.  32 waves fill a CU: two work-groups of 1024 or four of 512, each
// 1024 threads with at most 80 KB of LDS.
template <bool DENSE, int NT>
struct SjLds {
    static constexpr int kItems = sj_items(DENSE, NT);
    static constexpr uint32_t kRows = (uint32_t)kItems * NT;
    static constexpr uint32_t kSlots = 2 * NT;
    static constexpr int kBinBits = __builtin_ctz(kSlots);  // bins of a sparse bucket's key interval
    static constexpr int kPer = (DENSE ? 8 : 4) / (NT <= 512 ? 1 : 2);
    static constexpr uint32_t kBins = (uint32_t)kPer * NT;
    uint32_t cnt[kBins + 1];  // matches per bin, then where its run starts
    uint32_t pay[kSlots];
    int32_t spay[kRows];
    uint16_t slot[kRows];  // build key << sb | s_payload interval
    uint64_t bits[DENSE ? kSlots / 64 : 1];       // dense: slots that hold a key
    uint32_t off[DENSE ? 1 : kSlots];             // sparse: key offsets of the build tuples, ascending
    uint32_t bin[DENSE ? 1 : kSlots + 1];         // sparse: where each bin's build tuples start
    uint32_t w[NT / kWave];
    uint64_t base;
    uint32_t tile, long_run;
};

struct SjBuckets {
    const uint64_t *bucket;
    uint64_t cap;
    const uint32_t *ctr;
    QO_DEV uint32_t count(uint32_t f) const {
        const uint64_t c = ctr[(size_t)f * kCtrStride];
        return (uint32_t)(c < cap ? c : cap);
    }
};

// Rows of the bucket (s.spay, s.slot; total of them) into (slot, s_payload)
// order by digit passes in place: every row is in registers before any is
// written back.  For buckets with a run too long to rank row against row; the
// run starts in s.cnt give way to the waves' digit counts.
template <bool DENSE, int NT>
QO_DEV void sj_sort_rows(SjLds<DENSE, NT> &s, uint32_t total, int sb) {
    constexpr int IT = SjLds<DENSE, NT>::kItems;
    constexpr int kWaves = NT / kWave;
    static_assert(kWaves * 256 * sizeof(uint16_t) <= sizeof(s.cnt), "digit counts");
    uint16_t(*cnt)[256] = reinterpret_cast<uint16_t(*)[256]>(s.cnt);
    const unsigned w = wave_id(), lane = lane_id();
    for (int pass = 0; pass < 6; ++pass) {  // 4 digits of the s_payload, 2 of the slot (11 bits)
        __syncthreads();
        for (int i = 0; i < 256 / kWave; ++i) cnt[w][i * kWave + lane] = 0;
        uint32_t x[IT], at[IT];  // at: order within the wave's digit | slot << 13 | digit << 24
        static_assert(SjLds<DENSE, NT>::kRows <= 1u << 13 && 2 * NT <= 1 << 11, "fields of at");
        wave_lockstep();
#pragma unroll
        for (int j = 0; j < IT; ++j) {
            const uint32_t i = (w * IT + j) * kWave + lane;
            const bool valid = i < total;
            x[j] = valid ? (uint32_t)s.spay[i] : 0u;
            const uint32_t l = valid ? (uint32_t)s.slot[i] >> sb : 0u;
            const uint32_t d = (pass < 4 ? (x[j] ^ 0x80000000u) >> (8 * pass) : l >> (8 * (pass - 4))) & 255u;
            const uint64_t m = match_digit(d, valid);
            const uint32_t pre = cnt[w][d], r = popc(m & lanemask_lt());
            wave_lockstep();  // every lane has read its digit's count before the leaders advance it
            if (valid && r == 0) cnt[w][d] = (uint16_t)(pre + popc(m));
            wave_lockstep();
            at[j] = (pre + r) | (l << 13) | (d << 24);
        }
        __syncthreads();
        uint32_t tot = 0;
        if (threadIdx.x < 256) {
#pragma unroll
            for (int i = 0; i < kWaves; ++i) {
                const uint32_t c = cnt[i][threadIdx.x];
                cnt[i][threadIdx.x] = (uint16_t)tot;
                tot += c;
            }
        }
        const uint32_t start = block_excl_scan<kWaves>(tot, s.w);
        if (threadIdx.x < 256)
#pragma unroll
            for (int i = 0; i < kWaves; ++i) cnt[i][threadIdx.x] = (uint16_t)(cnt[i][threadIdx.x] + start);
        __syncthreads();
#pragma unroll
        for (int j = 0; j < IT; ++j) {
            if ((w * IT + j) * kWave + lane >= total) continue;
            const uint32_t p = cnt[w][at[j] >> 24] + (at[j] & 0x1FFFu);
            s.spay[p] = (int32_t)x[j];
            s.slot[p] = (uint16_t)(((at[j] >> 13) & 0x7FFu) << sb);
        }
    }
}

// Exclusive scan of c[0, PER * NT) in place, PER entries per thread;
// c[PER * NT] := the total, which is returned.  Barriers before and after.
template <int NT, int PER>
QO_DEV uint32_t sj_scan(uint32_t *c, uint32_t *s_w) {
    __syncthreads();
    uint32_t v[PER], sum = 0;
#pragma unroll
    for (int u = 0; u < PER; ++u) {
        v[u] = c[PER * threadIdx.x + u];
        sum += v[u];
    }
    uint32_t at = block_excl_scan<NT / kWave>(sum, s_w);
#pragma unroll
    for (int u = 0; u < PER; ++u) {
        c[PER * threadIdx.x + u] = at;
        at += v[u];
    }
    if (threadIdx.x == NT - 1) c[PER * NT] = at;
    __syncthreads();
    return c[PER * NT];
}

// Clears the counters of sj_bucket; a barrier has to follow.
template <bool DENSE, int NT>
QO_DEV void sj_clear(SjLds<DENSE, NT> &s) {
    if (threadIdx.x == 0) s.long_run = 0;
#pragma unroll
    for (int u = 0; u < SjLds<DENSE, NT>::kPer; ++u) s.cnt[threadIdx.x + u * NT] = 0;
    if (!DENSE) {
        s.bin[threadIdx.x] = 0;
        s.bin[threadIdx.x + NT] = 0;
    }
}

// Joins and writes one bucket: n tuples at src, keys in [kbase, kbase + 2^sh).
// DENSE: `slots` is the bucket's slice of the key-range table (2^sh <= 2 NT
// slots); else nr <= 2 NT build tuples at rsrc.  `start` says where the rows go:
// begin(total) (every thread), ask() (first wave only; what position() may read
// ahead), position(total) (first wave only; the first row's
// output position) and, for build tuples, repeated() when two have one key.
// Called by all NT threads after sj_clear and a barrier.
template <bool DENSE, int NT, class Start>
QO_DEV void sj_bucket(SjLds<DENSE, NT> &s, const uint64_t *__restrict__ src, uint32_t n,
                      const uint64_t *__restrict__ rsrc, uint32_t nr, const uint64_t *__restrict__ slots, uint32_t kbase,
                      int sh, const PayloadBins &pbins, const SoaEmit &emit, const Start &start) {
    using Lds = SjLds<DENSE, NT>;
    constexpr int IT = SjLds<DENSE, NT>::kItems;
    // The build side's loads go first: its work then runs while the S tuples are
    // still on their way.
    const uint32_t nb = DENSE ? 1u << sh : nr;  // slots of the slice, or build tuples
    const uint64_t *bsrc = DENSE ? slots : rsrc;
    uint64_t bw[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const uint32_t i = (uint32_t)u * NT + threadIdx.x;
        bw[u] = i < nb ? ld_stream(bsrc + i) : kEmptySlot;
    }
    uint64_t v[IT];
#pragma unroll
    for (int j = 0; j < IT; ++j) {
        const uint32_t i = (uint32_t)j * NT + threadIdx.x;
        v[j] = i < n ? ld_stream(src + i) : 0ull;
    }
    int sb;  // log2 of the s_payload intervals per build key
    if (DENSE) {
        sb = __builtin_ctz(Lds::kBins) - sh;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const uint32_t i = (uint32_t)u * NT + threadIdx.x;
            s.pay[i] = (uint32_t)(bw[u] >> 32);
            const uint64_t m = ballot(bw[u] != kEmptySlot);
            if (lane_id() == 0) s.bits[i / kWave] = m;
        }
        __syncthreads();
    } else {
        // Build tuples of the bucket, ordered by key: counted by bin, placed bin
        // by bin, then ranked among their bin's.
        sb = 31 - __clz((int)(Lds::kBins / (nr ? nr : 1u)));
        const int bsh = sh > Lds::kBinBits ? sh - Lds::kBinBits : 0;
        uint32_t d[2], p[2], at[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const uint32_t i = (uint32_t)u * NT + threadIdx.x;
            d[u] = (uint32_t)bw[u] - kbase;
            p[u] = (uint32_t)(bw[u] >> 32);
            at[u] = i < nr ? atomicAdd(&s.bin[d[u] >> bsh], 1u) : 0u;
        }
        sj_scan<NT, 2>(s.bin, s.w);
#pragma unroll
        for (int u = 0; u < 2; ++u)
            if ((uint32_t)u * NT + threadIdx.x < nr) s.off[s.bin[d[u] >> bsh] + at[u]] = d[u];
        __syncthreads();
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            if ((uint32_t)u * NT + threadIdx.x >= nr) continue;
            const uint32_t b0 = s.bin[d[u] >> bsh], b1 = s.bin[(d[u] >> bsh) + 1];
            uint32_t before = 0;
            uint32_t same = 0;
            for (uint32_t i = b0; i < b1; ++i) {
                before += s.off[i] < d[u];
                same += s.off[i] == d[u];
            }
            if (same > 1) start.repeated();
            at[u] = b0 + before;
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            if ((uint32_t)u * NT + threadIdx.x >= nr) continue;
            s.off[at[u]] = d[u];
            s.pay[at[u]] = p[u];
        }
        __syncthreads();
    }
    // Lookup: rank of the tuple's build key in the bucket, and its arrival order
    // among that key's matches: slot | order << 16, or kMiss.
    constexpr uint32_t kMiss = ~0u;
    uint32_t pk[IT];
#pragma unroll
    for (int j = 0; j < IT; ++j) {
        pk[j] = kMiss;
        if ((uint32_t)j * NT + threadIdx.x >= n) continue;
        const uint32_t d = (uint32_t)v[j] - kbase;
        uint32_t l = kMiss;
        if (DENSE) {
            if ((s.bits[d / kWave] >> (d % kWave)) & 1u) l = d;
        } else {
            const int bsh = sh > Lds::kBinBits ? sh - Lds::kBinBits : 0;
            const uint32_t b1 = s.bin[(d >> bsh) + 1];
            for (uint32_t i = s.bin[d >> bsh]; i < b1; ++i)
                if (s.off[i] == d) l = i;
        }
        if (l != kMiss) {
            const uint32_t bin = (l << sb) | pbins((uint32_t)(v[j] >> 32), sb);
            const uint32_t order = atomicAdd(&s.cnt[bin], 1u);
            pk[j] = bin | (order << 16);
            if (order >= kSjRankRun) s.long_run = 1u;
        }
    }
    const uint32_t total = sj_scan<NT, Lds::kPer>(s.cnt, s.w);
    start.begin(total);
#pragma unroll
    for (int j = 0; j < IT; ++j) {
        if (pk[j] == kMiss) continue;
        const uint32_t l = pk[j] & 0xFFFFu, p = s.cnt[l] + (pk[j] >> 16);
        s.spay[p] = (int32_t)(v[j] >> 32);
        s.slot[p] = (uint16_t)l;
    }
    __syncthreads();
    typename Start::Asked asked;
    if (s.long_run) {  // block-uniform
        sj_sort_rows<DENSE, NT>(s, total, sb);
        if (threadIdx.x < kWave) start.ask(asked);
    } else {
        // Position i of the rows in bin order: its rank in its bin's run by
        // s_payload, four rows of the run per step (reads past the run's end stay
        // inside the struct).
        uint32_t dst[IT];  // final position | slot << 16
        int32_t x[IT];
#pragma unroll
        for (int j = 0; j < IT; ++j) {
            const uint32_t i = (uint32_t)j * NT + threadIdx.x;
            dst[j] = 0;
            if (i >= total) continue;
            const uint32_t l = s.slot[i];
            x[j] = s.spay[i];
            const uint32_t b0 = s.cnt[l], b1 = s.cnt[l + 1];
            uint32_t before = 0;
            for (uint32_t q = b0; q < b1; q += 4) {
                const int32_t y0 = s.spay[q], y1 = s.spay[q + 1], y2 = s.spay[q + 2], y3 = s.spay[q + 3];
                before += (y0 < x[j] || (y0 == x[j] && q < i)) ? 1u : 0u;
                before += (q + 1 < b1 && (y1 < x[j] || (y1 == x[j] && q + 1 < i))) ? 1u : 0u;
                before += (q + 2 < b1 && (y2 < x[j] || (y2 == x[j] && q + 2 < i))) ? 1u : 0u;
                before += (q + 3 < b1 && (y3 < x[j] || (y3 == x[j] && q + 3 < i))) ? 1u : 0u;
            }
            dst[j] = (b0 + before) | (l << 16);
        }
        if (threadIdx.x < kWave) start.ask(asked);  // on their way over the barrier and the move
        __syncthreads();
#pragma unroll
        for (int j = 0; j < IT; ++j) {
            if ((uint32_t)j * NT + threadIdx.x >= total) continue;
            s.spay[dst[j] & 0xFFFFu] = x[j];
            s.slot[dst[j] & 0xFFFFu] = (uint16_t)(dst[j] >> 16);
        }
    }
    if (threadIdx.x < kWave) {
        const uint64_t e = start.position(total, asked);
        if (threadIdx.x == 0) s.base = e;
    }
    __syncthreads();
    emit.template flush_rows<NT>(s.base, total, [&](uint32_t i, int32_t &k, int32_t &r, int32_t &p) {
        const uint32_t l = (uint32_t)s.slot[i] >> sb;
        k = (int32_t)(kbase + (DENSE ? l : s.off[DENSE ? 0 : l]));
        r = (int32_t)s.pay[l];
        p = s.spay[i];
    });
}

}  // namespace qo
