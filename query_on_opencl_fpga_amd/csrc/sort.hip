// Sorting: a stable LSD radix sort over 64-bit keys (8-bit digits) with an
// optional 32-bit value.  Every pass ranks a 4096-key tile with wave-level
// match masks (8 ballots per key), stages the tile in LDS in digit order and
// writes contiguous runs per digit.
//
// Every pass is reduce-then-scan: per-tile digit counts in tile-major rows
// (LDS atomics, one read of the keys), a column scan of the rows that turns
// them into the output offset of every (tile, digit), and the placement
// kernel, which reads its tile's 256 offsets as one coalesced row and walks
// the tiles in XCD-contiguous order.  A batch of many arrays (one per query)
// sorts in the same launches: a segment owns a contiguous tile range, the
// column scan restarts at every segment's first tile, and the digit starts of
// every pass per segment come from one histogram up front.  A segment's
// element count may live in device memory (written by an earlier kernel), so a
// whole batch can be captured in one graph without host round trips.
//
// Reference path replaced: radixSortImpl_sm (host/host/testSort.cpp:24-136)
// driving bitonicSortShared / bitonicMergeGlobal (kernel/aggregation/1/
// group_by_cu_op_dp.cl:89-291): O(log^2 N) in-place passes over the array.
// Here a Record sort is 4 passes over .y; ties keep input order (stable).
#include <algorithm>

#include "qo_device.hpp"
#include "qo_internal.hpp"
#include "qo_sort.hpp"

namespace qo {

// Digit of key k in the pass at `shift`: key bits [shift, shift + 8), or, with
// MOD (a split into `mod` partitions), bits [shift, shift + 8) of the
// partition id hi32(k) % mod, so that the passes order keys by partition id.
template <bool MOD>
QO_DEV uint32_t key_digit(uint64_t k, int shift, uint32_t mod) {
    if constexpr (MOD) return (((uint32_t)(k >> 32) % mod) >> shift) & 255u;
    else return (uint32_t)(k >> shift) & 255u;
}

// Index of the segment that owns global tile `tile` (0 for a single segment).
QO_DEV int seg_index_of(const RadixSeg *segs, int nseg, uint32_t tile) {
    if (nseg <= 1) return 0;
    int lo = 0, hi = nseg - 1;
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (segs[mid].tile0 <= tile) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

QO_DEV size_t seg_count(const RadixSeg &s) {
    size_t v = s.d_n ? (size_t)*s.d_n : s.cap;
    return v < s.cap ? v : s.cap;
}

// ---------------------------------------------------------------------------
// Reduce-then-scan passes for a single array.
// ---------------------------------------------------------------------------
constexpr int kHistTiles = 2;             // tiles per block of k_tile_hist
constexpr uint32_t kRowsBlocks = 512;     // at most this many column-scan blocks
constexpr uint32_t kRowsMinSpan = 64;     // tiles per column-scan block, at least
constexpr uint32_t kRowsOneBlock = 256;   // up to this many tiles, one block scans the rows
constexpr uint32_t kRowsFew = 64;         // up to this many, each placement block does
static_assert(kRowsFew / kHistTiles <= kWave, "a lane per histogram block");

// Digit counts of one tile (rem keys at src) into 256 LDS counters; `vec`:
// src is 16-byte aligned, so two keys are read per load.  Returns the bits of
// any key >> 32 that differ from `first`.
template <bool MOD = false>
QO_DEV uint32_t hist_tile(const uint64_t *__restrict__ src, uint32_t rem, int shift, uint32_t *s_row, bool vec,
                          uint32_t mod, uint32_t first) {
    uint32_t diff = 0;
    auto count = [&](uint64_t k) {
        atomicAdd(&s_row[key_digit<MOD>(k, shift, mod)], 1u);
        diff |= (uint32_t)(k >> 32) ^ first;
    };
    if (vec) {
        constexpr int PER = kSortTile / 512;
        uint4 q[PER];
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            const uint32_t v = j * 256 + threadIdx.x;
            q[j] = (2 * v + 2 <= rem) ? ld_stream(reinterpret_cast<const uint4 *>(src) + v) : uint4{0, 0, 0, 0};
        }
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            const uint32_t v = j * 256 + threadIdx.x;
            if (2 * v + 2 <= rem) {
                count(((uint64_t)q[j].y << 32) | q[j].x);
                count(((uint64_t)q[j].w << 32) | q[j].z);
            } else if (2 * v < rem) {
                count(src[2 * v]);
            }
        }
    } else {
        for (uint32_t i = threadIdx.x; i < rem; i += 256) count(src[i]);
    }
    return diff;
}

// rows[t * 256 + d] = keys of global tile t whose digit is d (zero rows for
// tiles past their segment's element count).  A single array passes its
// segment as seg0 with segs = null; a batch passes the segment list.  diffs
// (first pass of a sort with the digits found out on the device): one word per
// block, the bits of key >> 32 in which its keys differ from the array's first.
template <bool MOD = false, bool DYN = false>
__global__ __launch_bounds__(256) void k_tile_hist(const uint64_t *__restrict__ keys, RadixSeg seg0,
                                                   const RadixSeg *segs, int nseg, uint32_t ntile, int shift,
                                                   uint32_t *__restrict__ rows, const uint32_t *run_if = nullptr,
                                                   uint32_t mod = 0, const uint32_t *__restrict__ sel = nullptr,
                                                   const uint64_t *kalt = nullptr, uint32_t *diffs = nullptr) {
    if (run_if && *run_if == 0) return;  // gated off: runs only when *run_if != 0
    if (DYN && !diffs) {  // (the first pass finds the digits out and always counts)
        const uint32_t plan = radix_pass(*sel, shift);
        if (!(plan & kPassPlace)) return;
        if (plan >> 8) keys = kalt;
    }
    __shared__ uint32_t s_h[kHistTiles][256];
    __shared__ uint32_t s_diff;
    if (DYN && threadIdx.x == 0) s_diff = 0;
    for (int i = threadIdx.x; i < kHistTiles * 256; i += 256) (&s_h[0][0])[i] = 0;
    __syncthreads();
    const uint32_t t0 = blockIdx.x * kHistTiles;
#pragma unroll
    for (int tt = 0; tt < kHistTiles; ++tt) {
        const uint32_t t = t0 + tt;
        if (t >= ntile) break;
        const RadixSeg sg = segs ? segs[seg_index_of(segs, nseg, t)] : seg0;
        const size_t n = seg_count(sg);
        const size_t tb = (size_t)(t - sg.tile0) * kSortTile;
        if (tb >= n) continue;
        const uint64_t *src = keys + sg.base + tb;
        const uint32_t d = hist_tile<MOD>(src, (uint32_t)std::min<size_t>(kSortTile, n - tb), shift, s_h[tt],
                                          (reinterpret_cast<uintptr_t>(src) & 15) == 0, mod,
                                          DYN && diffs ? (uint32_t)(keys[sg.base] >> 32) : 0u);
        if (DYN && diffs) {
            uint32_t w = d;
#pragma unroll
            for (int o = kWave / 2; o > 0; o >>= 1) w |= __shfl_xor(w, o, kWave);
            if (lane_id() == 0 && w) atomicOr(&s_diff, w);
        }
    }
    __syncthreads();
    if (DYN && diffs && threadIdx.x == 0) diffs[blockIdx.x] = s_diff;
#pragma unroll
    for (int tt = 0; tt < kHistTiles; ++tt)
        if (t0 + tt < ntile) rows[(size_t)(t0 + tt) * 256 + threadIdx.x] = s_h[tt][threadIdx.x];
}

// Column-scan layout: block b of the scan owns tiles [b * span, (b + 1) * span).
struct RowsPlan {
    uint32_t span, nb;
};
static RowsPlan rows_plan(uint32_t ntile) {
    RowsPlan r;
    r.span = std::max(kRowsMinSpan, (ntile + kRowsBlocks - 1) / kRowsBlocks);
    r.nb = (ntile + r.span - 1) / r.span;
    return r;
}

// The three column-scan kernels are chains of loads by few threads, so what
// bounds them is the loads in flight: 32 per thread instead of 8, with the values
// kept in registers between summing and writing (1 M keys, one-block scan, four
// passes: 133 -> 120 us in all).  A whole group of 8 is loaded and stored without
// a look at each entry's bound: with one, the apply kernel took 5.75 us for 500
// tiles and 4.0 with groups of 8 alone.
constexpr uint32_t kRowsU = 32, kRowsG = 8;

// Sum of column entries [t, t + U) of `col` (entries 256 words apart) below t1,
// loaded together.
template <uint32_t U>
QO_DEV uint32_t rows_batch(const uint32_t *col, uint32_t t, uint32_t t1, uint32_t (&v)[U]) {
    uint32_t sum = 0;
#pragma unroll
    for (uint32_t g = 0; g < U; g += kRowsG) {
        if (t + g + kRowsG <= t1) {
#pragma unroll
            for (uint32_t u = g; u < g + kRowsG; ++u) v[u] = col[(size_t)(t + u) * 256];
        } else {
#pragma unroll
            for (uint32_t u = g; u < g + kRowsG; ++u) v[u] = t + u < t1 ? col[(size_t)(t + u) * 256] : 0u;
        }
    }
#pragma unroll
    for (uint32_t u = 0; u < U; ++u) sum += v[u];
    return sum;
}

// Entries [t, t + U) below t1 := run + the entries before each in v.
template <uint32_t U>
QO_DEV uint32_t rows_write(uint32_t *col, uint32_t t, uint32_t t1, const uint32_t (&v)[U], uint32_t run) {
#pragma unroll
    for (uint32_t g = 0; g < U; g += kRowsG) {
        if (t + g >= t1) break;
        const bool whole = t + g + kRowsG <= t1;
#pragma unroll
        for (uint32_t u = g; u < g + kRowsG; ++u) {
            if (whole || t + u < t1) col[(size_t)(t + u) * 256] = run;
            run += v[u];
        }
    }
    return run;
}

// bsum[b * 256 + d] = digit-d keys of the tiles of block b.
__global__ __launch_bounds__(256) void k_rows_reduce(const uint32_t *__restrict__ rows, uint32_t ntile, uint32_t span,
                                                     uint32_t *__restrict__ bsum,
                                                     const uint32_t *__restrict__ sel = nullptr, int shift = 0) {
    if (sel && !(radix_pass(*sel, shift) & kPassPlace)) return;
    const uint32_t t0 = blockIdx.x * span, t1 = std::min(ntile, t0 + span);
    uint32_t sum = 0, v[kRowsU];
    for (uint32_t t = t0; t < t1; t += kRowsU) sum += rows_batch(rows + threadIdx.x, t, t1, v);
    bsum[(size_t)blockIdx.x * 256 + threadIdx.x] = sum;
}

// One block of 1024 threads: bsum[b][d] := start of digit d in the output +
// digit-d keys of blocks before b (exclusive, in place).  Thread (q, d) with
// q = threadIdx / 256 handles quarter q of the blocks for digit d.  First pass
// of a sort with the digits found out on the device: *diff := the union of the
// ndiff words at `diffs`.
__global__ __launch_bounds__(1024) void k_rows_starts(uint32_t *bsum, uint32_t nb, const uint32_t *diffs = nullptr,
                                                      uint32_t ndiff = 0, uint32_t *diff = nullptr,
                                                      const uint32_t *__restrict__ sel = nullptr, int shift = 0) {
    if (sel && !(radix_pass(*sel, shift) & kPassPlace)) return;
    __shared__ uint32_t s_part[4][256];
    __shared__ uint32_t s_w[16];
    __shared__ uint32_t s_diff;
    if (diff) {
        if (threadIdx.x == 0) s_diff = 0;
        __syncthreads();
        uint32_t d = 0;
        for (uint32_t i = threadIdx.x; i < ndiff; i += 1024) d |= diffs[i];
        if (d) atomicOr(&s_diff, d);
        __syncthreads();
        if (threadIdx.x == 0) *diff = s_diff;
    }
    const uint32_t d = threadIdx.x & 255u, q = threadIdx.x >> 8;
    const uint32_t per = (nb + 3) / 4, b0 = std::min(nb, q * per), b1 = std::min(nb, b0 + per);
    uint32_t *col = bsum + d;
    auto scan = [&](auto &v, auto starts) {
        constexpr uint32_t U = sizeof(v) / 4;
        uint32_t sum = 0;
        for (uint32_t b = b0 + U; b < b1; b += U) sum += rows_batch(col, b, b1, v);
        sum += rows_batch(col, b0, b1, v);  // the first batch stays in registers
        uint32_t run = starts(sum);
        run = rows_write(col, b0, b1, v, run);
        for (uint32_t b = b0 + U; b < b1; b += U) {
            rows_batch(col, b, b1, v);
            run = rows_write(col, b, b1, v, run);
        }
    };
    auto starts = [&](uint32_t sum) {
        s_part[q][d] = sum;
        __syncthreads();
        const uint32_t p0 = s_part[0][d], p1 = s_part[1][d], p2 = s_part[2][d], p3 = s_part[3][d];
        // Threads 0..255 come first in the block, so their exclusive scan is the digit start.
        const uint32_t start = block_excl_scan<16>(q == 0 ? p0 + p1 + p2 + p3 : 0u, s_w);
        __syncthreads();
        if (q == 0) s_part[0][d] = start;
        __syncthreads();
        return s_part[0][d] + (q > 0 ? p0 : 0u) + (q > 1 ? p1 : 0u) + (q > 2 ? p2 : 0u);
    };
    if (per <= kRowsG) {  // block-uniform: few blocks
        uint32_t v[kRowsG];
        scan(v, starts);
    } else {
        uint32_t v[kRowsU];
        scan(v, starts);
    }
}

// rows[t][d] := output offset of the first digit-d key of tile t (in place).
__global__ __launch_bounds__(256) void k_rows_apply(uint32_t *__restrict__ rows, uint32_t ntile, uint32_t span,
                                                    const uint32_t *__restrict__ bsum,
                                                    const uint32_t *__restrict__ sel = nullptr, int shift = 0) {
    if (sel && !(radix_pass(*sel, shift) & kPassPlace)) return;
    const uint32_t t0 = blockIdx.x * span, t1 = std::min(ntile, t0 + span);
    uint32_t run = bsum[(size_t)blockIdx.x * 256 + threadIdx.x], v[kRowsU];
    for (uint32_t t = t0; t < t1; t += kRowsU) {
        rows_batch(rows + threadIdx.x, t, t1, v);
        run = rows_write(rows + threadIdx.x, t, t1, v, run);
    }
}

// ---- segmented column scan (a batch: one array per segment) ----
// Walks global tiles t0, t0 + 1, ... and tells which of them start a segment.
struct SegWalk {
    const RadixSeg *segs;
    int nseg, si;
    QO_DEV SegWalk(const RadixSeg *s, int n, uint32_t t0) : segs(s), nseg(n), si(seg_index_of(s, n, t0)) {}
    QO_DEV bool starts(uint32_t t) {
        while (si + 1 < nseg && segs[si + 1].tile0 <= t) ++si;
        return segs[si].tile0 == t;
    }
};

// bsum[b][d] = digit-d keys of block b's tiles after the last segment start
// inside the block (all of them when none starts there); bflag[b] = a segment
// starts inside the block.
__global__ __launch_bounds__(256) void k_rows_reduce_seg(const uint32_t *__restrict__ rows, uint32_t ntile,
                                                         uint32_t span, const RadixSeg *segs, int nseg,
                                                         uint32_t *__restrict__ bsum, uint32_t *__restrict__ bflag,
                                                         const uint32_t *run_if = nullptr) {
    if (run_if && *run_if == 0) return;  // gated off: runs only when *run_if != 0
    const uint32_t t0 = blockIdx.x * span, t1 = std::min(ntile, t0 + span);
    const uint32_t *col = rows + threadIdx.x;
    SegWalk wk(segs, nseg, t0);
    uint32_t tail = 0, flag = 0;
    for (uint32_t t = t0; t < t1; ++t) {
        if (wk.starts(t)) {
            tail = 0;
            flag = 1;
        }
        tail += col[(size_t)t * 256];
    }
    bsum[(size_t)blockIdx.x * 256 + threadIdx.x] = tail;
    if (threadIdx.x == 0) bflag[blockIdx.x] = flag;
}

// One block of 1024 threads: bsum[b][d] := digit-d keys of the blocks before b
// back to the start of b's first segment (exclusive carry, in place).  Thread
// (q, d) walks quarter q of the blocks; the quarters' (flag, sum) pairs combine
// in order.
__global__ __launch_bounds__(1024) void k_rows_starts_seg(uint32_t *bsum, const uint32_t *bflag, uint32_t nb,
                                                          const uint32_t *run_if = nullptr) {
    if (run_if && *run_if == 0) return;  // gated off: runs only when *run_if != 0
    __shared__ uint32_t s_part[4][256];
    __shared__ uint32_t s_flag[4];
    const uint32_t d = threadIdx.x & 255u, q = threadIdx.x >> 8;
    const uint32_t per = (nb + 3) / 4, b0 = std::min(nb, q * per), b1 = std::min(nb, b0 + per);
    uint32_t *col = bsum + d;
    uint32_t agg = 0, f = 0;
    for (uint32_t b = b0; b < b1; ++b) {
        const uint32_t v = col[(size_t)b * 256];
        if (bflag[b]) {
            agg = v;
            f = 1;
        } else {
            agg += v;
        }
    }
    s_part[q][d] = agg;
    if (d == 0) s_flag[q] = f;
    __syncthreads();
    uint32_t c = 0;
    for (uint32_t qq = 0; qq < q; ++qq) c = s_flag[qq] ? s_part[qq][d] : c + s_part[qq][d];
    for (uint32_t b = b0; b < b1; ++b) {
        const uint32_t v = col[(size_t)b * 256];
        col[(size_t)b * 256] = c;
        c = bflag[b] ? v : c + v;
    }
}

// rows[t][d] := digit-d keys of the tiles of t's segment before t (in place).
__global__ __launch_bounds__(256) void k_rows_apply_seg(uint32_t *__restrict__ rows, uint32_t ntile, uint32_t span,
                                                        const RadixSeg *segs, int nseg,
                                                        const uint32_t *__restrict__ bsum,
                                                        const uint32_t *run_if = nullptr) {
    if (run_if && *run_if == 0) return;  // gated off: runs only when *run_if != 0
    const uint32_t t0 = blockIdx.x * span, t1 = std::min(ntile, t0 + span);
    uint32_t *col = rows + threadIdx.x;
    SegWalk wk(segs, nseg, t0);
    uint32_t run = bsum[(size_t)blockIdx.x * 256 + threadIdx.x];
    for (uint32_t t = t0; t < t1; ++t) {
        if (wk.starts(t)) run = 0;
        const uint32_t v = col[(size_t)t * 256];
        col[(size_t)t * 256] = run;
        run += v;
    }
}

// Places global tile xcd_tile(blockIdx.x): ranks its keys by digit (stable),
// stages them in LDS in digit order and writes each digit's run at the offset
// from its row (plus, for a batch, the digit's start in the segment's output).
//
// Without values four blocks fit a CU's LDS, so the registers are held to 128
// (two spilled): 2^26 keys 246 -> 226 us per pass.
//
// DYN: *sel picks the pass (radix_pass).  FEW: at most kRowsFew tiles,
// whose offsets the block works out from the counts itself instead of a scan
// launch (100,000 keys in four passes 84 -> 76 us); the first pass then unites the
// histogram's `diffs` too.
template <bool HAS_VAL, bool UNPACK = false, bool MOD = false, bool DYN = false, bool FEW = false>
__global__ __launch_bounds__(256, HAS_VAL || FEW ? 2 : 4) void k_radix_place(const uint64_t *__restrict__ kin, const uint32_t *__restrict__ vin,
                                                     uint64_t *__restrict__ kout, uint32_t *__restrict__ vout,
                                                     RadixSeg seg0, const RadixSeg *segs, int nseg, uint32_t ntile,
                                                     int shift, const uint32_t *__restrict__ offs,
                                                     const uint32_t *__restrict__ dstart, uint32_t sstride,
                                                     RowOut out0 = RowOut{}, const RowOut *outs = nullptr,
                                                     const uint32_t *run_if = nullptr, uint32_t mod = 0,
                                                     const uint32_t *__restrict__ sel = nullptr,
                                                     const uint32_t *diffs = nullptr, uint32_t ndiff = 0,
                                                     uint32_t *diff = nullptr) {
    if (run_if && *run_if == 0) return;  // gated off: runs only when *run_if != 0
    uint32_t plan = kPassPlace;
    if (DYN) {
        if (FEW && diffs) {  // first pass: ndiff <= 64 words
            uint32_t d = lane_id() < ndiff ? diffs[lane_id()] : 0u;
#pragma unroll
            for (int o = kWave / 2; o > 0; o >>= 1) d |= __shfl_xor(d, o, kWave);
            if (blockIdx.x == 0 && threadIdx.x == 0) *diff = d;  // for the later passes
            plan = radix_pass(d, shift);
        } else {
            plan = radix_pass(*sel, shift);
        }
        if ((plan & 255u) == 0) return;
        if (plan >> 8) {  // the keys lie in kout: the pass goes the other way
            const uint64_t *const t = kin;
            kin = kout;
            kout = const_cast<uint64_t *>(t);
        }
    }
    __shared__ uint32_t s_cnt[4][256];
    __shared__ uint32_t s_dpre[256];
    __shared__ uint32_t s_gofs[256];
    __shared__ uint32_t s_w[4];
    __shared__ uint64_t s_k[kSortTile];
    __shared__ uint32_t s_v[HAS_VAL ? kSortTile : 1];
    const uint32_t t = xcd_tile(blockIdx.x, ntile);
    const int si = segs ? seg_index_of(segs, nseg, t) : 0;
    const RadixSeg sg = segs ? segs[si] : seg0;
    const size_t n = seg_count(sg);
    const size_t tb = (size_t)(t - sg.tile0) * kSortTile;
    if (tb >= n) return;
    const uint32_t rem = (uint32_t)std::min<size_t>(kSortTile, n - tb);
    const uint64_t *ks = kin + sg.base + tb;
    if (DYN && (plan & kPassCopy)) {
        uint64_t *to = kout + sg.base + tb;
        uint64_t c[kSortItems];
#pragma unroll
        for (int j = 0; j < kSortItems; ++j) {
            const uint32_t i = (uint32_t)j * 256 + threadIdx.x;
            c[j] = i < rem ? ks[i] : 0ull;
        }
#pragma unroll
        for (int j = 0; j < kSortItems; ++j) {
            const uint32_t i = (uint32_t)j * 256 + threadIdx.x;
            if (i < rem) to[i] = c[j];
        }
        return;
    }
    const uint32_t *vs = HAS_VAL ? vin + sg.base + tb : nullptr;
    for (int i = threadIdx.x; i < 1024; i += 256) (&s_cnt[0][0])[i] = 0;
    __syncthreads();
    const unsigned w = wave_id(), lane = lane_id();
    const uint32_t wb = w * (kSortTile / 4);
    uint64_t k[kSortItems];
    uint32_t v[kSortItems];
    uint32_t rank[kSortItems];
#pragma unroll
    for (int j = 0; j < kSortItems; ++j) {
        const uint32_t idx = wb + j * kWave + lane;
        const bool valid = idx < rem;
        k[j] = valid ? ks[idx] : ~uint64_t(0);
        if (HAS_VAL) v[j] = valid ? vs[idx] : 0u;
    }
#pragma unroll
    for (int j = 0; j < kSortItems; ++j) {
        const uint32_t idx = wb + j * kWave + lane;
        const bool valid = idx < rem;
        const uint32_t d = key_digit<MOD>(k[j], shift, mod);
        const uint64_t m = match_digit(d, valid);
        const uint32_t pre = s_cnt[w][d];
        const uint32_t r = popc(m & lanemask_lt());
        wave_lockstep();  // every lane has read its digit's count before the leaders advance it
        if (valid && r == 0) s_cnt[w][d] = pre + popc(m);
        rank[j] = pre + r;
    }
    __syncthreads();
    {
        const unsigned d = threadIdx.x;
        const uint32_t c0 = s_cnt[0][d], c1 = s_cnt[1][d], c2 = s_cnt[2][d], c3 = s_cnt[3][d];
        if (FEW) {
            // Keys of digit d in the tiles before this one, and in all of them.
            uint32_t pre = 0, tot = 0;
#pragma unroll 16
            for (uint32_t u = 0; u < ntile; ++u) {
                const uint32_t c = offs[(size_t)u * 256 + d];
                pre += u < t ? c : 0u;
                tot += c;
            }
            const uint32_t start = block_excl_scan256(tot, s_w);
            __syncthreads();  // s_w is reused below
            s_gofs[d] = start + pre;
        } else {
            s_gofs[d] = offs[(size_t)t * 256 + d] + (dstart ? dstart[(size_t)si * sstride + d] : 0u);
        }
        s_dpre[d] = block_excl_scan256(c0 + c1 + c2 + c3, s_w);
        s_cnt[0][d] = 0;
        s_cnt[1][d] = c0;
        s_cnt[2][d] = c0 + c1;
        s_cnt[3][d] = c0 + c1 + c2;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kSortItems; ++j) {
        const uint32_t idx = wb + j * kWave + lane;
        if (idx < rem) {
            const uint32_t d = key_digit<MOD>(k[j], shift, mod);
            const uint32_t p = s_dpre[d] + s_cnt[w][d] + rank[j];
            s_k[p] = k[j];
            if (HAS_VAL) s_v[p] = v[j];
        }
    }
    __syncthreads();
    if constexpr (UNPACK) {
        // Last pass of a join-row sort: the segment's output columns.
        const RowOut o = outs ? outs[si] : out0;
        for (uint32_t i = threadIdx.x; i < rem; i += 256) {
            const uint64_t kk = s_k[i];
            const uint32_t d = key_digit<MOD>(kk, shift, mod);
            const uint32_t gp = s_gofs[d] + (i - s_dpre[d]);
            o.key[gp] = join_sort_key_key(kk);
            o.spay[gp] = join_sort_key_spay(kk);
            o.rpay[gp] = (int32_t)s_v[i];
        }
        return;
    }
    uint64_t *kd = kout + sg.base;
    uint32_t *vd = HAS_VAL ? vout + sg.base : nullptr;
    for (uint32_t i = threadIdx.x; i < rem; i += 256) {
        const uint64_t kk = s_k[i];
        const uint32_t d = key_digit<MOD>(kk, shift, mod);
        const uint32_t gp = s_gofs[d] + (i - s_dpre[d]);
        kd[gp] = kk;
        if (HAS_VAL) vd[gp] = s_v[i];
    }
}

// Workspace of the reduce-then-scan passes over `tiles` tiles.
struct RowsBufs {
    uint32_t *rows, *bsum;
    uint32_t *diff = nullptr;  // sorts with the digits found out on the device
};
static RowsBufs rows_carve(uint32_t tiles, Carver &cv) {
    RowsBufs b;
    b.rows = cv.take<uint32_t>((size_t)tiles * 256);
    // rows_plan(t).nb <= min(kRowsBlocks, ceil(t / kRowsMinSpan)) for every t <= tiles.
    b.bsum = cv.take<uint32_t>((size_t)std::min(kRowsBlocks, (tiles + kRowsMinSpan - 1) / kRowsMinSpan) * 256);
    return b;
}

static int launch_radix_rows(uint64_t *keys, uint32_t *vals, uint64_t *kalt, uint32_t *valt, const RadixSeg &sg,
                             int lo_bit, int hi_bit, const RowsBufs &b, hipStream_t st, bool *in_alt,
                             const RowOut *unpack = nullptr) {
    *in_alt = false;
    QO_REQUIRE(lo_bit >= 0 && hi_bit <= 64 && lo_bit < hi_bit, "bad bit range");
    if (sg.ntile == 0) return QO_OK;
    const RowsPlan rp = rows_plan(sg.ntile);
    const unsigned hblocks = (sg.ntile + kHistTiles - 1) / kHistTiles;
    uint64_t *ksrc = keys, *kdst = kalt;
    uint32_t *vsrc = vals, *vdst = valt;
    for (int sh = lo_bit; sh < hi_bit; sh += 8) {
        k_tile_hist<<<hblocks, 256, 0, st>>>(ksrc, sg, nullptr, 1, sg.ntile, sh, b.rows);
        QO_LAUNCHED();
        if (sg.ntile <= kRowsOneBlock) {
            // Few tiles: one block scans the rows themselves (one launch, not three).
            k_rows_starts<<<1, 1024, 0, st>>>(b.rows, sg.ntile);
            QO_LAUNCHED();
        } else {
            k_rows_reduce<<<rp.nb, 256, 0, st>>>(b.rows, sg.ntile, rp.span, b.bsum);
            QO_LAUNCHED();
            k_rows_starts<<<1, 1024, 0, st>>>(b.bsum, rp.nb);
            QO_LAUNCHED();
            k_rows_apply<<<rp.nb, 256, 0, st>>>(b.rows, sg.ntile, rp.span, b.bsum);
            QO_LAUNCHED();
        }
        if (vals && unpack && sh + 8 >= hi_bit)
            k_radix_place<true, true><<<sg.ntile, 256, 0, st>>>(ksrc, vsrc, kdst, vdst, sg, nullptr, 1, sg.ntile, sh,
                                                                 b.rows, nullptr, 0, *unpack, nullptr);
        else if (vals)
            k_radix_place<true><<<sg.ntile, 256, 0, st>>>(ksrc, vsrc, kdst, vdst, sg, nullptr, 1, sg.ntile, sh,
                                                           b.rows, nullptr, 0);
        else
            k_radix_place<false><<<sg.ntile, 256, 0, st>>>(ksrc, nullptr, kdst, nullptr, sg, nullptr, 1, sg.ntile,
                                                            sh, b.rows, nullptr, 0);
        QO_LAUNCHED();
        std::swap(ksrc, kdst);
        std::swap(vsrc, vdst);
        *in_alt = !*in_alt;
    }
    return QO_OK;
}

// Digits in which all keys agree cost a sort by the high 32 bits nothing: 2^26
// keys below 100 1.88 -> 0.72 ms, below 10,000 1.89 -> 0.98, below 10^6 1.76 ->
// 1.44; keys over all 32 bits 1.78 -> 1.71.
//
// The passes of a sort by the high 32 bits with the digits found out on the
// device (see radix_pass).  `diff`: a word and one per histogram block.
static int launch_radix_rows_dyn(uint64_t *keys, uint64_t *kalt, const RadixSeg &sg, const RowsBufs &b, uint32_t *diff,
                                 hipStream_t st) {
    if (sg.ntile == 0) return QO_OK;
    const RowsPlan rp = rows_plan(sg.ntile);
    const unsigned hblocks = (sg.ntile + kHistTiles - 1) / kHistTiles;
    uint32_t *diffs = diff + 1;  // one word per histogram block
    for (int sh = 32; sh < 64; sh += 8) {
        const bool first = sh == 32;
        const uint32_t *from = first ? diffs : nullptr;
        uint32_t *to = first ? diff : nullptr;
        const uint32_t *sel = first ? nullptr : diff;  // later column scans are skipped with their pass
        k_tile_hist<false, true><<<hblocks, 256, 0, st>>>(keys, sg, nullptr, 1, sg.ntile, sh, b.rows, nullptr, 0,
                                                          diff, kalt, first ? diffs : nullptr);
        QO_LAUNCHED();
        if (sg.ntile <= kRowsFew) {
            k_radix_place<false, false, false, true, true><<<sg.ntile, 256, 0, st>>>(
                keys, nullptr, kalt, nullptr, sg, nullptr, 1, sg.ntile, sh, b.rows, nullptr, 0, RowOut{}, nullptr, nullptr,
                0, diff, from, hblocks, to);
            QO_LAUNCHED();
            continue;
        }
        if (sg.ntile <= kRowsOneBlock) {
            k_rows_starts<<<1, 1024, 0, st>>>(b.rows, sg.ntile, from, hblocks, to, sel, sh);
            QO_LAUNCHED();
        } else {
            k_rows_reduce<<<rp.nb, 256, 0, st>>>(b.rows, sg.ntile, rp.span, b.bsum, sel, sh);
            QO_LAUNCHED();
            k_rows_starts<<<1, 1024, 0, st>>>(b.bsum, rp.nb, from, hblocks, to, sel, sh);
            QO_LAUNCHED();
            k_rows_apply<<<rp.nb, 256, 0, st>>>(b.rows, sg.ntile, rp.span, b.bsum, diff, sh);
            QO_LAUNCHED();
        }
        k_radix_place<false, false, false, true><<<sg.ntile, 256, 0, st>>>(keys, nullptr, kalt, nullptr, sg, nullptr, 1,
                                                                            sg.ntile, sh, b.rows, nullptr, 0, RowOut{},
                                                                            nullptr, nullptr, 0, diff);
        QO_LAUNCHED();
    }
    return QO_OK;
}

// ---------------------------------------------------------------------------
// A batch of arrays (one per query) in the same launches: the digit starts of
// every pass per segment come from one histogram over the keys up front
// (chunks of kSweepChunkTiles tiles); each pass then takes the tile
// histogram, a segmented column scan and the placement above.
// ---------------------------------------------------------------------------
constexpr int kSweepMaxPass = 8;

// Segmented digit counts: block c counts tiles [t0, t1) of segment `seg` of
// chunk c (segment-local tile numbers), one row of npass*256 per chunk.
__global__ __launch_bounds__(256) void k_sweep_counts_seg(const uint64_t *__restrict__ keys, const RadixSeg *segs,
                                                          const SweepChunk *chunks, int lo_bit, int npass,
                                                          uint32_t *partial, const uint32_t *run_if = nullptr) {
    if (run_if && *run_if == 0) return;  // gated off: runs only when *run_if != 0
    __shared__ uint32_t s_h[kSweepMaxPass * 256];
    for (int i = threadIdx.x; i < npass * 256; i += 256) s_h[i] = 0;
    __syncthreads();
    const SweepChunk ch = chunks[blockIdx.x];
    const RadixSeg sg = segs[ch.seg];
    const size_t n = seg_count(sg);
    const size_t e1 = std::min<size_t>((size_t)ch.t1 * kSortTile, n);
    for (size_t i = (size_t)ch.t0 * kSortTile + threadIdx.x; i < e1; i += 256) {
        const uint64_t k = ld_stream(keys + sg.base + i);
        for (int p = 0; p < npass; ++p) atomicAdd(&s_h[p * 256 + ((k >> (lo_bit + 8 * p)) & 255u)], 1u);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < npass * 256; i += 256) partial[(size_t)blockIdx.x * npass * 256 + i] = s_h[i];
}

// Per segment and pass: exclusive digit starts from the segment's chunk rows
// [chunk0[s], chunk0[s + 1]).  Block b = s * npass + p.
__global__ __launch_bounds__(256) void k_sweep_starts_seg(const uint32_t *partial, const uint32_t *chunk0, int npass,
                                                          uint32_t *starts, const uint32_t *run_if = nullptr) {
    if (run_if && *run_if == 0) return;  // gated off: runs only when *run_if != 0
    __shared__ uint32_t s_w[4];
    const int s = blockIdx.x / npass, p = blockIdx.x % npass;
    uint32_t c = 0;
    for (uint32_t r = chunk0[s]; r < chunk0[s + 1]; ++r) c += partial[(size_t)r * npass * 256 + p * 256 + threadIdx.x];
    starts[(size_t)blockIdx.x * 256 + threadIdx.x] = block_excl_scan256(c, s_w);
}

static uint32_t radix_tiles(size_t n) { return (uint32_t)((n + kSortTile - 1) / kSortTile); }

// Workspace of launch_radix_rows_segments (same order as its carve-up).
size_t radix_rows_seg_bytes(uint32_t total_tiles, int nseg, uint32_t nchunks) {
    Carver cv(nullptr);
    cv.take<uint32_t>((size_t)nchunks * kSweepMaxPass * 256);
    cv.take<uint32_t>((size_t)nseg * kSweepMaxPass * 256);
    cv.take<uint32_t>((size_t)total_tiles * 256);
    const uint32_t nbmax = std::min(kRowsBlocks, (total_tiles + kRowsMinSpan - 1) / kRowsMinSpan);
    cv.take<uint32_t>((size_t)nbmax * 256);
    cv.take<uint32_t>(nbmax);
    return cv.off + 256;
}

int launch_radix_rows_segments(uint64_t *keys, uint32_t *vals, uint64_t *kalt, uint32_t *valt,
                               const RadixSeg *d_segs, int nseg, uint32_t total_tiles, const SweepChunk *d_chunks,
                               uint32_t nchunks, const uint32_t *d_chunk0, int lo_bit, int hi_bit, void *ws,
                               hipStream_t st, bool *in_alt, const RowOut *d_outs, const uint32_t *run_if) {
    *in_alt = false;
    if (total_tiles == 0 || nchunks == 0) return QO_OK;
    QO_REQUIRE(!d_outs || vals, "unpacked output needs values");
    const int npass = (hi_bit - lo_bit + 7) / 8;
    QO_REQUIRE(npass >= 1 && npass <= kSweepMaxPass && lo_bit >= 0 && hi_bit <= 64, "bad bit range");
    QO_REQUIRE(nseg >= 1 && (size_t)nseg * npass < 0x7FFFFFFFull, "bad segment count");
    QO_REQUIRE((size_t)total_tiles * 256 < 0xFFFFFFFFull, "sort input too large");
    Carver cv(ws);
    uint32_t *partial = cv.take<uint32_t>((size_t)nchunks * npass * 256);
    uint32_t *starts = cv.take<uint32_t>((size_t)nseg * npass * 256);
    uint32_t *rows = cv.take<uint32_t>((size_t)total_tiles * 256);
    const RowsPlan rp = rows_plan(total_tiles);
    uint32_t *bsum = cv.take<uint32_t>((size_t)rp.nb * 256);
    uint32_t *bflag = cv.take<uint32_t>(rp.nb);
    // Digit starts of every pass per segment, from one read of the keys.
    k_sweep_counts_seg<<<nchunks, 256, 0, st>>>(keys, d_segs, d_chunks, lo_bit, npass, partial, run_if);
    QO_LAUNCHED();
    k_sweep_starts_seg<<<(unsigned)(nseg * npass), 256, 0, st>>>(partial, d_chunk0, npass, starts, run_if);
    QO_LAUNCHED();
    const RadixSeg none{0, 0, nullptr, 0, 0};
    const unsigned hblocks = (total_tiles + kHistTiles - 1) / kHistTiles;
    uint64_t *ksrc = keys, *kdst = kalt;
    uint32_t *vsrc = vals, *vdst = valt;
    for (int p = 0; p < npass; ++p) {
        const int sh = lo_bit + 8 * p;
        k_tile_hist<<<hblocks, 256, 0, st>>>(ksrc, none, d_segs, nseg, total_tiles, sh, rows, run_if);
        QO_LAUNCHED();
        k_rows_reduce_seg<<<rp.nb, 256, 0, st>>>(rows, total_tiles, rp.span, d_segs, nseg, bsum, bflag, run_if);
        QO_LAUNCHED();
        k_rows_starts_seg<<<1, 1024, 0, st>>>(bsum, bflag, rp.nb, run_if);
        QO_LAUNCHED();
        k_rows_apply_seg<<<rp.nb, 256, 0, st>>>(rows, total_tiles, rp.span, d_segs, nseg, bsum, run_if);
        QO_LAUNCHED();
        if (vals && d_outs && p == npass - 1)
            k_radix_place<true, true><<<total_tiles, 256, 0, st>>>(ksrc, vsrc, kdst, vdst, none, d_segs, nseg,
                                                                   total_tiles, sh, rows, starts + p * 256,
                                                                   (uint32_t)npass * 256, RowOut{}, d_outs, run_if);
        else if (vals)
            k_radix_place<true><<<total_tiles, 256, 0, st>>>(ksrc, vsrc, kdst, vdst, none, d_segs, nseg, total_tiles,
                                                             sh, rows, starts + p * 256, (uint32_t)npass * 256,
                                                             RowOut{}, nullptr, run_if);
        else
            k_radix_place<false><<<total_tiles, 256, 0, st>>>(ksrc, nullptr, kdst, nullptr, none, d_segs, nseg,
                                                              total_tiles, sh, rows, starts + p * 256,
                                                              (uint32_t)npass * 256, RowOut{}, nullptr, run_if);
        QO_LAUNCHED();
        std::swap(ksrc, kdst);
        std::swap(vsrc, vdst);
        *in_alt = !*in_alt;
    }
    return QO_OK;
}

// Long runs that are sorted by work-groups; more send all rows through the
// full-width sort.  A run takes its work-group 35 to 40 us whatever its length and
// two fit a CU, so 512 run at once; the full width costs 75 us (10,000 to 100,000
// rows), 100 (1 M) or 330 (10 M).  By work-groups, full width, in us: 100,000 rows
// with 500 long runs 185, 231, with 1428 252, 227; 1 M with 1000 272, 286, with
// 5000 569, 286; 10 M with 1667 882, 879, with 10,000 1400, 876.
static uint32_t long_runs_cap(size_t m) { return (uint32_t)(1024 + m / 16384); }

static void radix_carve(size_t n, bool with_vals, Carver &cv, uint64_t **kalt, uint32_t **valt, RowsBufs *rb,
                        uint32_t **runs = nullptr) {
    const uint32_t tiles = radix_tiles(n) + 1;
    *kalt = cv.take<uint64_t>(n ? n : 1);
    *valt = with_vals ? cv.take<uint32_t>(n ? n : 1) : nullptr;
    *rb = rows_carve(tiles, cv);
    rb->diff = cv.take<uint32_t>(1 + (tiles + kHistTiles - 1) / kHistTiles);
    if (with_vals) {
        uint32_t *list = cv.take<uint32_t>(long_runs_cap(n));
        if (runs) *runs = list;
    }
}

size_t radix_workspace_bytes(size_t n, bool with_vals) {
    Carver cv(nullptr);
    uint64_t *kalt;
    uint32_t *valt;
    RowsBufs rb;
    radix_carve(n, with_vals, cv, &kalt, &valt, &rb);
    return cv.off + 256;
}

// An array of at most kSmallSort keys: one work-group sorts it in LDS, in place
// (every key is read before any is written) or, with out.key set, into the
// output columns of join rows.
template <int ITEMS, bool HAS_VAL>
__global__ __launch_bounds__(kBlockSortThreads) void k_sort_small(uint64_t *keys, uint32_t *vals, uint32_t cap,
                                                                  const uint64_t *d_n, int lo_bit, int hi_bit,
                                                                  RowOut out) {
    __shared__ BlockSort<ITEMS, HAS_VAL> S;
    uint32_t n = cap;
    if (d_n && *d_n < cap) n = (uint32_t)*d_n;
    if (n == 0) return;
    for (uint32_t i = threadIdx.x; i < n; i += kBlockSortThreads) {
        S.key[i] = keys[i];
        if (HAS_VAL) S.val[i] = vals[i];
    }
    __syncthreads();
    block_sort<ITEMS, HAS_VAL>(S, n, lo_bit, hi_bit);
    for (uint32_t i = threadIdx.x; i < n; i += kBlockSortThreads) {
        const uint64_t k = S.key[i];
        if (HAS_VAL && out.key) {
            out.key[i] = join_sort_key_key(k);
            out.spay[i] = join_sort_key_spay(k);
            out.rpay[i] = (int32_t)S.val[i];
        } else {
            keys[i] = k;
            if (HAS_VAL) vals[i] = S.val[i];
        }
    }
}

// Up to this many keys one work-group sorts the array, and larger ones take the
// passes over tiles: four digits of 64-bit keys take 10.2 us instead of 52.7 at
// 200 keys, 10.9 / 54.9 at 1024, 20.5 / 57.7 at 4096 and 32.9 / 66.9 at 8192
// (the times grow by 2.9 us per 1024 keys, and twice the keys would not fit LDS
// with their values).
constexpr size_t kSmallSort = 8192;
constexpr size_t kSmallItems1 = kBlockSortThreads, kSmallItems4 = 4 * kBlockSortThreads;

template <bool HAS_VAL>
static int launch_sort_small(uint64_t *keys, uint32_t *vals, size_t n, const uint64_t *d_n, int lo_bit, int hi_bit,
                             hipStream_t st, const RowOut &out) {
    const uint32_t cap = (uint32_t)n;
    if (n <= kSmallItems1)
        k_sort_small<1, HAS_VAL><<<1, kBlockSortThreads, 0, st>>>(keys, vals, cap, d_n, lo_bit, hi_bit, out);
    else if (n <= kSmallItems4)
        k_sort_small<4, HAS_VAL><<<1, kBlockSortThreads, 0, st>>>(keys, vals, cap, d_n, lo_bit, hi_bit, out);
    else
        k_sort_small<8, HAS_VAL><<<1, kBlockSortThreads, 0, st>>>(keys, vals, cap, d_n, lo_bit, hi_bit, out);
    QO_LAUNCHED();
    return QO_OK;
}

static int radix_impl(uint64_t *keys, uint32_t *vals, size_t n, const uint64_t *d_n, int lo_bit, int hi_bit,
                      void *ws, hipStream_t st, const RowOut *unpack = nullptr) {
    if (n == 0) return QO_OK;
    QO_REQUIRE(n < 0xFFFFFFFFull, "sort input too large");
    QO_REQUIRE(lo_bit >= 0 && hi_bit <= 64 && lo_bit < hi_bit, "bad bit range");
    if (n <= kSmallSort) {
        const RowOut none{};
        return vals ? launch_sort_small<true>(keys, vals, n, d_n, lo_bit, hi_bit, st, unpack ? *unpack : none)
                    : launch_sort_small<false>(keys, vals, n, d_n, lo_bit, hi_bit, st, none);
    }
    const uint32_t tiles = radix_tiles(n);
    Carver cv(ws);
    uint64_t *kalt = nullptr;
    uint32_t *valt = nullptr;
    RowsBufs rb{};
    radix_carve(n, vals != nullptr, cv, &kalt, &valt, &rb);
    RadixSeg seg{0, n, d_n, 0, tiles};
    bool in_alt = false;
    QO_TRY(launch_radix_rows(keys, vals, kalt, valt, seg, lo_bit, hi_bit, rb, st, &in_alt, unpack));
    if (in_alt && !unpack) {
        // Odd number of passes: the result is in the alternate buffers.  The
        // count may only be known on the device, so copy the full capacity.
        QO_HIP(hipMemcpyAsync(keys, kalt, n * 8, hipMemcpyDeviceToDevice, st));
        if (vals) QO_HIP(hipMemcpyAsync(vals, valt, n * 4, hipMemcpyDeviceToDevice, st));
    }
    return QO_OK;
}

int launch_radix_sort_list(uint64_t *keys, const uint64_t *d_n, size_t n, void *ws, hipStream_t st) {
    if (n <= kSmallSort) return radix_impl(keys, nullptr, n, d_n, 32, 64, ws, st);
    QO_REQUIRE(n < 0xFFFFFFFFull, "sort input too large");
    const uint32_t tiles = radix_tiles(n);
    Carver cv(ws);
    uint64_t *kalt = nullptr;
    uint32_t *valt = nullptr;
    RowsBufs rb{};
    radix_carve(n, false, cv, &kalt, &valt, &rb);
    return launch_radix_rows_dyn(keys, kalt, RadixSeg{0, n, d_n, 0, tiles}, rb, rb.diff, st);
}

// ---------------------------------------------------------------------------
// Split of Records into `parts` partitions by pid = R.y % parts (stable within a
// partition): the radix passes above with the partition id as the key, one pass
// for parts <= 256, two (low, then high byte of the pid) up to 65536; then the
// partition bounds by binary search over the split output.
// ---------------------------------------------------------------------------
constexpr uint32_t kSplitMaxParts = 65536;

// bound[p] = {start, end} of partition p: the first output position whose pid
// is >= p, and the same for p + 1 (n for the last partition).
__global__ __launch_bounds__(256) void k_split_bounds(const uint64_t *__restrict__ out, size_t n, uint32_t parts,
                                                      uint2 *__restrict__ bound) {
    const uint32_t p = blockIdx.x * 256 + threadIdx.x;
    if (p >= parts) return;
    auto first_at_least = [&](uint32_t q) {
        size_t lo = 0, hi = n;
        while (lo < hi) {
            const size_t mid = lo + (hi - lo) / 2;
            if ((uint32_t)(out[mid] >> 32) % parts < q) lo = mid + 1;
            else hi = mid;
        }
        return lo;
    };
    bound[p] = uint2{(uint32_t)first_at_least(p), p + 1 < parts ? (uint32_t)first_at_least(p + 1) : (uint32_t)n};
}

size_t split_records_ws_bytes(size_t n, uint32_t parts) {
    Carver cv(nullptr);
    if (parts > 256) cv.take<uint64_t>(n ? n : 1);
    rows_carve(radix_tiles(n) + 1, cv);
    return cv.off + 256;
}

int launch_split_records(const uint64_t *in, size_t n, uint32_t parts, uint64_t *out, uint2 *bound, void *ws,
                         hipStream_t st) {
    QO_REQUIRE(parts >= 1 && parts <= kSplitMaxParts, "numPart %u outside [1, %u]", parts, kSplitMaxParts);
    QO_REQUIRE(n < 0xFFFFFFFFull, "split input too large");
    if (n > 0) {
        Carver cv(ws);
        uint64_t *alt = parts > 256 ? cv.take<uint64_t>(n) : nullptr;
        const uint32_t tiles = radix_tiles(n);
        const RowsBufs b = rows_carve(tiles + 1, cv);
        const RadixSeg sg{0, n, nullptr, 0, tiles};
        const RowsPlan rp = rows_plan(tiles);
        const unsigned hblocks = (tiles + kHistTiles - 1) / kHistTiles;
        const int npass = parts > 256 ? 2 : 1;
        for (int pass = 0; pass < npass; ++pass) {
            const uint64_t *src = pass == 0 ? in : alt;
            uint64_t *dst = pass == npass - 1 ? out : alt;
            const int sh = 8 * pass;
            k_tile_hist<true><<<hblocks, 256, 0, st>>>(src, sg, nullptr, 1, tiles, sh, b.rows, nullptr, parts);
            QO_LAUNCHED();
            if (tiles <= kRowsOneBlock) {
                k_rows_starts<<<1, 1024, 0, st>>>(b.rows, tiles);
                QO_LAUNCHED();
            } else {
                k_rows_reduce<<<rp.nb, 256, 0, st>>>(b.rows, tiles, rp.span, b.bsum);
                QO_LAUNCHED();
                k_rows_starts<<<1, 1024, 0, st>>>(b.bsum, rp.nb);
                QO_LAUNCHED();
                k_rows_apply<<<rp.nb, 256, 0, st>>>(b.rows, tiles, rp.span, b.bsum);
                QO_LAUNCHED();
            }
            k_radix_place<false, false, true><<<tiles, 256, 0, st>>>(src, nullptr, dst, nullptr, sg, nullptr, 1, tiles,
                                                                      sh, b.rows, nullptr, 0, RowOut{}, nullptr,
                                                                      nullptr, parts);
            QO_LAUNCHED();
        }
    }
    if (bound) {
        k_split_bounds<<<(parts + 255) / 256, 256, 0, st>>>(out, n, parts, bound);
        QO_LAUNCHED();
    }
    return QO_OK;
}

// (key, s_payload) as signed int32 -> order-preserving unsigned 64-bit key.
__global__ void k_pack_join(const int32_t *key, const int32_t *spay, const int32_t *rpay, size_t m, uint64_t *k64,
                            uint32_t *v32) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    size_t stride = (size_t)gridDim.x * blockDim.x;
    for (; i < m; i += stride) {
        k64[i] = join_sort_key(key[i], spay[i]);
        v32[i] = (uint32_t)rpay[i];
    }
}

__global__ void k_unpack_join(const uint64_t *k64, const uint32_t *v32, size_t m, int32_t *key, int32_t *spay,
                              int32_t *rpay) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    size_t stride = (size_t)gridDim.x * blockDim.x;
    for (; i < m; i += stride) {
        uint64_t k = k64[i];
        key[i] = join_sort_key_key(k);
        spay[i] = join_sort_key_spay(k);
        rpay[i] = (int32_t)v32[i];
    }
}

int sort_join_rows_ws(int32_t *key, int32_t *rpay, int32_t *spay, size_t m, void *ws, hipStream_t st) {
    if (m < 2) return QO_OK;
    Carver cv(ws);
    uint64_t *k64 = cv.take<uint64_t>(m);
    uint32_t *v32 = cv.take<uint32_t>(m);
    void *rws = cv.take<char>(radix_workspace_bytes(m, true));
    unsigned g = grid_for(m, 256, (unsigned)props().cu_count * 8);
    uint32_t *flag = cv.take<uint32_t>(2);
    k_pack_join<<<g, 256, 0, st>>>(key, spay, rpay, m, k64, v32);
    QO_LAUNCHED();
    return sort_packed_join_rows(k64, v32, m, rws, key, rpay, spay, st, 64, flag);
}

size_t sort_join_rows_ws_bytes(size_t m) { return m * 12 + 2048 + radix_workspace_bytes(m, true); }

// Runs of equal key after a stable sort of the packed join rows on their key
// bits (the high 32): each block owns kFixTile positions and loads kFixRun more,
// so that every run that starts in its range and has at most kFixRun rows lies
// in LDS whole.  One ballot per 64-position chunk marks where runs start; a
// row finds its run's bounds from its own chunk's marks and its neighbours',
// counts the run's rows that order before it (smaller s_payload, or equal and
// earlier: stable) and writes itself to the output columns at run start + that
// count.  Rows of runs that start outside the block's range are left to the
// block that owns the start; a run longer than kFixRun is not written: its
// start goes to the list of long runs (k_fix_long), or, without a list, it sets
// the flag.
constexpr uint32_t kFixTile = 4096;
constexpr uint32_t kFixRun = 64;
constexpr uint32_t kFixWin = kFixTile + kFixRun;
constexpr uint32_t kFixThreads = 512;  // four blocks per CU (34 KB LDS each), 8 waves per SIMD
constexpr uint32_t kFixRounds = (kFixWin + kFixThreads - 1) / kFixThreads;
constexpr uint32_t kFixChunks = kFixWin / kWave + 2;  // marks of the window's chunks and one past it

constexpr int kLongItems = 6;
constexpr uint32_t kLongLds = kLongItems * kBlockSortThreads;  // longest run sorted in LDS

// Where the run pass leaves the runs longer than kFixRun.
struct LongRuns {
    uint32_t *flag;            // set: the rows need the full-width sort
    uint32_t *n = nullptr;     // starts of the long runs (counted past cap too)
    uint32_t *list = nullptr;  // null: a long run sets the flag
    uint32_t cap = 0;
};
constexpr uint32_t kFixLongMax = kFixTile / (kFixRun + 1) + 1;  // long runs that start in a tile

// Block work of the run pass: positions [t0, t0 + kFixTile) of m rows (k, v).
QO_DEV void fix_runs_tile(const uint64_t *__restrict__ k, const uint32_t *__restrict__ v, size_t m, size_t t0,
                          const RowOut &out, const LongRuns &lr) {
    static_assert(kFixWin % kWave == 0, "window of whole chunks");
    __shared__ uint32_t s_hi[kFixWin];
    __shared__ uint32_t s_lo[kFixWin + 4];  // 4 words of slack for the unrolled rank loop
    __shared__ uint64_t s_mark[kFixChunks];
    __shared__ uint32_t s_long[kFixLongMax], s_nlong, s_at;
    if (threadIdx.x == 0) s_nlong = 0;
    const uint32_t own = (uint32_t)(m - t0 < kFixTile ? m - t0 : kFixTile);
    const uint32_t len = (uint32_t)(m - t0 < kFixWin ? m - t0 : kFixWin);
    const bool data_end = t0 + len == m;  // the window reaches the last row
#pragma unroll
    for (uint32_t u = 0; u < kFixRounds; ++u) {
        const uint32_t i = u * kFixThreads + threadIdx.x;
        if (i < len) {
            const uint64_t x = k[t0 + i];
            s_hi[i] = (uint32_t)(x >> 32);
            s_lo[i] = (uint32_t)x;
        }
    }
    const uint32_t prev_key = t0 > 0 ? (uint32_t)(k[t0 - 1] >> 32) : 0u;
    __syncthreads();
    // Run-start marks: position p starts a run if its key differs from the row
    // before it (the first row of all rows starts one); past the last row every
    // position counts as a start, past a cut-off window none does.
    const unsigned lane = lane_id();
    for (uint32_t c = wave_id(); c < kFixChunks; c += kFixThreads / kWave) {
        const uint32_t p = c * kWave + lane;
        bool start;
        if (p < len) start = p == 0 ? (t0 == 0 || prev_key != s_hi[0]) : s_hi[p] != s_hi[p - 1];
        else start = data_end;
        const uint64_t mk = ballot(start);
        if (lane == 0) s_mark[c] = mk;
    }
    __syncthreads();
    bool long_run = false;
    auto is_long = [&](uint32_t i, uint32_t s) {
        long_run = true;
        if (i != s) return;
        s_long[atomicAdd(&s_nlong, 1u)] = s;  // the run's first row lists it
        if (lr.list && t0 + s + kLongLds < m && (uint32_t)(k[t0 + s + kLongLds] >> 32) == s_hi[s]) *lr.flag = 1u;
    };
    for (uint32_t i = threadIdx.x; i < len; i += kFixThreads) {
        const uint32_t c = i / kWave;  // uniform across the wave
        const uint64_t at_or_below = lane == kWave - 1 ? ~0ull : (2ull << lane) - 1;
        const uint64_t mc = s_mark[c];
        uint32_t s;
        if (mc & at_or_below) {
            s = c * kWave + 63u - (uint32_t)__builtin_clzll(mc & at_or_below);
        } else if (c == 0) {
            continue;  // the run began before the block's range
        } else if (s_mark[c - 1]) {
            s = (c - 1) * kWave + 63u - (uint32_t)__builtin_clzll(s_mark[c - 1]);
        } else {
            long_run = true;  // no start within 64 positions back
            continue;
        }
        if (s >= own) continue;  // the next block's run
        const uint64_t above = mc & ~at_or_below;
        uint32_t e;
        if (above) {
            e = c * kWave + (uint32_t)__builtin_ctzll(above);
        } else if (s_mark[c + 1]) {
            e = (c + 1) * kWave + (uint32_t)__builtin_ctzll(s_mark[c + 1]);
        } else {
            is_long(i, s);
            continue;
        }
        if (e - s > kFixRun) {
            is_long(i, s);
            continue;
        }
        const uint32_t xl = s_lo[i];
        uint32_t rank = 0;
        for (uint32_t j = s; j < e; j += 4) {
            const uint32_t y0 = s_lo[j], y1 = s_lo[j + 1], y2 = s_lo[j + 2], y3 = s_lo[j + 3];
            rank += (y0 < xl || (y0 == xl && j < i)) ? 1u : 0u;
            rank += (j + 1 < e && (y1 < xl || (y1 == xl && j + 1 < i))) ? 1u : 0u;
            rank += (j + 2 < e && (y2 < xl || (y2 == xl && j + 2 < i))) ? 1u : 0u;
            rank += (j + 3 < e && (y3 < xl || (y3 == xl && j + 3 < i))) ? 1u : 0u;
        }
        const size_t dst = t0 + s + rank;
        const uint64_t x = ((uint64_t)s_hi[i] << 32) | xl;
        out.key[dst] = join_sort_key_key(x);
        out.spay[dst] = join_sort_key_spay(x);
        out.rpay[dst] = (int32_t)v[t0 + i];
    }
    if (!lr.list) {
        if (long_run) atomicOr(lr.flag, 1u);
        return;
    }
    // One reservation per block: one per run, from every wave of the chip to one
    // address, took 1 ms for 140,000 runs.
    __syncthreads();
    if (s_nlong == 0) return;
    if (threadIdx.x == 0) s_at = atomicAdd(lr.n, s_nlong);
    __syncthreads();
    if (threadIdx.x < s_nlong) {
        const uint32_t at = s_at + threadIdx.x;
        if (at < lr.cap) lr.list[at] = (uint32_t)t0 + s_long[threadIdx.x];
    }
}

__global__ __launch_bounds__(kFixThreads) void k_fix_runs(const uint64_t *__restrict__ k, const uint32_t *__restrict__ v,
                                                          size_t m, RowOut out, LongRuns lr) {
    fix_runs_tile(k, v, m, (size_t)blockIdx.x * kFixTile, out, lr);
}

// The long runs of k_fix_runs, one work-group each in turn, sorted by s_payload
// in LDS.  A run longer than kLongLds rows, or more runs than the list holds,
// sets the flag before any is sorted (the full-width sort then takes all rows).
// Bound by the passes' chain of dependent LDS steps: 40 us for a run of 6000
// rows, where the full-width sort of 10,000 to 100,000 rows costs 75.  Runs past
// LDS, by digit passes of one work-group through memory, took 79 us at 7000 rows,
// 171 at 20,000 and 735 at 100,000, so from there on the full width is the
// cheaper one (10 M rows in runs of 20,000: 1.06 ms and 0.88).

// End of the run of equal key that starts at s, looked for up to `hi` (returned
// when the run goes on there), by the whole work-group: 1024 probes a round.
QO_DEV uint64_t run_end(const uint64_t *k, uint64_t s, uint64_t hi, uint32_t *s_min) {
    const uint32_t key = (uint32_t)(k[s] >> 32);
    uint64_t lo = s;  // the run's; the end lies in (lo, hi]
    while (hi - lo > 1) {
        const uint64_t step = (hi - lo + kBlockSortThreads - 1) / kBlockSortThreads;
        const uint32_t probes = (uint32_t)((hi - lo - 1) / step);  // below hi; at most 1023
        if (threadIdx.x == 0) *s_min = probes;
        __syncthreads();
        if (threadIdx.x < probes && (uint32_t)(k[lo + (threadIdx.x + 1) * step] >> 32) != key) atomicMin(s_min, threadIdx.x);
        __syncthreads();
        const uint32_t c = *s_min;  // probes inside the run: the end lies in (probe c - 1, probe c] or up to hi
        __syncthreads();
        lo += c * step;
        hi = lo + step < hi ? lo + step : hi;
    }
    return hi;
}

struct LongLds {
    BlockSort<kLongItems, false> S;
    uint32_t min;
};

// The run [s, s + len) of one key, by the whole work-group; len <= kLongLds.
// Ends with a barrier.
QO_DEV void fix_run_lds(LongLds &L, const uint64_t *k, const uint32_t *v, uint64_t s, uint32_t len, const RowOut &out) {
    const int32_t key = join_sort_key_key(k[s]);
    // Sorted as s_payload (order-preserving) << 32 | r_payload.
    for (uint32_t i = threadIdx.x; i < len; i += kBlockSortThreads) L.S.key[i] = (k[s + i] << 32) | v[s + i];
    __syncthreads();
    block_sort<kLongItems, false>(L.S, len, 32, 64);
    for (uint32_t i = threadIdx.x; i < len; i += kBlockSortThreads) {
        const uint64_t x = L.S.key[i];
        out.key[s + i] = key;
        out.spay[s + i] = (int32_t)((uint32_t)(x >> 32) ^ 0x80000000u);
        out.rpay[s + i] = (int32_t)(uint32_t)x;
    }
    __syncthreads();  // S is reused
}

__global__ __launch_bounds__(kBlockSortThreads) void k_fix_long(const uint64_t *k, const uint32_t *v, size_t m, RowOut out,
                                                                LongRuns lr) {
    __shared__ LongLds L;
    const uint32_t n = *lr.n;
    if (n == 0 || *lr.flag) return;  // whole block
    if (n > lr.cap) {
        if (threadIdx.x == 0) *lr.flag = 1u;
        return;  // every block
    }
    for (uint32_t r = blockIdx.x; r < n; r += gridDim.x) {
        const uint64_t s = lr.list[r];
        const uint64_t e = run_end(k, s, std::min<uint64_t>(m, s + kLongLds), &L.min);
        fix_run_lds(L, k, v, s, (uint32_t)(e - s), out);
    }
}

// Segmented form: block b is global tile b of the segments (kSortTile rows per
// tile; n = *d_n clamped to cap rows per segment).
__global__ __launch_bounds__(kFixThreads) void k_fix_runs_seg(const uint64_t *__restrict__ k,
                                                              const uint32_t *__restrict__ v, const RadixSeg *segs,
                                                              int nseg, const RowOut *outs, LongRuns lr) {
    const int si = seg_index_of(segs, nseg, blockIdx.x);
    const RadixSeg sg = segs[si];
    uint64_t n = sg.d_n ? *sg.d_n : sg.cap;
    if (n > sg.cap) n = sg.cap;
    const size_t t0 = (size_t)(blockIdx.x - sg.tile0) * kFixTile;
    if (t0 >= n) return;  // whole block
    fix_runs_tile(k + sg.base, v + sg.base, n, t0, outs[si], lr);
}

int launch_fix_runs_segments(const uint64_t *keys, const uint32_t *vals, const RadixSeg *d_segs, int nseg,
                             uint32_t total_tiles, const RowOut *d_outs, uint32_t *long_flag, hipStream_t st) {
    static_assert(kFixTile == (uint32_t)kSortTile, "run pass tiles are sort tiles");
    if (total_tiles == 0) return QO_OK;
    k_fix_runs_seg<<<total_tiles, kFixThreads, 0, st>>>(keys, vals, d_segs, nseg, d_outs, LongRuns{long_flag});
    QO_LAUNCHED();
    return QO_OK;
}

int sort_packed_join_rows(uint64_t *k64, uint32_t *v32, size_t m, void *rws, int32_t *key, int32_t *rpay,
                          int32_t *spay, hipStream_t st, int hi_bit, uint32_t *flag) {
    if (m == 0) return QO_OK;
    if (m == 1) {
        k_unpack_join<<<1, 256, 0, st>>>(k64, v32, m, key, spay, rpay);
        QO_LAUNCHED();
        return QO_OK;
    }
    hi_bit = std::max(1, std::min(64, hi_bit));
    // The last radix pass writes the output columns (no separate unpack pass).
    const RowOut out{key, rpay, spay};
    // Few rows: one work-group sorts them on the full width, and no flag is read back.
    if (!flag || hi_bit <= 32 || m <= kSmallSort) return radix_impl(k64, v32, m, nullptr, 0, hi_bit, rws, st, &out);
    // Radix passes over the key bits only (stable: a key's rows keep the probe's
    // order), then one pass that sorts every run of equal key by s_payload and
    // writes the output columns: for 2^24 build keys 3 passes + 1 instead of 7.
    QO_REQUIRE(m < 0xFFFFFFFFull, "sort input too large");
    Carver cv(rws);
    uint64_t *kalt = nullptr;
    uint32_t *valt = nullptr;
    RowsBufs rb{};
    uint32_t *runs = nullptr;
    radix_carve(m, true, cv, &kalt, &valt, &rb, &runs);
    const RadixSeg seg{0, m, nullptr, 0, radix_tiles(m)};
    bool in_alt = false;
    QO_TRY(launch_radix_rows(k64, v32, kalt, valt, seg, 32, hi_bit, rb, st, &in_alt, nullptr));
    QO_TRY(launch_fill_u32(flag, 0, 2, st));
    const size_t blocks = (m + kFixTile - 1) / kFixTile;
    const LongRuns lr{flag, flag + 1, runs, long_runs_cap(m)};
    const uint64_t *ks = in_alt ? kalt : k64;
    const uint32_t *vs = in_alt ? valt : v32;
    k_fix_runs<<<(unsigned)blocks, kFixThreads, 0, st>>>(ks, vs, m, out, lr);
    QO_LAUNCHED();
    k_fix_long<<<(unsigned)props().cu_count * 2, kBlockSortThreads, 0, st>>>(ks, vs, m, out, lr);
    QO_LAUNCHED();
    uint32_t long_run = 0;
    QO_HIP(hipMemcpyAsync(&long_run, flag, 4, hipMemcpyDeviceToHost, st));
    QO_HIP(hipStreamSynchronize(st));
    if (!long_run) return QO_OK;
    // Very long runs, or very many long ones: sort all rows on the full width
    // (the result does not depend on the rows' current order).
    if (in_alt) {
        QO_HIP(hipMemcpyAsync(k64, kalt, m * 8, hipMemcpyDeviceToDevice, st));
        QO_HIP(hipMemcpyAsync(v32, valt, m * 4, hipMemcpyDeviceToDevice, st));
    }
    return radix_impl(k64, v32, m, nullptr, 0, hi_bit, rws, st, &out);
}

}  // namespace qo

using namespace qo;

extern "C" {

int qo_sort_records(qo_record *data, size_t n, qo_stream s) {
    QO_ENTER();
    if (n < 2) return QO_OK;
    QO_REQUIRE(data && ((uintptr_t)data % 8) == 0, "records must be 8-byte aligned device memory");
    hipStream_t st = stream_of(s);
    int status = QO_OK;
    void *ws = workspace(st, radix_workspace_bytes(n, false), &status);
    if (!ws) return status;
    // A Record {x, y} read as little-endian uint64 has y in bits 32..63.
    return launch_radix_sort_list(reinterpret_cast<uint64_t *>(data), nullptr, n, ws, st);
}

int qo_sort_join_rows(int32_t *key, int32_t *rpay, int32_t *spay, size_t m, qo_stream s) {
    QO_ENTER();
    if (m < 2) return QO_OK;
    QO_REQUIRE(key && rpay && spay, "null pointer");
    hipStream_t st = stream_of(s);
    int status = QO_OK;
    void *ws = workspace(st, sort_join_rows_ws_bytes(m), &status);
    if (!ws) return status;
    return sort_join_rows_ws(key, rpay, spay, m, ws, st);
}

}  // extern "C"
