// Segmented radix sort interface and the join-row sort key shared by the plain
// and batched paths.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "qo_device.hpp"

namespace qo {

constexpr int kSortItems = 16;
constexpr int kSortTile = 256 * kSortItems;

// One independently sorted array: elements [base, base + n) of the shared key /
// value arrays, n = *d_n (clamped to cap) or cap when d_n is null.  The
// segment owns global tiles [tile0, tile0 + ntile), ntile = ceil(cap / tile).
struct RadixSeg {
    uint64_t base;
    uint64_t cap;
    const uint64_t *d_n;
    uint32_t tile0;
    uint32_t ntile;
};

// Output columns of a sorted join-row segment: the last pass of a join-row
// sort writes (key, r_payload, s_payload) here instead of the packed rows.
struct RowOut {
    int32_t *key, *rpay, *spay;
};

// Tiles [t0, t1) (segment-local) of segment `seg`: one block of the up-front
// digit count of a segmented sort.
struct SweepChunk {
    uint32_t seg, t0, t1;
};
constexpr uint32_t kSweepChunkTiles = 16;
// Workspace of launch_radix_rows_segments.
size_t radix_rows_seg_bytes(uint32_t total_tiles, int nseg, uint32_t nchunks);
// Segmented sort by bits [lo_bit, hi_bit): digit starts per segment from the
// chunks (segment s owns chunks [chunk0[s], chunk0[s + 1])), then per pass a
// tile histogram, a segmented column scan and the placement.  On return
// *in_alt tells whether the data ended in kalt / valt.
// With d_outs (one RowOut per segment, device memory) the keys are join
// sort keys with r_payload values and the last pass writes each segment's
// rows unpacked into its RowOut; the packed result is then not kept.  With
// run_if every kernel returns at once unless *run_if != 0 (decided on the
// device, for stream captures).
int launch_radix_rows_segments(uint64_t *keys, uint32_t *vals, uint64_t *kalt, uint32_t *valt,
                               const RadixSeg *d_segs, int nseg, uint32_t total_tiles, const SweepChunk *d_chunks,
                               uint32_t nchunks, const uint32_t *d_chunk0, int lo_bit, int hi_bit, void *ws,
                               hipStream_t st, bool *in_alt, const RowOut *d_outs = nullptr,
                               const uint32_t *run_if = nullptr);
// After a segmented sort of join rows on their key bits only [32, 64): sorts
// every run of equal key by s_payload and writes each segment's rows to its
// RowOut (segment tiles of kSortTile rows); a run longer than 64 rows sets
// *long_flag and is not written.
int launch_fix_runs_segments(const uint64_t *keys, const uint32_t *vals, const RadixSeg *d_segs, int nseg,
                             uint32_t total_tiles, const RowOut *d_outs, uint32_t *long_flag, hipStream_t st);
// Join rows sort ascending by (key, s_payload) as signed int32: flip the sign
// bits so unsigned 64-bit order is the signed lexicographic order.
__host__ __device__ __forceinline__ uint64_t join_sort_key(int32_t key, int32_t spay) {
    return ((uint64_t)((uint32_t)key ^ 0x80000000u) << 32) | ((uint32_t)spay ^ 0x80000000u);
}
__host__ __device__ __forceinline__ int32_t join_sort_key_key(uint64_t k) {
    return (int32_t)((uint32_t)(k >> 32) ^ 0x80000000u);
}
__host__ __device__ __forceinline__ int32_t join_sort_key_spay(uint64_t k) {
    return (int32_t)((uint32_t)k ^ 0x80000000u);
}

// Lanes of this wave that are active and hold the same 8-bit digit.
QO_DEV uint64_t match_digit(uint32_t d, bool valid) {
    uint64_t m = ballot(valid);
#pragma unroll
    for (int b = 0; b < 8; ++b) {
        uint64_t bb = ballot((d >> b) & 1u);
        m &= ((d >> b) & 1u) ? bb : ~bb;
    }
    return m;
}

// A sort by the high 32 key bits whose passes are picked on the device: a digit
// in which all keys agree gets no placement.  An odd number of placements would
// leave the keys in the other buffer, so the pass of the lowest such digit then
// copies them over (with four digits there is one).  diff: the bits (of key >> 32)
// in which any key differs from the first.  Returns what the pass at `shift` does
// (0: nothing) and, in bit 8, whether the keys are in the other buffer before it.
// Kernels read diff through a __restrict__ argument: as a scalar load it is there
// in a fraction of the microsecond a vector load takes at the start of every block.
constexpr uint32_t kPassPlace = 1, kPassCopy = 2;
QO_DEV uint32_t radix_pass(uint32_t diff, int shift) {
    uint32_t mask = 0;  // passes that place
#pragma unroll
    for (int p = 0; p < 4; ++p) mask |= (((diff >> (8 * p)) & 255u) != 0 ? 1u : 0u) << p;
    const uint32_t copy = (__popc(mask) & 1) ? ~mask & (mask + 1u) : 0u;  // lowest pass without a placement
    const uint32_t p = 1u << ((shift - 32) / 8);
    const uint32_t before = __popc((mask | copy) & (p - 1u));
    return ((mask & p) ? kPassPlace : (copy & p) ? kPassCopy : 0u) | ((before & 1u) << 8);
}
// Sorts `list` by the high 32 bits, n = *d_n (at most `capacity`).
int launch_radix_sort_list(uint64_t *list, const uint64_t *d_n, size_t capacity, void *ws, hipStream_t st);

// One-block stable radix sort of up to kBlockSortThreads * ITEMS 64-bit keys
// (and 32-bit values) that lie in LDS.  What bounds it is the chain of passes:
// a pass reads the block's keys, ranks them with wave ballots, scans 16 x 256
// digit counts and scatters them back, about 2 us each at one key per thread
// and 7 us at eight.  A launch per step of a pass (histogram, scan, placement)
// takes 13 to 17 us per pass for arrays of this size.  Digits in which all
// keys agree get no pass, so a narrow key range costs nothing.
constexpr int kBlockSortThreads = 1024;
constexpr int kBlockSortWaves = kBlockSortThreads / kWave;

template <int ITEMS, bool HAS_VAL>
struct BlockSort {
    static constexpr uint32_t kMax = (uint32_t)kBlockSortThreads * ITEMS;
    uint64_t key[kMax];
    uint32_t val[HAS_VAL ? kMax : 1];
    uint32_t cnt[kBlockSortWaves][256];
    uint32_t dpre[256];
    uint32_t w[kBlockSortWaves];
    uint64_t diff[kBlockSortWaves];
};

// Sorts S.key[0, n) (and S.val) by bits [lo_bit, hi_bit) (whole 8-bit digits
// from lo_bit).  All threads call it after a barrier that follows the writes of
// S; on return (after a barrier) S holds the sorted array.
template <int ITEMS, bool HAS_VAL>
QO_DEV void block_sort(BlockSort<ITEMS, HAS_VAL> &S, uint32_t n, int lo_bit, int hi_bit) {
    const unsigned w = wave_id(), lane = lane_id();
    // Wave w owns positions [w * 64 J, (w + 1) * 64 J): all waves share a short array.
    const int J = (int)((n + kBlockSortThreads - 1) / kBlockSortThreads);
    const uint32_t wb = w * (uint32_t)J * kWave;
    uint64_t k[ITEMS];
    uint32_t v[ITEMS], rank[ITEMS];
    // Bits in which any key differs from the first.
    uint64_t diff = 0;
    const uint64_t first = S.key[0];
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
        const uint32_t idx = wb + j * kWave + lane;
        if (j < J && idx < n) diff |= S.key[idx] ^ first;
    }
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) diff |= __shfl_xor(diff, o, kWave);
    if (lane == 0) S.diff[w] = diff;
    __syncthreads();
    diff = 0;
#pragma unroll
    for (int i = 0; i < kBlockSortWaves; ++i) diff |= S.diff[i];
    for (int sh = lo_bit; sh < hi_bit; sh += 8) {
        if (((diff >> sh) & 255u) == 0) continue;  // block-uniform
#pragma unroll
        for (int i = 0; i < 256 / kWave; ++i) S.cnt[w][i * kWave + lane] = 0;
        wave_lockstep();
#pragma unroll
        for (int j = 0; j < ITEMS; ++j) {
            if (j >= J) break;
            const uint32_t idx = wb + j * kWave + lane;
            const bool valid = idx < n;
            k[j] = valid ? S.key[idx] : 0;
            if (HAS_VAL) v[j] = valid ? S.val[idx] : 0u;
        }
#pragma unroll
        for (int j = 0; j < ITEMS; ++j) {
            if (j >= J) break;
            const bool valid = wb + j * kWave + lane < n;
            const uint32_t d = (uint32_t)(k[j] >> sh) & 255u;
            const uint64_t m = match_digit(d, valid);
            const uint32_t pre = S.cnt[w][d];
            const uint32_t r = popc(m & lanemask_lt());
            wave_lockstep();  // every lane has read its digit's count before the leaders advance it
            if (valid && r == 0) S.cnt[w][d] = pre + popc(m);
            wave_lockstep();
            rank[j] = pre + r;
        }
        __syncthreads();
        uint32_t tot = 0;
        if (threadIdx.x < 256) {
            uint32_t c[kBlockSortWaves];
#pragma unroll
            for (int i = 0; i < kBlockSortWaves; ++i) c[i] = S.cnt[i][threadIdx.x];
#pragma unroll
            for (int i = 0; i < kBlockSortWaves; ++i) {
                S.cnt[i][threadIdx.x] = tot;
                tot += c[i];
            }
        }
        // Threads 0..255 come first in the block, so their exclusive scan is the digit start.
        const uint32_t start = block_excl_scan<kBlockSortWaves>(tot, S.w);
        if (threadIdx.x < 256) S.dpre[threadIdx.x] = start;
        __syncthreads();
#pragma unroll
        for (int j = 0; j < ITEMS; ++j) {
            if (j >= J) break;
            if (wb + j * kWave + lane < n) {
                const uint32_t d = (uint32_t)(k[j] >> sh) & 255u;
                const uint32_t p = S.dpre[d] + S.cnt[w][d] + rank[j];
                S.key[p] = k[j];
                if (HAS_VAL) S.val[p] = v[j];
            }
        }
        __syncthreads();
    }
}

}  // namespace qo
