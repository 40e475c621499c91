// bin_execute.h - EXECUTE by binning: every row's minimum writer found in LDS.
//
// The register paths touch one random 128-byte register line per operation.
// Here the operations are binned by row first and each bucket's rows are
// decided in LDS; the per-row registers in HBM are not touched:
//   order    are the TIDs non-decreasing in batch position (the usual batch)?
//            Then position alone is the priority;
//   bin      one pass over the batch.  A 1024-thread block takes a tile of
//            P * 1024 consecutive op slots, drops operations that a writer in
//            the same tile already decides (below), ranks the others per
//            bucket with LDS counters, places them bucket by bucket, writes
//            before reads, in LDS and writes the tile out in that order, with
//            the start of each bucket's writes and reads (16 bits each) in a
//            table;
//   flags    one block per bucket: reads the writes of the bucket's run of
//            every tile, for the W minima of its rows in LDS, then the whole
//            runs, setting the fast form's flags from the minima: a writer
//            behind the minimum is doomed; a reader behind it has raw; a
//            reader ahead of it gives the minimum writer war.  Without a write
//            in the batch there is nothing to do.
// A row's bucket is the top bits of row * odd mod 2^K (a bijection), so ranges
// of hot rows spread over the buckets.  An entry is 4 bytes -- row within the
// bucket, is-write, slot within the tile; the tile gives the
// rest -- so no position or counting pass goes through memory: the batch
// is read once, and 4 bytes per operation written once, read once and, of
// writes, twice (the second time mostly from the L2).
//
// The in-tile filter: writers enter (position, row) into a direct-mapped LDS
// table with a 64-bit minimum.  An operation that finds its own row there
// under a lower position is behind a writer: a write has waw, a read raw, and
// neither can matter to any other transaction (it is not its row's minimum
// writer, and as a reader it is behind that minimum, so gives no war).  It is
// flagged at once and leaves the batch, which keeps a skewed epoch's hot rows
// from filling one bucket.  With TIDs out of order (TID, row) takes the place
// of (position, row), and equal TIDs drop nothing.
//
// Reads of a hot row that no writer in their tile decides do fill one bucket.
// A bucket whose long runs (four times its share of a tile) hold more than 8192
// + twice the average entries is hot: it is left to the blocks behind the
// buckets' own, 16 of which share it.  2^20 x 16 reads and writes, Zipf 0.99 on
// 10M rows, 99.9 % reads: 406 us with a block for every bucket, 189 so.
//
// The minima of a bucket sit in an array by row when it has at most
// 2^kBinRowBits rows; buckets of more rows (up to 2^kBinHashBits: many rows
// against few operations) use a hash table of the rows written, or, where those
// fill it, the array once per part of their rows.  TIDs out of order are 64 bits
// a minimum: the array takes the rows in two parts, the hash table as many
// shares of them as the bucket's writes need.
//
// 2^20 transactions x 16 ops on 10M rows: 486 us on the registers (285
// registration, 202 read marking) -> 190 us at Zipf 0.6 (order 3, bin 65,
// flags 122), 515 -> 157 us at Zipf 0.99.  The bin kernel moves 268 MB at 4.1
// TB/s; the flags kernel is bound by instruction issue (1M runs of 16 entries,
// half of the lanes idle; 130 us with each entry's transaction by division)
// and, at Zipf 0.6, by its 9M scattered flag bytes (58 us without them).  With
// shuffled TIDs 340 to 400 us, of which the random loads of TIDs are the most;
// without the filter and the shares it took 1.5 to 2.5 ms under skew.
//
// A Source gives the operation of op slot i: load(i) its words (every slot
// below n_ops may be loaded), decode() whether it registers, its row (< 2^32),
// whether it is a write, and the slot's range errors.  kSmallTiles: its shapes
// are tiles of 4 slots per thread and at most 1024 buckets.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <type_traits>

#include "device_common.h"
#include "ltpg_internal.h"

namespace ltpg {
namespace {

constexpr uint32_t kBinBlock = 1024;
constexpr uint32_t kBinRows = 1u << kBinRowBits;
constexpr uint32_t kBinMul = 0x9E3779B1u;  // odd
constexpr uint32_t kBinHashSlots = kBinRows / 2;

// An epoch's commit counts start at zero (one block calls it).
__device__ __forceinline__ void zero_epoch_counts(DeviceCounters *ctr, uint32_t threads)
{
    for (uint32_t c = threadIdx.x; c < kCounterStripes * kCountedTypes; c += threads)
        ctr->commits[c / kCountedTypes][c % kCountedTypes] = 0;
    if (threadIdx.x == 0) ctr->kv_list_n = 0;
}

// i mod d and i / d for i < 2^32 by one high multiply: with m = floor(2^32 /
// d) (2^32 - 1 for d = 1) the quotient is exact or one too small.
struct FastMod {
    uint32_t d, m;
};

__device__ __forceinline__ uint32_t fast_div(const FastMod &f, uint32_t i, uint32_t *rem)
{
    uint32_t q = __umulhi(i, f.m);
    uint32_t r = i - q * f.d;
    if (r >= f.d) {
        r -= f.d;
        ++q;
    }
    *rem = r;
    return q;
}

struct BinArgs {
    // set by the caller of launch_bin
    uint32_t width;        // op slot i is slot i / width of transaction i % width, or with rm the other way round
    uint32_t n_ops;
    bool rm;
    const uint32_t *tids;
    uint32_t B;            // transactions
    uint8_t *doomed, *raw_flag, *war_flag;
    // set by launch_bin
    uint32_t mask, row_bits, nb, tiles, tile_bits;  // 2^K - 1; log2 rows per bucket; buckets; tiles; log2 slots per tile
    FastMod per;
    uint8_t epoch;
    uint32_t *ent;         // [tiles << tile_bits]
    uint32_t *off;         // [tiles][nb + 1] each bucket's run in the tile: its start, and << 16 its reads'
    uint32_t *marks;       // [kMarkHot + nb], see BinBuffers
    uint32_t long_run;     // tile runs beyond this count towards their bucket's long ones,
    uint32_t hot;          // which is hot if those hold more entries than this
    DeviceCounters *ctr;
};

__device__ __forceinline__ uint32_t bin_txn(const BinArgs &a, uint32_t i)
{
    uint32_t r;
    const uint32_t q = fast_div(a.per, i, &r);
    return a.rm ? q : r;
}

// Exclusive prefix sum over the block of one value per thread; *total gets
// the sum.  Wave scans by shuffles, then the 16 wave totals through LDS.
__device__ __forceinline__ uint32_t block_exclusive_sum(uint32_t v, uint32_t *s_wt, uint32_t *total)
{
    constexpr uint32_t kWaves = kBinBlock / 64;
    const uint32_t lane = threadIdx.x % 64, wave = threadIdx.x / 64;
    uint32_t inc = v;
#pragma unroll
    for (uint32_t d = 1; d < 64; d <<= 1) {
        const uint32_t x = __shfl_up(inc, d);
        if (lane >= d) inc += x;
    }
    if (lane == 63) s_wt[wave] = inc;
    __syncthreads();
    uint32_t before = 0, all = 0;
#pragma unroll
    for (uint32_t w = 0; w < kWaves; ++w) {
        const uint32_t t = s_wt[w];
        before += w < wave ? t : 0u;
        all += t;
    }
    *total = all;
    return before + inc - v;
}

// No bucket has long runs yet (one block calls it, before the bin kernel).
__device__ __forceinline__ void bin_no_long_runs(uint32_t *marks, uint32_t nb, uint32_t threads)
{
    for (uint32_t b = threadIdx.x; b < nb; b += threads) marks[kMarkLong + b] = 0;
    if (threadIdx.x == 0) marks[kMarkHot] = 0;
}

// With `clear` (the epoch that keeps no state between calls) also the flags of
// the block's transactions and the range errors start over.
constexpr uint32_t kOrderBlock = 256;
__global__ __launch_bounds__(kOrderBlock) void bin_order_kernel(BinArgs a, bool zero_counts, bool clear)
{
    if (zero_counts && blockIdx.x == 0) zero_epoch_counts(a.ctr, kOrderBlock);
    if (blockIdx.x == 0) bin_no_long_runs(a.marks, a.nb, kOrderBlock);
    if (clear) {
        if (blockIdx.x == 0 && threadIdx.x == 0) a.ctr->range_errors = 0;
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) {
            const uint32_t t = blockIdx.x * (4 * kOrderBlock) + u * kOrderBlock + threadIdx.x;
            if (t < a.B) a.doomed[t] = a.raw_flag[t] = a.war_flag[t] = 0;
        }
    }
    // four pairs per thread, all loads in flight together
    const uint32_t first = blockIdx.x * (4 * kOrderBlock) + threadIdx.x;
    uint32_t lo[4], hi[4];
#pragma unroll
    for (uint32_t u = 0; u < 4; ++u) {
        const uint32_t t = first + u * kOrderBlock;
        lo[u] = a.tids[t < a.B - 1 ? t : a.B - 1];
        hi[u] = a.tids[t < a.B - 1 ? t + 1 : a.B - 1];
    }
    bool out = false;
#pragma unroll
    for (uint32_t u = 0; u < 4; ++u) out |= lo[u] > hi[u];
    // a stale equal number (255 epochs ago) only costs the slower path
    if (out) a.marks[kMarkUnsorted] = a.epoch;
}

// A tile's LDS.  Both orders' code is in one kernel, which learns the order on
// the device; with one body for both the registers that one needs spill in the
// other (bin kernel of the above 61 us, 75 and more so).
template <uint32_t P, uint32_t MaxB>
struct BinTile {
    static constexpr uint32_t kSlots = P * kBinBlock, kFilter = kSlots / 2;
    __align__(16) uint32_t ent[kSlots];  // the filter first, then the tile in bucket order
    __align__(8) uint32_t at[2 * MaxB];  // counts of each bucket's writes and reads, then their starts
    uint32_t wt[kBinBlock / 64];
};

// ORDERED: TIDs ascend with the position, which is compared instead.
template <class Source, uint32_t P, uint32_t MaxB, bool ORDERED>
__device__ __forceinline__ void bin_tile(const BinArgs &a, const Source &src, BinTile<P, MaxB> &tile)
{
    constexpr uint32_t T = P * kBinBlock, kFilter = BinTile<P, MaxB>::kFilter;
    constexpr uint32_t kPer = MaxB / kBinBlock;  // buckets per thread at most
    constexpr uint32_t G = 4;                    // slots whose loads are in flight per thread
    uint32_t *s_ent = tile.ent, *s_at = tile.at;
    unsigned long long *s_min = reinterpret_cast<unsigned long long *>(tile.ent);
    const uint32_t base = blockIdx.x * T + threadIdx.x;
    for (uint32_t k = threadIdx.x; k < kFilter; k += kBinBlock) s_min[k] = ~0ull;
    for (uint32_t c = threadIdx.x; c < 2 * a.nb; c += kBinBlock) s_at[c] = 0;
    __syncthreads();
    uint32_t hb[P];  // hashed row << 1 | is-write, or all-ones: nothing to register
    uint32_t bad = 0;
#pragma unroll
    for (uint32_t g = 0; g < P; g += G) {
        typename Source::Raw raw[G];
        uint32_t first[G];
#pragma unroll
        for (uint32_t u = 0; u < G; ++u) {
            const uint32_t i = base + (g + u) * kBinBlock, j = i < a.n_ops ? i : 0u;
            raw[u] = src.load(a, j);
            first[u] = ORDERED ? 0u : a.tids[bin_txn(a, j)];
        }
#pragma unroll
        for (uint32_t u = 0; u < G; ++u) {
            const uint32_t i = base + (g + u) * kBinBlock;
            bool use;
            uint32_t row;
            bool write;
            bad += src.decode(a, raw[u], i, i < a.n_ops, &use, &row, &write);
            const uint32_t x = (row * kBinMul) & a.mask;
            hb[g + u] = use ? x << 1 | (write ? 1u : 0u) : ~0u;
            if (use && write)
                atomicMin(&s_min[(x ^ (x >> 12)) & (kFilter - 1)],
                          (unsigned long long)(ORDERED ? bin_txn(a, i) : first[u]) << 32 | x);
        }
    }
    if (bad) atomicAdd(&a.ctr->range_errors, bad);
    __syncthreads();
    uint32_t rank[P];
#pragma unroll
    for (uint32_t u = 0; u < P; ++u) {
        const uint32_t x = hb[u] >> 1;
        const bool write = hb[u] & 1u;
        if (hb[u] != ~0u) {
            const unsigned long long v = s_min[(x ^ (x >> 12)) & (kFilter - 1)];
            if ((uint32_t)v == x) {
                const uint32_t t = bin_txn(a, base + u * kBinBlock);
                if ((uint32_t)(v >> 32) < (ORDERED ? t : a.tids[t])) {
                    if (write)
                        a.doomed[t] = a.epoch;
                    else
                        a.raw_flag[t] = a.epoch;
                    hb[u] = ~0u;
                }
            }
        }
        rank[u] = hb[u] != ~0u ? atomicAdd(&s_at[(x >> a.row_bits) * 2 + (write ? 0 : 1)], 1u) : 0u;
    }
    __syncthreads();
    // thread j owns buckets [j * per, (j + 1) * per)
    const uint32_t per = (a.nb + kBinBlock - 1) / kBinBlock, b0 = threadIdx.x * per;
    uint2 cnt[kPer];
    uint32_t sum = 0, writes = 0, total;
#pragma unroll
    for (uint32_t j = 0; j < kPer; ++j) {
        cnt[j] = (j < per && b0 + j < a.nb) ? reinterpret_cast<const uint2 *>(s_at)[b0 + j] : make_uint2(0u, 0u);
        sum += cnt[j].x + cnt[j].y;
        if (cnt[j].x + cnt[j].y > a.long_run &&
            atomicAdd(&a.marks[kMarkLong + b0 + j], cnt[j].x + cnt[j].y) + cnt[j].x + cnt[j].y > a.hot)
            a.marks[kMarkHot] = 1;
        writes += cnt[j].x;
    }
    if (__ballot(writes != 0) && threadIdx.x % 64 == 0) a.marks[kMarkWritten] = a.epoch;
    uint32_t run = block_exclusive_sum(sum, tile.wt, &total);
    uint32_t *off = a.off + (uint64_t)blockIdx.x * (a.nb + 1);
#pragma unroll
    for (uint32_t j = 0; j < kPer; ++j) {
        if (j < per && b0 + j < a.nb) {
            reinterpret_cast<uint2 *>(s_at)[b0 + j] = make_uint2(run, run + cnt[j].x);
            off[b0 + j] = run | (run + cnt[j].x) << 16;
        }
        run += cnt[j].x + cnt[j].y;
    }
    if (threadIdx.x == 0) off[a.nb] = total;
    __syncthreads();
    const uint32_t inner = (1u << a.row_bits) - 1u;
#pragma unroll
    for (uint32_t u = 0; u < P; ++u) {
        if (hb[u] == ~0u) continue;
        const uint32_t x = hb[u] >> 1;
        s_ent[s_at[(x >> a.row_bits) * 2 + (~hb[u] & 1u)] + rank[u]] =
            (x & inner) << (kBinSlotBits + 1) | (hb[u] & 1u) << kBinSlotBits | (u * kBinBlock + threadIdx.x);
    }
    __syncthreads();
    // whole 16-byte vectors: the last one may carry stale words, which stay
    // inside the tile's own part of ent
    uint4 *dst = reinterpret_cast<uint4 *>(a.ent + (uint64_t)blockIdx.x * T);
    const uint4 *from = reinterpret_cast<const uint4 *>(s_ent);
    for (uint32_t j = threadIdx.x; j < (total + 3) / 4; j += kBinBlock) dst[j] = from[j];
}

template <class Source, uint32_t P, uint32_t MaxB>
__global__ __launch_bounds__(kBinBlock, MaxB <= kBinBlock ? 8 : 4) void bin_kernel(BinArgs a, Source src)
{
    __shared__ BinTile<P, MaxB> s_tile;
    if (a.marks[kMarkUnsorted] != a.epoch)
        bin_tile<Source, P, MaxB, true>(a, src, s_tile);
    else
        bin_tile<Source, P, MaxB, false>(a, src, s_tile);
}

// A bucket's runs are read by groups of 16 lanes, one run per group at a time;
// lane l of group g holds the run of tile c0 + l * kRunGroups + g: where it
// starts, its writes and its length, and the transaction of the tile's first slot.
constexpr uint32_t kRunLanes = 16, kRunGroups = kBinBlock / kRunLanes;

struct BinRun {
    uint32_t start, writes, len, t0;
};

// part: all of the tiles (all-ones), or one of kHotParts parts of them; the runs
// of the others have their writes only.
constexpr uint32_t kHotParts = kRunLanes, kAllParts = ~0u;
__device__ __forceinline__ BinRun bin_run(const BinArgs &a, uint32_t b, uint32_t c0, uint32_t part)
{
    const uint32_t tile = c0 + (threadIdx.x % kRunLanes) * kRunGroups + threadIdx.x / kRunLanes;
    BinRun r = {0u, 0u, 0u, 0u};
    if (tile < a.tiles) {
        const uint32_t *o = a.off + (uint64_t)tile * (a.nb + 1) + b;
        const uint32_t at = o[0] & 0xffffu, end = o[1] & 0xffffu;
        r.start = bin_run_start(tile, a.tile_bits, at, end);
        r.writes = (o[0] >> 16) - at;
        r.len = part == kAllParts || part == threadIdx.x % kRunLanes ? end - at : 0u;
        r.t0 = bin_txn(a, tile << a.tile_bits);
    }
    return r;
}

// The W minimum of each row of a bucket (all-ones: no writer).
template <typename W>
struct RowArray {  // rows [lo, lo + n)
    W *s_w;
    uint32_t lo, n;
    __device__ __forceinline__ bool holds(uint32_t row) const { return row - lo < n; }
    __device__ __forceinline__ void write(uint32_t row, W me) const { atomicMin(&s_w[row - lo], me); }
    __device__ __forceinline__ W minimum(uint32_t row) const { return s_w[row - lo]; }
};

// s_key: row, all-ones = empty.  A row is entered within kProbes slots of its
// own, or *s_full is set and the bucket is left to more shares or the arrays:
// probing always ends, and a lookup needs no more steps either.  The table holds
// share number `share` of `shares` (a power of two) of the rows.
template <typename W>
struct RowHash {
    static constexpr uint32_t kProbes = 64;
    // two blocks per CU: 64 KB, or 75 with 12 bytes per slot
    static constexpr uint32_t kSlots = sizeof(W) == 4 ? kBinHashSlots : 6400;
    uint32_t *s_key, *s_full;
    W *s_w;
    uint32_t shares, share;
    static constexpr bool kMask = (kSlots & (kSlots - 1)) == 0;
    static __device__ __forceinline__ uint32_t slot(uint32_t row)
    {
        const uint32_t h = row * kBinMul >> 16;
        return kMask ? h & (kSlots - 1) : h * kSlots >> 16;
    }
    static __device__ __forceinline__ uint32_t next(uint32_t h)
    {
        return kMask ? (h + 1) & (kSlots - 1) : h + 1 < kSlots ? h + 1 : 0u;
    }
    __device__ __forceinline__ void clear() const
    {
        for (uint32_t r = threadIdx.x; r < kSlots; r += kBinBlock) {
            s_key[r] = ~0u;
            s_w[r] = (W)~(W)0;
        }
        if (threadIdx.x == 0) *s_full = 0u;
    }
    __device__ __forceinline__ bool holds(uint32_t row) const
    {
        return sizeof(W) == 4 || shares == 1 || (row * 0x85EBCA6Bu >> 24 & (shares - 1)) == share;
    }
    __device__ __forceinline__ void write(uint32_t row, W me) const
    {
        uint32_t h = slot(row);
        for (uint32_t p = 0; p < kProbes; ++p) {
            const uint32_t k = atomicCAS(&s_key[h], ~0u, row);
            if (k == ~0u || k == row) {
                atomicMin(&s_w[h], me);
                return;
            }
            h = next(h);
        }
        *s_full = 1u;
    }
    __device__ __forceinline__ W minimum(uint32_t row) const
    {
        uint32_t h = slot(row);
        for (uint32_t p = 0; p < kProbes; ++p) {
            const uint32_t k = s_key[h];
            if (k == row) return s_w[h];
            if (k == ~0u) break;
            h = next(h);
        }
        return (W)~(W)0;
    }
};

// One pass over bucket b's entries of the tiles [c0, c0 + kBinBlock), four
// runs' first 32 entries in flight per group.  MARK false: the W minima of the
// rows that `rows` holds, from the runs' writes; MARK true: the flags from them.
// The priority is the position (u32) or, with TIDs out of order, TID << 24 |
// position (u64).
// DIRECT: slot-major and no narrower than a tile, so a slot's transaction is
// its tile's first plus its place, once around at most.
template <typename W, class Rows, bool MARK, bool DIRECT>
__device__ __forceinline__ void bin_pass(const BinArgs &a, const BinRun &mine, uint32_t c0, const Rows &rows)
{
    constexpr uint32_t U = 4, kSlot = (1u << kBinSlotBits) - 1u;
    const uint32_t g = threadIdx.x / kRunLanes, l = threadIdx.x % kRunLanes;
    const int base_lane = (int)(__lane_id() & ~(kRunLanes - 1));
    // the transaction of an entry of the tile whose first is t0
    auto txn = [&](uint32_t x, uint32_t t0, uint32_t tile) -> uint32_t {
        if (!DIRECT) return bin_txn(a, (tile << a.tile_bits) + (x & kSlot));
        const uint32_t t = t0 + (x & kSlot);
        return t < a.width ? t : t - a.width;
    };
    auto looked_at = [&](uint32_t x) -> bool { return rows.holds(x >> (kBinSlotBits + 1)); };
    const uint32_t entries = MARK ? mine.len : mine.writes;  // what the pass reads of a run
    auto one = [&](uint32_t x, uint32_t t, W me) {
        const uint32_t r = x >> (kBinSlotBits + 1);
        if (!MARK) {
            rows.write(r, me);
            return;
        }
        const W w = rows.minimum(r);
        if ((x >> kBinSlotBits) & 1u) {
            if (w < me) a.doomed[t] = a.epoch;
        } else if (w < me) {
            a.raw_flag[t] = a.epoch;
        } else if (w > me && w != (W)~(W)0) {
            a.war_flag[w & (W)kPosMask] = a.epoch;
        }
    };
    // up to four entries; by TID, whose loads are all in flight
    auto four = [&](const uint32_t *x, const bool *in, const uint32_t *t0, const uint32_t *tile) {
        if (sizeof(W) == 4) {
#pragma unroll
            for (uint32_t k = 0; k < 4; ++k) {
                if (!in[k] || !looked_at(x[k])) continue;
                const uint32_t t = txn(x[k], t0[k], tile[k]);
                one(x[k], t, (W)t);
            }
            return;
        }
        uint32_t t[4], tid[4];
        bool use[4];
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) {
            use[k] = in[k] && looked_at(x[k]);
            t[k] = use[k] ? txn(x[k], t0[k], tile[k]) : 0u;
            tid[k] = a.tids[t[k]];
        }
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k)
            if (use[k]) one(x[k], t[k], (W)((unsigned long long)tid[k] << kTidShift | t[k]));
    };
    const uint32_t left = a.tiles - c0;
    const uint32_t nj = left >= kBinBlock ? kRunLanes : (left + kRunGroups - 1) / kRunGroups;
    for (uint32_t j0 = 0; j0 < nj; j0 += U) {
        uint32_t t0[2 * U], tile[2 * U], x[2 * U], longest = 0;
        bool in[2 * U];
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
            const uint32_t s = __shfl(mine.start, base_lane + (int)(j0 + u));
            const uint32_t len = __shfl(entries, base_lane + (int)(j0 + u));
            t0[2 * u] = t0[2 * u + 1] = DIRECT ? __shfl(mine.t0, base_lane + (int)(j0 + u)) : 0u;
            tile[2 * u] = tile[2 * u + 1] = c0 + (j0 + u) * kRunGroups + g;
            longest = max(longest, len);
            // unconditional loads (a run's first entry when idle, entry 0 of an empty run)
            in[2 * u] = l < len;
            in[2 * u + 1] = l + kRunLanes < len;
            x[2 * u] = a.ent[s + (in[2 * u] ? l : 0u)];
            x[2 * u + 1] = a.ent[s + (in[2 * u + 1] ? l + kRunLanes : 0u)];
        }
#pragma unroll
        for (uint32_t k = 0; k < 2 * U; k += 4) four(x + k, in + k, t0 + k, tile + k);
        if (!__ballot(longest > 2 * kRunLanes)) continue;
        // the rest of long runs, eight loads in flight (a hot row's run is
        // hundreds of entries: one at a time it took four times as long)
#pragma unroll 1
        for (uint32_t u = 0; u < U; ++u) {
            const uint32_t s = __shfl(mine.start, base_lane + (int)(j0 + u));
            const uint32_t len = __shfl(entries, base_lane + (int)(j0 + u));
            const uint32_t first = __shfl(mine.t0, base_lane + (int)(j0 + u));
#pragma unroll 1
            for (uint32_t e = l + 2 * kRunLanes; e < len; e += 8 * kRunLanes) {
#pragma unroll
                for (uint32_t v = 0; v < 8; ++v) {
                    const uint32_t at = e + v * kRunLanes;
                    in[v] = at < len;
                    x[v] = a.ent[s + (in[v] ? at : 0u)];
                    t0[v] = first;
                    tile[v] = c0 + (j0 + u) * kRunGroups + g;
                }
#pragma unroll
                for (uint32_t k = 0; k < 8; k += 4) four(x + k, in + k, t0 + k, tile + k);
            }
        }
    }
}

// Both passes; false, with nothing flagged, if a hash table filled up.
template <typename W, class Rows, bool DIRECT>
__device__ __forceinline__ bool bin_passes(const BinArgs &a, uint32_t b, const BinRun &first, const Rows &rows,
                                           uint32_t part, const uint32_t *s_full = nullptr)
{
    __syncthreads();
    for (uint32_t c0 = 0; c0 < a.tiles; c0 += kBinBlock)
        bin_pass<W, Rows, false, DIRECT>(a, c0 ? bin_run(a, b, c0, part) : first, c0, rows);
    __syncthreads();
    const bool ok = !s_full || *s_full == 0u;
    if (ok)
        for (uint32_t c0 = 0; c0 < a.tiles; c0 += kBinBlock)
            bin_pass<W, Rows, true, DIRECT>(a, c0 ? bin_run(a, b, c0, part) : first, c0, rows);
    __syncthreads();
    return ok;
}

template <typename W, bool DIRECT>
__device__ __forceinline__ void bin_array(const BinArgs &a, uint32_t b, const BinRun &first, W *s_w, uint32_t cap,
                                          uint32_t part)
{
    for (uint32_t lo = 0; lo < (1u << a.row_bits); lo += cap) {
        const uint32_t n = min(1u << a.row_bits, cap);
        for (uint32_t r = threadIdx.x; r < n; r += kBinBlock) s_w[r] = (W)~(W)0;
        bin_passes<W, RowArray<W>, DIRECT>(a, b, first, RowArray<W>{s_w, lo, n}, part);
    }
}

// A bucket through hash tables: of all its rows, or of as many shares of them
// as its writes ask for, fewer than the array needs.  False if there is none.
template <typename W, bool DIRECT>
__device__ __forceinline__ bool bin_hash(const BinArgs &a, uint32_t b, const BinRun &first, unsigned long long *s_mem,
                                         uint32_t *s_wt, uint32_t *s_full, uint32_t part)
{
    W *s_w = reinterpret_cast<W *>(s_mem);
    uint32_t *s_key = reinterpret_cast<uint32_t *>(s_w + RowHash<W>::kSlots);
    uint32_t shares = 1, most = 1;
    if (sizeof(W) > 4) {
        most = (1u << a.row_bits) / (kBinRows / 2) / 2;
        uint32_t writes = first.writes, all;
        for (uint32_t c0 = kBinBlock; c0 < a.tiles; c0 += kBinBlock) writes += bin_run(a, b, c0, part).writes;
        (void)block_exclusive_sum(writes, s_wt, &all);
        while (shares < most && all / shares > RowHash<W>::kSlots / 8 * 7) shares *= 2;
    }
    for (; shares <= most; shares *= 2) {
        bool ok = true;
        for (uint32_t share = 0; ok && share < shares; ++share) {
            const RowHash<W> rows = {s_key, s_full, s_w, shares, share};
            rows.clear();
            ok = bin_passes<W, RowHash<W>, DIRECT>(a, b, first, rows, part, s_full);
        }
        if (ok) return true;
    }
    return false;
}

// A bucket's flags, or one part's of them.
template <bool HASH>
__device__ __forceinline__ void bin_bucket(const BinArgs &a, uint32_t b, uint32_t part, bool by_tid,
                                           unsigned long long *s_mem, uint32_t *s_wt, uint32_t *s_full)
{
    const BinRun first = bin_run(a, b, 0, part);
    const auto flags = [&](auto zero, auto is_direct) {
        using W = decltype(zero);
        constexpr bool D = decltype(is_direct)::value;
        if constexpr (HASH)
            if (bin_hash<W, D>(a, b, first, s_mem, s_wt, s_full, part)) return;
        bin_array<W, D>(a, b, first, reinterpret_cast<W *>(s_mem), (uint32_t)(kBinRows * 4 / sizeof(W)), part);
    };
    if (by_tid) flags(0ull, std::false_type());
    else if (!a.rm && a.width >= (1u << a.tile_bits)) flags(0u, std::true_type());
    else flags(0u, std::false_type());
}

// One block per bucket that is not hot, then blocks that share the hot ones'
// flags: each takes one of 16 parts of a hot bucket's tiles at a time, and
// finds the bucket's minima for itself, whose writes are few as a rule (where
// they are many the filter has dropped most of the run).  Two calls of
// bin_bucket rather than one: what the second keeps does not spill in the first
// (92 us at Zipf 0.99, 98 to 112 with one).
constexpr uint32_t kHotBlocks = 256;
template <bool HASH>
__global__ __launch_bounds__(kBinBlock, 8) void bin_flags_kernel(BinArgs a)
{
    // TIDs out of order are compared as they are, 64 bits a row
    constexpr uint32_t kMem = HASH ? RowHash<unsigned long long>::kSlots * 12 / 8 : kBinRows / 2;
    __shared__ unsigned long long s_mem[kMem];
    __shared__ uint32_t s_wt[kBinBlock / 64], s_full, s_bucket;
    const bool written = a.marks[kMarkWritten] == a.epoch, by_tid = a.marks[kMarkUnsorted] == a.epoch;
    if (blockIdx.x < a.nb) {
        // blocks of one XCD take neighbouring buckets, whose runs and table
        // entries share cache lines
        const uint32_t x = blockIdx.x;
        const uint32_t b = a.nb >= 8 ? (x & 7u) * (a.nb / 8) + (x >> 3) : x;
        // without a write there are no conflicts
        if (written && a.marks[kMarkLong + b] <= a.hot)
            bin_bucket<HASH>(a, b, kAllParts, by_tid, s_mem, s_wt, &s_full);
        return;
    }
    if (!written || a.marks[kMarkHot] == 0) return;
    // thread j looks after buckets [j * per, (j + 1) * per), at most 8
    const uint32_t per = (a.nb + kBinBlock - 1) / kBinBlock;
    uint32_t hot = 0, n;
    for (uint32_t j = 0; j < per; ++j) {
        const uint32_t k = threadIdx.x * per + j;
        hot |= (uint32_t)(k < a.nb && a.marks[kMarkLong + k] > a.hot) << j;
    }
    const uint32_t before = block_exclusive_sum((uint32_t)__popc(hot), s_wt, &n);
    for (uint32_t w = blockIdx.x - a.nb; w < n * kHotParts; w += kHotBlocks) {
        uint32_t at = before;
        for (uint32_t j = 0; j < per; ++j)
            if ((hot >> j) & 1u && at++ == w / kHotParts) s_bucket = threadIdx.x * per + j;
        __syncthreads();
        bin_bucket<HASH>(a, s_bucket, w % kHotParts, by_tid, s_mem, s_wt, &s_full);
        __syncthreads();
    }
}

// a: the caller's part of the arguments; `f` must fit `buf` (bin_fits).
// check_order false: a kernel before has set the order mark if need be.
template <class Source>
hipError_t launch_bin(const Source &src, BinArgs a, const BinShape &f, const BinBuffers &buf, const EpochTag &e,
                      DeviceCounters *ctr, bool zero_counts, bool clear, bool check_order, hipStream_t s)
{
    a.mask = f.mask;
    a.row_bits = f.row_bits;
    a.nb = f.buckets;
    a.tiles = f.tiles;
    a.tile_bits = f.tile_bits;
    a.per.d = a.width;
    a.per.m = a.per.d > 1 ? (uint32_t)((1ull << 32) / a.per.d) : ~0u;
    a.epoch = e.epoch;
    a.ent = buf.ent;
    a.off = buf.off;
    a.marks = buf.marks;
    // four times a bucket's share of a tile, and no fewer than 64; what a block
    // goes through in the time of a few ordinary buckets
    a.long_run = std::max(64u, (4u << f.tile_bits) / f.buckets);
    a.hot = (1u << 13) + 2 * (a.n_ops / f.buckets);
    a.ctr = ctr;
    if (check_order)
        hipLaunchKernelGGL(bin_order_kernel, dim3((a.B + 4 * kOrderBlock - 1) / (4 * kOrderBlock)), dim3(kOrderBlock),
                           0, s, a, zero_counts, clear);
    const dim3 tiles(f.tiles), blk(kBinBlock);
    if (f.tile_bits < kBinSlotBits) {
        hipLaunchKernelGGL((bin_kernel<Source, 4, kBinBlock>), tiles, blk, 0, s, a, src);
    } else if constexpr (!Source::kSmallTiles) {
        if (f.buckets <= kBinBlock)
            hipLaunchKernelGGL((bin_kernel<Source, 16, kBinBlock>), tiles, blk, 0, s, a, src);
        else
            hipLaunchKernelGGL((bin_kernel<Source, 16, 8192>), tiles, blk, 0, s, a, src);
    }
    if (f.row_bits > kBinRowBits)
        hipLaunchKernelGGL(bin_flags_kernel<true>, dim3(f.buckets + kHotBlocks), blk, 0, s, a);
    else
        hipLaunchKernelGGL(bin_flags_kernel<false>, dim3(f.buckets + kHotBlocks), blk, 0, s, a);
    return hipGetLastError();
}

}  // namespace
}  // namespace ltpg
