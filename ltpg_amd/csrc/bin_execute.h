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
//            bucket with LDS counters, places them bucket by bucket in LDS and
//            writes the tile out in that order, with the start of each
//            bucket's run (16 bits) in a table;
//   flags    one block per bucket: reads the bucket's run of every tile twice,
//            first into the W minima of its rows in LDS, then setting the
//            fast form's flags from them: a writer behind the minimum is
//            doomed; a reader behind it has raw; a reader ahead of it gives
//            the minimum writer war.
// A row's bucket is the top bits of row * odd mod 2^K (a bijection), so ranges
// of hot rows spread over the buckets.  An entry is 4 bytes -- row within the
// bucket, is-write, slot within the tile; the tile gives the
// rest -- so no TID, position or counting pass goes through memory: the batch
// is read once, and 4 bytes per operation written once and read twice (the
// second time mostly from the L2).
//
// The in-tile filter: writers enter (position, row) into a direct-mapped LDS
// table with a 64-bit minimum.  An operation that finds its own row there
// under a lower position is behind a writer: a write has waw, a read raw, and
// neither can matter to any other transaction (it is not its row's minimum
// writer, and as a reader it is behind that minimum, so gives no war).  It is
// flagged at once and leaves the batch, which keeps a skewed epoch's hot rows
// from filling one bucket.  Only with ordered TIDs.
//
// The minima of a bucket sit in an array by row when it has at most
// 2^kBinRowBits rows; buckets of more rows (up to 2^kBinHashBits: many rows
// against few operations) use a hash table of the rows written, or, where those
// fill it, the array once per part of their rows.
//
// 2^20 transactions x 16 ops on 10M rows: 486 us on the registers (285
// registration, 202 read marking) -> 189 us at Zipf 0.6 (order 5, bin 62,
// flags 122), 515 -> 160 us at Zipf 0.99.  The bin kernel moves 268 MB at 4.3
// TB/s; the flags kernel is bound by instruction issue (1M runs of 16 entries,
// half of the lanes idle; 130 us with each entry's transaction by division)
// and, at Zipf 0.6, by its 9M scattered flag bytes (58 us without them).
//
// A Source gives the operation of op slot i: load(i) its words (every slot
// below n_ops may be loaded), decode() whether it registers, its row (< 2^32),
// whether it is a write, and the slot's range errors.  kSmallTiles: its shapes
// are tiles of 4 slots per thread and at most 1024 buckets.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

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
    uint16_t *off;         // [tiles][nb + 1] start of each bucket's run in the tile
    uint32_t *unsorted;    // epoch number of the last epoch whose TIDs were out of order
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

// With `clear` (the epoch that keeps no state between calls) also the flags of
// the block's transactions and the range errors start over.
constexpr uint32_t kOrderBlock = 256;
__global__ __launch_bounds__(kOrderBlock) void bin_order_kernel(BinArgs a, bool zero_counts, bool clear)
{
    if (zero_counts && blockIdx.x == 0) zero_epoch_counts(a.ctr, kOrderBlock);
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
    if (out) *a.unsorted = a.epoch;
}

template <class Source, uint32_t P, uint32_t MaxB>
__global__ __launch_bounds__(kBinBlock, MaxB <= kBinBlock ? 8 : 4) void bin_kernel(BinArgs a, Source src)
{
    constexpr uint32_t T = P * kBinBlock, kFilter = T / 2;
    constexpr uint32_t kPer = MaxB / kBinBlock;  // buckets per thread at most
    constexpr uint32_t G = 4;                    // slots whose loads are in flight per thread
    __shared__ __align__(16) uint32_t s_ent[T];  // the filter first, then the tile in bucket order
    __shared__ uint32_t s_at[MaxB];              // counts, then starts
    __shared__ uint32_t s_wt[kBinBlock / 64];
    unsigned long long *s_min = reinterpret_cast<unsigned long long *>(s_ent);
    const uint32_t base = blockIdx.x * T + threadIdx.x;
    const bool fold = *a.unsorted != a.epoch;
    for (uint32_t k = threadIdx.x; k < kFilter; k += kBinBlock) s_min[k] = ~0ull;
    for (uint32_t b = threadIdx.x; b < a.nb; b += kBinBlock) s_at[b] = 0;
    __syncthreads();
    uint32_t hb[P];  // hashed row << 1 | is-write, or all-ones: nothing to register
    uint32_t bad = 0;
#pragma unroll
    for (uint32_t g = 0; g < P; g += G) {
        typename Source::Raw raw[G];
#pragma unroll
        for (uint32_t u = 0; u < G; ++u) {
            const uint32_t i = base + (g + u) * kBinBlock;
            raw[u] = src.load(a, i < a.n_ops ? i : 0u);
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
            if (fold && use && write)
                atomicMin(&s_min[(x ^ (x >> 12)) & (kFilter - 1)], (unsigned long long)bin_txn(a, i) << 32 | x);
        }
    }
    if (bad) atomicAdd(&a.ctr->range_errors, bad);
    __syncthreads();
    uint32_t rank[P];
#pragma unroll
    for (uint32_t u = 0; u < P; ++u) {
        const uint32_t x = hb[u] >> 1;
        const bool write = hb[u] & 1u;
        if (fold && hb[u] != ~0u) {
            const unsigned long long v = s_min[(x ^ (x >> 12)) & (kFilter - 1)];
            if ((uint32_t)v == x) {
                const uint32_t t = bin_txn(a, base + u * kBinBlock);
                if ((uint32_t)(v >> 32) < t) {
                    if (write)
                        a.doomed[t] = a.epoch;
                    else
                        a.raw_flag[t] = a.epoch;
                    hb[u] = ~0u;
                }
            }
        }
        rank[u] = hb[u] != ~0u ? atomicAdd(&s_at[x >> a.row_bits], 1u) : 0u;
    }
    __syncthreads();
    // thread j owns buckets [j * per, (j + 1) * per)
    const uint32_t per = (a.nb + kBinBlock - 1) / kBinBlock, b0 = threadIdx.x * per;
    uint32_t cnt[kPer], sum = 0, total;
#pragma unroll
    for (uint32_t j = 0; j < kPer; ++j) {
        cnt[j] = (j < per && b0 + j < a.nb) ? s_at[b0 + j] : 0u;
        sum += cnt[j];
    }
    uint32_t run = block_exclusive_sum(sum, s_wt, &total);
    uint16_t *off = a.off + (uint64_t)blockIdx.x * (a.nb + 1);
#pragma unroll
    for (uint32_t j = 0; j < kPer; ++j) {
        if (j < per && b0 + j < a.nb) {
            s_at[b0 + j] = run;
            off[b0 + j] = (uint16_t)run;
        }
        run += cnt[j];
    }
    if (threadIdx.x == 0) off[a.nb] = (uint16_t)total;
    __syncthreads();
    const uint32_t inner = (1u << a.row_bits) - 1u;
#pragma unroll
    for (uint32_t u = 0; u < P; ++u) {
        if (hb[u] == ~0u) continue;
        const uint32_t x = hb[u] >> 1;
        s_ent[s_at[x >> a.row_bits] + rank[u]] =
            (x & inner) << (kBinSlotBits + 1) | (hb[u] & 1u) << kBinSlotBits | (u * kBinBlock + threadIdx.x);
    }
    __syncthreads();
    // whole 16-byte vectors: the last one may carry stale words, which stay
    // inside the tile's own part of ent
    uint4 *dst = reinterpret_cast<uint4 *>(a.ent + (uint64_t)blockIdx.x * T);
    const uint4 *from = reinterpret_cast<const uint4 *>(s_ent);
    for (uint32_t j = threadIdx.x; j < (total + 3) / 4; j += kBinBlock) dst[j] = from[j];
}

// A bucket's runs are read by groups of 16 lanes, one run per group at a time;
// lane l of group g holds the run of tile c0 + l * kRunGroups + g: where it
// starts, its length, and the transaction of the tile's first slot.
constexpr uint32_t kRunLanes = 16, kRunGroups = kBinBlock / kRunLanes;

struct BinRun {
    uint32_t start, len, t0;
};

__device__ __forceinline__ BinRun bin_run(const BinArgs &a, uint32_t b, uint32_t c0)
{
    const uint32_t tile = c0 + (threadIdx.x % kRunLanes) * kRunGroups + threadIdx.x / kRunLanes;
    BinRun r = {0u, 0u, 0u};
    if (tile < a.tiles) {
        const uint16_t *o = a.off + (uint64_t)tile * (a.nb + 1) + b;
        r.start = bin_run_start(tile, a.tile_bits, o[0], o[1]);
        r.len = (uint32_t)o[1] - o[0];
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
// own, or *s_full is set and the bucket is left to the arrays: probing always
// ends, and a lookup needs no more steps either.
struct RowHash {
    static constexpr uint32_t kProbes = 64;
    uint32_t *s_key, *s_w, *s_full;
    static __device__ __forceinline__ uint32_t slot(uint32_t row) { return (row * kBinMul >> 16) & (kBinHashSlots - 1); }
    __device__ __forceinline__ bool holds(uint32_t) const { return true; }
    __device__ __forceinline__ void write(uint32_t row, uint32_t me) const
    {
        uint32_t h = slot(row);
        for (uint32_t p = 0; p < kProbes; ++p) {
            const uint32_t k = atomicCAS(&s_key[h], ~0u, row);
            if (k == ~0u || k == row) {
                atomicMin(&s_w[h], me);
                return;
            }
            h = (h + 1) & (kBinHashSlots - 1);
        }
        *s_full = 1u;
    }
    __device__ __forceinline__ uint32_t minimum(uint32_t row) const
    {
        uint32_t h = slot(row);
        for (uint32_t p = 0; p < kProbes; ++p) {
            const uint32_t k = s_key[h];
            if (k == row) return s_w[h];
            if (k == ~0u) break;
            h = (h + 1) & (kBinHashSlots - 1);
        }
        return ~0u;
    }
};

// One pass over bucket b's entries of the tiles [c0, c0 + kBinBlock), four
// runs' first 32 entries in flight per group.  MARK false: the W minima of the
// rows that `rows` holds; MARK true: the flags from them.  The priority is the
// position (u32) or, with TIDs out of order, TID << 24 | position (u64).
// DIRECT: slot-major and no narrower than a tile, so a slot's transaction is
// its tile's first plus its place, once around at most.
template <typename W, class Rows, bool MARK, bool DIRECT>
__device__ __forceinline__ void bin_pass(const BinArgs &a, const BinRun &mine, uint32_t c0, const Rows &rows)
{
    constexpr uint32_t U = 4, kSlot = (1u << kBinSlotBits) - 1u;
    const uint32_t g = threadIdx.x / kRunLanes, l = threadIdx.x % kRunLanes;
    const int base_lane = (int)(__lane_id() & ~(kRunLanes - 1));
    auto one = [&](uint32_t x, uint32_t t0, uint32_t tile) {
        const uint32_t r = x >> (kBinSlotBits + 1);
        const bool wr = (x >> kBinSlotBits) & 1u;
        if ((!MARK && !wr) || !rows.holds(r)) return;
        uint32_t t;
        if (DIRECT) {
            t = t0 + (x & kSlot);
            t = min(t, t - a.width);  // around: t - width wraps below zero otherwise
        } else {
            t = bin_txn(a, (tile << a.tile_bits) + (x & kSlot));
        }
        const W me = sizeof(W) == 4 ? (W)t : (W)((unsigned long long)a.tids[t] << kTidShift | t);
        if (!MARK) {
            rows.write(r, me);
            return;
        }
        const W w = rows.minimum(r);
        if (wr) {
            if (w < me) a.doomed[t] = a.epoch;
        } else if (w < me) {
            a.raw_flag[t] = a.epoch;
        } else if (w > me && w != (W)~(W)0) {
            a.war_flag[w & (W)kPosMask] = a.epoch;
        }
    };
    const uint32_t left = a.tiles - c0;
    const uint32_t nj = left >= kBinBlock ? kRunLanes : (left + kRunGroups - 1) / kRunGroups;
    for (uint32_t j0 = 0; j0 < nj; j0 += U) {
        uint32_t s[U], len[U], t0[U], x[U][2];
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
            s[u] = __shfl(mine.start, base_lane + (int)(j0 + u));
            len[u] = __shfl(mine.len, base_lane + (int)(j0 + u));
            t0[u] = DIRECT ? __shfl(mine.t0, base_lane + (int)(j0 + u)) : 0u;
            // unconditional loads (a run's first entry when idle, entry 0 of an empty run)
            x[u][0] = a.ent[s[u] + (l < len[u] ? l : 0u)];
            x[u][1] = a.ent[s[u] + (l + kRunLanes < len[u] ? l + kRunLanes : 0u)];
        }
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
            const uint32_t tile = c0 + (j0 + u) * kRunGroups + g;
            if (l < len[u]) one(x[u][0], t0[u], tile);
            if (l + kRunLanes < len[u]) one(x[u][1], t0[u], tile);
            for (uint32_t e = l + 2 * kRunLanes; e < len[u]; e += kRunLanes) one(a.ent[s[u] + e], t0[u], tile);
        }
    }
}

// Both passes; false, with nothing flagged, if a hash table filled up.
template <typename W, class Rows, bool DIRECT>
__device__ __forceinline__ bool bin_passes(const BinArgs &a, uint32_t b, const BinRun &first, const Rows &rows,
                                           const uint32_t *s_full = nullptr)
{
    __syncthreads();
    for (uint32_t c0 = 0; c0 < a.tiles; c0 += kBinBlock)
        bin_pass<W, Rows, false, DIRECT>(a, c0 ? bin_run(a, b, c0) : first, c0, rows);
    __syncthreads();
    const bool ok = !s_full || *s_full == 0u;
    if (ok)
        for (uint32_t c0 = 0; c0 < a.tiles; c0 += kBinBlock)
            bin_pass<W, Rows, true, DIRECT>(a, c0 ? bin_run(a, b, c0) : first, c0, rows);
    __syncthreads();
    return ok;
}

template <typename W, bool DIRECT>
__device__ __forceinline__ void bin_array(const BinArgs &a, uint32_t b, const BinRun &first, W *s_w, uint32_t cap)
{
    for (uint32_t lo = 0; lo < (1u << a.row_bits); lo += cap) {
        const uint32_t n = min(1u << a.row_bits, cap);
        for (uint32_t r = threadIdx.x; r < n; r += kBinBlock) s_w[r] = (W)~(W)0;
        bin_passes<W, RowArray<W>, DIRECT>(a, b, first, RowArray<W>{s_w, lo, n});
    }
}

template <bool HASH>
__global__ __launch_bounds__(kBinBlock, 8) void bin_flags_kernel(BinArgs a)
{
    __shared__ unsigned long long s_w[kBinRows / 2];
    // blocks of one XCD take neighbouring buckets, whose runs and table
    // entries share cache lines
    const uint32_t x = blockIdx.x;
    const uint32_t b = a.nb >= 8 ? (x & 7u) * (a.nb / 8) + (x >> 3) : x;
    const BinRun first = bin_run(a, b, 0);
    uint32_t *s_w32 = reinterpret_cast<uint32_t *>(s_w);
    if (*a.unsorted == a.epoch) {
        bin_array<unsigned long long, false>(a, b, first, s_w, kBinRows / 2);
        return;
    }
    const bool direct = !a.rm && a.width >= (1u << a.tile_bits);
    if constexpr (HASH) {
        __shared__ uint32_t s_full;
        for (uint32_t r = threadIdx.x; r < 2 * kBinHashSlots; r += kBinBlock) s_w32[r] = ~0u;
        if (threadIdx.x == 0) s_full = 0;
        const RowHash rows = {s_w32, s_w32 + kBinHashSlots, &s_full};
        if (direct ? bin_passes<uint32_t, RowHash, true>(a, b, first, rows, &s_full)
                   : bin_passes<uint32_t, RowHash, false>(a, b, first, rows, &s_full))
            return;
    }
    if (direct)
        bin_array<uint32_t, true>(a, b, first, s_w32, kBinRows);
    else
        bin_array<uint32_t, false>(a, b, first, s_w32, kBinRows);
}

// a: the caller's part of the arguments; `f` must fit `buf` (bin_fits).
// check_order false: a kernel before has set *buf.unsorted if need be.
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
    a.unsorted = buf.unsorted;
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
        hipLaunchKernelGGL(bin_flags_kernel<true>, dim3(f.buckets), blk, 0, s, a);
    else
        hipLaunchKernelGGL(bin_flags_kernel<false>, dim3(f.buckets), blk, 0, s, a);
    return hipGetLastError();
}

}  // namespace
}  // namespace ltpg
