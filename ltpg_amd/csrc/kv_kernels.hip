// kv_kernels.hip - key-value execute / check / readout / write-back kernels
// for gfx950.
//
// Replaces KERNEL_EXECUTE / KERNEL_CHECK / KERNEL_WRITEBACK of
// LTPG/YCSB/0/ycsb.cu:9-58 and the per-op bodies of YCSB/0/Execute.h:11-252
// and Genericfunction.h:31-158.
//
// Mapping.  The batch is slot-major (slot s of transaction t at [s*B + t],
// the reference's LOC[B*op + NO]).  One lane owns one transaction and walks
// its slots, so every slot-level load of a wave is 64 consecutive elements
// (coalesced), per-transaction state stays in registers (no per-op
// atomicAdd on raw/war/waw[NO]), and the commit decision is fused into the
// check: a wave64 ballot of the commit predicate is one 64-bit word of the
// commit bitmap.
//
// Registers.  A row's R and W registers sit at rl.r(row) and rl.w(row)
// (RegLayout: interleaved pairs or two arrays), each a u64 priority
//     tag:8 | TID:32 | batch position:24
// where tag = 255 - epoch (epochs 1..255; the library refills every register
// with all-ones when the epoch counter wraps).  Lower value = higher
// priority, and every value of an older epoch is larger than every value of
// the current one, so a single atomicMin both registers and evicts a stale
// value, and "register < my priority" already implies "registered in this
// epoch" -- stale registers never produce a conflict.
//
// Early waw.  atomicMin returns the old value.  A write whose registration
// finds a lower priority already there has waw > 0; a write that lowers the
// register from v displaces the writer whose position is in v, which then
// has waw > 0.  Every writer except the minimum one is caught by exactly one
// of the two (the first registration that goes below a writer sees exactly
// that writer's value), so after EXECUTE the doomed[] bytes mark precisely
// the transactions with waw > 0, and CHECK only walks the others.
//
// Field copies.  A field is field_words u32 words inside a row-major record
// whose fields start at multiples of field_stride words (field_stride =
// field_words rounded up to 16 words = 64 bytes for fields of 64 bytes or
// more, so a 100-byte field touches exactly two 64-byte segments).  A wave
// moves the fields of its ops cooperatively, each op's addresses fetched from
// its owner lane: in CHECK's read-out and in WRITEBACK through a list in LDS,
// 16 bytes per lane and as many lanes per field as it has 16-byte pieces
// (stage_flush; fields of less than 16 bytes one lane each), or, with the
// LANE_COPY shape, one lane per field (lane_copy); in the counting form's
// read-out LP lanes per op (LP = next power of two >= field_words, at most
// 64), fetched by __shfl.
#include <algorithm>

#include "bin_execute.h"
#include "device_common.h"
#include "ltpg_internal.h"

namespace ltpg {
namespace {

constexpr int kBlock = 256;

__device__ __forceinline__ int lane_id() { return (int)__lane_id(); }

// Copy (or read-modify-write) the fields of the active ops of a wave.
// Lane j's op: src_base[src_off + w] (+ delta) -> dst_base[dst_off + w] for
// w < fw.  Requires fw <= LP.  Ops of one call never alias each other
// (different transactions of one wave never write one row in the same
// slot), so the loads of U steps are issued before their stores.  A lane
// always handles the same word positions of the same transaction, so
// successive calls on one row by one transaction are ordered.
template <int LP, int U>
__device__ __forceinline__ void wave_copy(unsigned long long mask, uint64_t src_off,
                                          uint64_t dst_off, uint32_t delta,
                                          const uint32_t *src_base, uint32_t *dst_base,
                                          uint32_t fw)
{
    constexpr int PER = 64 / LP;  // ops per step
    const int lane = lane_id();
    const int sub = lane / LP;
    const uint32_t w0 = (uint32_t)(lane % LP);
    const bool word_ok = w0 < fw;
#pragma unroll 1
    for (int s0 = 0; s0 < LP; s0 += U) {
        uint32_t v[U];
        uint64_t d[U];
        bool a[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int j = (s0 + u) * PER + sub;
            const uint64_t so = __shfl(src_off, j);
            d[u] = __shfl(dst_off, j);
            const uint32_t dl = __shfl(delta, j);
            a[u] = word_ok && ((mask >> j) & 1ull);
            v[u] = a[u] ? src_base[so + w0] + dl : 0u;
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (a[u]) dst_base[d[u] + w0] = v[u];
    }
}

// Fields wider than 64 words: one op at a time, 64 words per instruction.
__device__ __forceinline__ void wave_copy_wide(unsigned long long mask, uint64_t src_off,
                                               uint64_t dst_off, uint32_t delta,
                                               const uint32_t *src_base, uint32_t *dst_base,
                                               uint32_t fw)
{
    const int lane = lane_id();
    while (mask) {
        const int j = __ffsll((long long)mask) - 1;
        mask &= mask - 1;
        const uint64_t so = __shfl(src_off, j);
        const uint64_t d = __shfl(dst_off, j);
        const uint32_t dl = __shfl(delta, j);
        for (uint32_t w = (uint32_t)lane; w < fw; w += 64) dst_base[d + w] = src_base[so + w] + dl;
    }
}

template <int LP>
__device__ __forceinline__ void copy_fields(unsigned long long mask, uint64_t src_off,
                                            uint64_t dst_off, uint32_t delta,
                                            const uint32_t *src_base, uint32_t *dst_base,
                                            uint32_t fw)
{
    if constexpr (LP == 0)
        wave_copy_wide(mask, src_off, dst_off, delta, src_base, dst_base, fw);
    else
        wave_copy<LP, (LP < 8 ? LP : 8)>(mask, src_off, dst_off, delta, src_base, dst_base, fw);
}

// Commit and attempt counts go to one of kCounterStripes stripes (256 bytes
// apart): thousands of blocks adding to one address serialize in the
// memory-side atomic unit (4096 same-address atomics cost ~50 us on MI355X).
__device__ __forceinline__ void add_counts(DeviceCounters *ctr, uint32_t stripe, uint32_t type,
                                           uint32_t commits, uint32_t attempts)
{
    if (commits) {
        atomicAdd(&ctr->commits[stripe][type], commits);
        atomicAdd(&ctr->totals[stripe][type], (unsigned long long)commits);
    }
    if (attempts) atomicAdd(&ctr->totals[stripe][kAttempts + type], (unsigned long long)attempts);
}

// Per-op decode shared by every phase.
struct Op {
    uint64_t row;
    uint32_t kind;
    uint32_t field;
    uint32_t len;  // rows read: 1 for a read, the clipped range for a scan, 0 otherwise
    bool valid;
};

// A slot's op from its row and meta word.  A scan (kind 3) is valid only if
// its length is at most max_scan; kernels that never look at reads pass 0.
__device__ __forceinline__ Op decode_op(uint64_t row, uint32_t m, uint64_t rows, uint32_t fields,
                                        uint32_t max_scan)
{
    Op o;
    o.row = row;
    o.kind = m & 3u;
    o.field = (m >> 8) & 0xffffu;
    const uint32_t sl = (m >> 24) + 1u;
    o.valid = o.kind != LTPG_KV_NONE && o.row < rows && o.field < fields &&
              (o.kind != LTPG_KV_SCAN || sl <= max_scan);
    const uint64_t left = o.row < rows ? rows - o.row : 0ull;
    o.len = !o.valid || o.kind == LTPG_KV_WRITE ? 0u
            : o.kind == LTPG_KV_READ            ? 1u
                                                : (uint32_t)(sl < left ? sl : left);
    return o;
}

// Loads are unconditional on a clamped index (element 0 of a non-empty batch
// when the lane has no op) and the result is selected afterwards: a load
// under a lane-dependent branch sits in its own basic block and the compiler
// waits for it before the next one, which would serialize the misses.
__device__ __forceinline__ Op load_op(const uint64_t *__restrict__ keys,
                                      const uint32_t *__restrict__ meta, uint64_t i, bool live,
                                      uint64_t rows, uint32_t fields, uint32_t max_scan = 0)
{
    const uint64_t j = live ? i : 0ull;
    const uint32_t m0 = meta[j];
    const uint64_t r0 = keys[j];
    return decode_op(live ? r0 : 0ull, live ? m0 : 0u, rows, fields, max_scan);
}

// Batch layouts.  Slot s of transaction t sits at s * B + t (slot-major,
// the reference's LOC[B*op + NO]) or, with rm, at t * S + s (request-major:
// the served form's staging, where a transaction's slots are one contiguous
// run).  Committed reads always go to the slot-major position.
__device__ __forceinline__ uint64_t op_at(uint32_t s, uint32_t t, uint32_t B, uint32_t S, bool rm)
{
    return rm ? (uint64_t)t * S + s : (uint64_t)s * B + t;
}

__device__ __forceinline__ uint32_t txn_of(uint64_t i, uint32_t B, uint32_t S, bool rm)
{
    return rm ? (uint32_t)(i / S) : (uint32_t)(i % B);
}

// Zero the per-epoch commit counts (a kernel rather than a memset so the
// epoch can be captured in a graph).
__global__ void reset_epoch_counters_kernel(DeviceCounters *ctr)
{
    zero_epoch_counts(ctr, blockDim.x);
}

// Streaming 16-byte copy, grid-stride.
__global__ void copy_u128_kernel(uint4 *__restrict__ dst, const uint4 *__restrict__ src, uint64_t n)
{
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) dst[i] = src[i];
}

__global__ void fill_u64_kernel(unsigned long long *p, uint64_t n, unsigned long long v)
{
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) p[i] = v;
}

// Registers and flags back to their initial state, all in one kernel with
// 16-byte stores: a replayed run of both workloads starts with 8 arrays of the
// key-value context (two register sets of 10M rows, their flags) and 4 of the
// order-entry one, whose fills took 79 and 29 us one by one.
__global__ __launch_bounds__(256) void fill_set_kernel(FillSet f)
{
    const uint64_t first = (uint64_t)blockIdx.x * 256 + threadIdx.x, step = (uint64_t)gridDim.x * 256;
    for (uint32_t k = 0; k < f.n; k++) {
        const uint32_t v = f.ones[k] ? ~0u : 0u;
        const uint64_t vecs = f.bytes[k] / 16;
        uint4 *p = static_cast<uint4 *>(f.p[k]);
        for (uint64_t i = first; i < vecs; i += step) p[i] = make_uint4(v, v, v, v);
        if (first < f.bytes[k] % 16) reinterpret_cast<uint8_t *>(p + vecs)[first] = (uint8_t)v;
    }
}

// u32 copy, grid-stride; the source may be pinned host memory (the served
// form's staging: a kernel on the epoch's own stream costs one launch, where
// a copy-engine transfer costs a copy call plus a cross-stream event).
__global__ void copy_u32_kernel(uint32_t *__restrict__ dst, const uint32_t *__restrict__ src, uint64_t n)
{
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) dst[i] = src[i];
}

// Publish an epoch's commit bitmaps to pinned host memory, then its sequence
// number with a system-scope release: a host that reads the sequence number
// with an acquire load also reads the bitmaps.  One block.
__global__ void publish_kernel(PublishSet p, uint64_t *seq_out, uint64_t seq)
{
    for (int k = 0; k < 5; k++)
        for (uint32_t w = threadIdx.x; w < p.n[k]; w += blockDim.x) p.dst[k][w] = p.src[k][w];
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x == 0) __hip_atomic_store(seq_out, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// A small result to pinned host memory: the last block to finish stores the
// sequence number that the host polls.  With the stream's work still running
// the host has the result 2 us (1 KB) to 4 us (128 KB) before a wait for the
// stream alone returns, where that wait and a copy to pageable memory took
// 12 to 14 us more; on an idle stream 8 us against 12 (1 KB), 14 against 61
// (128 KB).  Bound by the PCIe writes and the round trip of the last one.
constexpr uint32_t kReadbackWords = 2048;  // per block
__global__ __launch_bounds__(256) void readback_kernel(uint32_t *__restrict__ dst, const uint32_t *__restrict__ src,
                                                       uint32_t words, uint32_t *blocks, uint64_t *seq_out,
                                                       uint64_t seq)
{
    const uint32_t first = blockIdx.x * kReadbackWords;
    const uint32_t end = min(words, first + kReadbackWords);
    for (uint32_t i = first + 2 * threadIdx.x; i + 1 < end; i += 2 * blockDim.x)
        *reinterpret_cast<uint64_t *>(dst + i) = *reinterpret_cast<const uint64_t *>(src + i);
    if ((end & 1) && threadIdx.x == 0) dst[end - 1] = src[end - 1];
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x) return;
    if (__hip_atomic_fetch_add(blocks, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) + 1 < gridDim.x) return;
    *blocks = 0;
    __hip_atomic_store(seq_out, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// A batch's commit bitmaps into the archive of a run, which may sit in pinned
// host memory, and the device clock into its stamp: one kernel, where a copy
// for each bitmap and one for the stamp were up to six.
// With `reset` the next batch's commit counts and list start over (a run whose
// EXECUTE overlaps the batch before cannot do that there).
__global__ void archive_kernel(PublishSet p, unsigned long long *stamp, DeviceCounters *reset)
{
    if (reset && blockIdx.x == 0) zero_epoch_counts(reset, blockDim.x);
    const uint32_t stride = gridDim.x * blockDim.x;
    for (int k = 0; k < 5; k++)
        for (uint32_t w = blockIdx.x * blockDim.x + threadIdx.x; w < p.n[k]; w += stride) p.dst[k][w] = p.src[k][w];
    __threadfence_system();
    if (stamp && blockIdx.x == 0 && threadIdx.x == 0) *stamp = wall_clock64();
}

// Random-access calibration: n random 8-byte loads, or n random probe +
// atomicMin pairs, over a[0..len).  The sink store is never taken for the
// all-ones contents (it keeps the loads from being optimised away).
__device__ __forceinline__ uint64_t calib_index(uint64_t i, uint64_t len)
{
    i ^= i >> 33;
    i *= 0xff51afd7ed558ccdull;
    i ^= i >> 33;
    i *= 0xc4ceb9fe1a85ec53ull;
    i ^= i >> 33;
    return i % len;
}

__global__ void calib_load_kernel(const unsigned long long *a, uint64_t len, uint64_t n, uint32_t per,
                                  unsigned long long *sink)
{
    const uint64_t base = ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) * per;
    unsigned long long acc = 0;
    for (uint32_t k = 0; k < per; ++k)
        if (base + k < n) acc += a[calib_index(base + k, len)];
    if (acc == 1ull) sink[0] = acc;
}

__global__ void calib_atomic_kernel(unsigned long long *a, uint64_t len, uint64_t n, uint32_t per,
                                    unsigned long long *sink)
{
    const uint64_t base = ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) * per;
    unsigned long long acc = 0;
    for (uint32_t k = 0; k < per; ++k) {
        if (base + k >= n) break;
        unsigned long long *p = &a[calib_index(base + k, len)];
        const unsigned long long me = base + k;
        if (probe(p) > me) acc += atomicMin(p, me);
    }
    if (acc == 1ull) sink[0] = acc;
}

// Cost of a grid-wide barrier, the step a persistent batched kernel would
// take between phases: gridDim.x workgroups (resident together: the kernel
// is launched cooperatively) pass `reps` barriers.  Lane 0 of each
// workgroup reads the generation, arrives on the counter, and the last to
// arrive resets the counter and advances the generation; the others poll
// the generation.  Every poll is bounded: past spin_limit polls the
// workgroup records an error and leaves, so the kernel always ends.
__global__ void grid_barrier_kernel(unsigned int *count, unsigned int *gen, uint32_t reps, uint32_t spin_limit,
                                    unsigned int *err)
{
    __shared__ uint32_t s_stop;
    for (uint32_t r = 0; r < reps; ++r) {
        if (threadIdx.x == 0) {
            uint32_t stop = __hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u;
            const unsigned g = __hip_atomic_load(gen, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT);
            if (!stop) {
                const unsigned arrived =
                    __hip_atomic_fetch_add(count, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
                if (arrived == gridDim.x - 1) {
                    __hip_atomic_store(count, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    __hip_atomic_fetch_add(gen, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
                } else {
                    uint32_t spins = 0;
                    while (__hip_atomic_load(gen, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT) == g) {
                        if (++spins > spin_limit) {
                            __hip_atomic_fetch_or(err, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                            stop = 1;
                            break;
                        }
                        __builtin_amdgcn_s_sleep(1);
                    }
                }
            }
            s_stop = stop;
        }
        __syncthreads();
        if (s_stop) return;
    }
}

// One store per workgroup: the smallest kernel, whose back-to-back launches
// time a kernel boundary.
__global__ void boundary_kernel(unsigned int *p) { if (threadIdx.x == 0) p[blockIdx.x] = blockIdx.x; }

// Device wall-clock stamp (constant-rate counter), one lane.
__global__ void stamp_kernel(unsigned long long *out) { out[threadIdx.x] = wall_clock64(); }

__global__ void fill_u8_kernel(uint8_t *p, uint64_t n, uint8_t v)
{
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) p[i] = v;
}

// Reference initial contents: every word of field c holds c
// (YCSB/0/Database.h:77-86 writes Y_c = c into column c); padding words 0.
__global__ void kv_fill_reference_kernel(uint32_t *table, uint64_t n_words, uint32_t fields,
                                         uint32_t fw, uint32_t fsw)
{
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n_words; i += stride) {
        const uint64_t f = i / fsw;
        const uint32_t w = (uint32_t)(i - f * fsw);
        table[i] = w < fw ? (uint32_t)(f % fields) : 0u;
    }
}

// Dense fields (field_words apart) <-> strided fields (field_stride apart).
__global__ void repack_kernel(const uint32_t *__restrict__ src, uint32_t *__restrict__ dst,
                              uint64_t n_fields, uint32_t fw, uint32_t fsw, int to_strided)
{
    const uint64_t n = n_fields * fw;
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        const uint64_t f = i / fw;
        const uint64_t w = i - f * fw;
        if (to_strided)
            dst[f * fsw + w] = src[i];
        else
            dst[i] = src[f * fsw + w];
    }
}

// Column-major <-> row-major for u32 tables (rows x cols); with T = u64 also
// the request-major -> slot-major transpose of served key-value epochs.
template <typename T>
__global__ void transpose_kernel(const T *__restrict__ src, T *__restrict__ dst, uint64_t rows, uint32_t cols,
                                 int to_row_major)
{
    const uint64_t n = rows * cols;
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        // i indexes the destination
        if (to_row_major) {
            const uint64_t r = i / cols, c = i % cols;
            dst[i] = src[c * rows + r];
        } else {
            const uint64_t c = i / rows, r = i % rows;
            dst[i] = src[r * cols + c];
        }
    }
}

// EXECUTE: register every valid op's priority on R (read) or W (write)
// (read_0 / write_0 -> __REGISTER, YCSB/0/Execute.h:11-53,
// Genericfunction.h:61-100) and record waw by displacement.  The load before
// the atomic skips registrations that cannot lower the register (a register
// only decreases, so even a stale cached value is >= its current value); on
// hot rows this turns a serialized chain of same-address atomics into
// cached loads.
//
// Reads register R only for the counting form.  The fast form needs war
// only for transactions without waw, i.e. for the minimum writer of each row
// they write, and a reader with a lower priority than that writer can flag
// it directly from the W register (kv_mark_reads_kernel).  Random 64-bit
// atomics run at about half the rate of random loads on this part, so
// leaving read ops to a load-only pass halves the atomics of an epoch.
__global__ __launch_bounds__(kBlock) void kv_execute_kernel(
    const uint64_t *__restrict__ keys, const uint32_t *__restrict__ meta,
    const uint32_t *__restrict__ tids, uint32_t B, uint32_t S, uint64_t rows, uint32_t fields,
    unsigned long long *__restrict__ regs, RegLayout rl, uint64_t hot, uint32_t tag,
    uint8_t *__restrict__ doomed, uint8_t epoch, bool reg_reads, bool zero_counts, uint32_t max_scan,
    DeviceCounters *__restrict__ ctr, bool rm)
{
    const uint32_t t = blockIdx.x * kBlock + threadIdx.x;
    const bool live = t < B;
    // the epoch's commit counts start at zero (CHECK adds to them)
    if (zero_counts && blockIdx.x == 0) zero_epoch_counts(ctr, kBlock);
    const unsigned long long me = live ? priority(tag, tids[t], t) : 0ull;
    bool waw = false;
    uint32_t bad = 0;
    for (uint32_t s = 0; s < S; ++s) {
        const Op o = load_op(keys, meta, op_at(s, t, B, S, rm), live, rows, fields, max_scan);
        bad += (o.kind != LTPG_KV_NONE && !o.valid) ? 1u : 0u;
        if (!o.valid) continue;
        if (o.kind == LTPG_KV_WRITE) {
            if (o.row != hot)  // the hot row never registers
                waw |= register_write(&regs[rl.w(o.row)], me, tag, doomed, epoch);
        } else if (reg_reads) {
            for (uint32_t k = 0; k < o.len; ++k)
                if (o.row + k != hot) register_read(&regs[rl.r(o.row + k)], me);
        }
    }
    if (waw) doomed[t] = epoch;
    if (bad) atomicAdd(&ctr->range_errors, bad);
}

// EXECUTE, one lane per op (batch index i) instead of one
// lane per transaction: S times the lanes, each with a single registration,
// for small or ragged batches that would leave the chip idle.
__global__ __launch_bounds__(kBlock) void kv_execute_ops_kernel(
    const uint64_t *__restrict__ keys, const uint32_t *__restrict__ meta,
    const uint32_t *__restrict__ tids, uint32_t B, uint32_t S, uint64_t rows, uint32_t fields,
    unsigned long long *__restrict__ regs, RegLayout rl, uint64_t hot, uint32_t tag,
    uint8_t *__restrict__ doomed, uint8_t epoch, bool reg_reads, bool zero_counts, uint32_t max_scan,
    DeviceCounters *__restrict__ ctr, bool rm)
{
    if (zero_counts && blockIdx.x == 0) zero_epoch_counts(ctr, kBlock);
    const uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
    const bool live = i < (uint64_t)S * B;
    const uint32_t t = live ? txn_of(i, B, S, rm) : 0u;
    const Op o = load_op(keys, meta, live ? i : 0, live, rows, fields, max_scan);
    const bool bad = o.kind != LTPG_KV_NONE && !o.valid;
    if (o.valid) {
        const unsigned long long me = priority(tag, tids[t], t);
        if (o.kind == LTPG_KV_WRITE) {
            if (o.row != hot && register_write(&regs[rl.w(o.row)], me, tag, doomed, epoch)) doomed[t] = epoch;
        } else if (reg_reads) {
            for (uint32_t k = 0; k < o.len; ++k)
                if (o.row + k != hot) register_read(&regs[rl.r(o.row + k)], me);
        }
    }
    if (bad) atomicAdd(&ctr->range_errors, 1u);
}

// EXECUTE, fast form, one lane per op with the block's duplicate rows
// folded first.  Under skew thousands of in-flight writes hit the same hot
// register at once, all see it stale, and their atomics serialize on one
// address.  Here each block takes P * kBlock consecutive ops (P per lane),
// finds the minimum writer priority of every row among them in an LDS hash
// table, and only that writer goes to the global register; the block's
// other writers of the row already have waw (a lower writer exists).  Every
// non-minimum writer of a row is still doomed exactly once.
// P (ops per lane) is 2, or 4 with LTPG_TUNE_MORE_ITEMS: a wider fold and
// more loads in flight per lane, against half the blocks.
template <uint32_t P>
__global__ __launch_bounds__(kBlock) void kv_execute_dedup_kernel(
    const uint64_t *__restrict__ keys, const uint32_t *__restrict__ meta,
    const uint32_t *__restrict__ tids, uint32_t B, uint32_t S, uint64_t rows, uint32_t fields,
    unsigned long long *__restrict__ regs, RegLayout rl, uint64_t hot, uint32_t tag,
    uint8_t *__restrict__ doomed, uint8_t epoch, bool zero_counts, uint32_t max_scan,
    DeviceCounters *__restrict__ ctr, bool rm)
{
    constexpr uint32_t kDedupOps = P * kBlock;
    constexpr uint32_t kDedupSlots = 2 * kDedupOps;  // load factor <= 1/2: probing always ends
    __shared__ unsigned long long s_key[kDedupSlots];  // row + 1, 0 = empty
    __shared__ unsigned long long s_min[kDedupSlots];
    if (zero_counts && blockIdx.x == 0) zero_epoch_counts(ctr, kBlock);
    for (uint32_t k = threadIdx.x; k < kDedupSlots; k += kBlock) {
        s_key[k] = 0ull;
        s_min[k] = ~0ull;
    }
    __syncthreads();
    const uint64_t n_ops = (uint64_t)S * B;
    const uint64_t base = (uint64_t)blockIdx.x * kDedupOps;
    uint64_t row[P];
    unsigned long long me[P];
    uint32_t tt[P], slot[P];
    bool wr[P];
    uint32_t bad = 0;
#pragma unroll
    for (uint32_t k = 0; k < P; ++k) {
        const uint64_t i = base + (uint64_t)k * kBlock + threadIdx.x;
        const bool live = i < n_ops;
        const uint32_t t = live ? txn_of(i, B, S, rm) : 0u;
        const Op o = load_op(keys, meta, live ? i : 0, live, rows, fields, max_scan);
        bad += (o.kind != LTPG_KV_NONE && !o.valid) ? 1u : 0u;
        wr[k] = o.valid && o.kind == LTPG_KV_WRITE && o.row != hot;
        row[k] = o.row;
        tt[k] = t;
        me[k] = wr[k] ? priority(tag, tids[t], t) : 0ull;
        slot[k] = 0;
    }
#pragma unroll
    for (uint32_t k = 0; k < P; ++k) {
        if (!wr[k]) continue;
        const unsigned long long key = row[k] + 1ull;
        uint32_t h = (uint32_t)((row[k] * 0x9E3779B97F4A7C15ull) >> 40) & (kDedupSlots - 1);
        while (true) {
            const unsigned long long prev = atomicCAS(&s_key[h], 0ull, key);
            if (prev == 0ull || prev == key) break;
            h = (h + 1) & (kDedupSlots - 1);
        }
        slot[k] = h;
        atomicMin(&s_min[h], me[k]);
    }
    __syncthreads();
    // register_write for the block minima, split into phases so that the
    // four probes, then the four atomics, are in flight together
    bool lead[P], waw[P];
    unsigned long long cur[P], old[P];
#pragma unroll
    for (uint32_t k = 0; k < P; ++k) {
        waw[k] = wr[k] && s_min[slot[k]] < me[k];
        lead[k] = wr[k] && !waw[k];
        cur[k] = lead[k] ? probe(&regs[rl.w(row[k])]) : ~0ull;
    }
#pragma unroll
    for (uint32_t k = 0; k < P; ++k) {
        old[k] = ~0ull;
        if (lead[k] && cur[k] > me[k]) old[k] = atomicMin(&regs[rl.w(row[k])], me[k]);
    }
#pragma unroll
    for (uint32_t k = 0; k < P; ++k) {
        if (!lead[k]) continue;
        if (cur[k] < me[k] || old[k] < me[k]) {
            waw[k] = true;
        } else if (cur[k] > me[k] && old[k] > me[k] && old[k] != ~0ull &&
                   (uint32_t)(old[k] >> kTagShift) == tag) {
            doomed[old[k] & kPosMask] = epoch;  // displaced: that writer has waw
        }
    }
#pragma unroll
    for (uint32_t k = 0; k < P; ++k)
        if (waw[k]) doomed[tt[k]] = epoch;
    if (bad) atomicAdd(&ctr->range_errors, bad);
}

// ---- row-partitioned EXECUTE with scans (LTPG_TUNE_PARTITIONED, fast form) --
// ---- (batches of point operations only are binned below) ------------------
//
// The register phase touches one random register line per operation; the
// lines of a 10M-row table overflow the L2s, so each 8-byte probe or atomic
// moves a 128-byte line.  Here the epoch's register operations (every write
// op, every row a read or scan op reads; hot-row ops never register) are
// first binned by row range into buckets of 2^kPartShift rows:
//   count    streaming pass over the ops: per-bucket sizes (LDS histogram,
//            one global add per bucket and block), range errors;
//   scan     one workgroup: bucket starts, cursors, and slices of at most
//            kPartSlice operations (a skewed bucket gets several);
//   scatter  second pass over the ops: each operation's (priority, row in
//            bucket, is-write) to its bucket, a block reserving one run per
//            bucket;
//   process  one workgroup per slice: the W minima of the bucket's rows in
//            LDS (probe, then a 64-bit LDS atomicMin), then the flags of the
//            fast form from them -- a writer behind the minimum is doomed; a
//            reader behind it has raw; a reader ahead of it gives the minimum
//            writer war.  A bucket split over several slices folds each
//            slice's minima into the global W registers instead;
//   flags    one workgroup per slice of such a bucket: the same flags from
//            the global W registers.
// The flags equal those of kv_execute_kernel + kv_mark_reads_kernel: both
// compare every operation with the minimum W priority of its row.
constexpr uint32_t kPartBlock = 1024;
constexpr uint32_t kPartPer = 16;  // operations per thread in the binning passes
constexpr uint32_t kPartChunk = kPartBlock * kPartPer;
constexpr uint32_t kPartRows = 1u << kPartShift;

struct PartArgs {
    const uint64_t *keys;
    const uint32_t *meta;
    const uint32_t *tids;
    uint32_t B, S;
    uint64_t rows;
    uint32_t fields, max_scan;
    uint64_t hot;
    uint32_t nb, cap_slices;
    uint32_t *count, *start, *cursor, *slices;
    unsigned long long *ent_me;
    uint32_t *ent_key;
    unsigned long long *regs;
    RegLayout rl;
    uint32_t tag;
    uint8_t epoch;
    bool rm;
    uint8_t *doomed, *raw_flag, *war_flag;
    DeviceCounters *ctr;
};

// kPartGroup consecutive op slots of a thread (stride kPartBlock), all
// loads issued before any is used.
constexpr uint32_t kPartGroup = 4;

template <uint32_t G>
__device__ __forceinline__ void part_load(const PartArgs &a, uint64_t first, Op (&o)[G])
{
    const uint64_t n_ops = (uint64_t)a.S * a.B;
    uint64_t r[G];
    uint32_t m[G];
#pragma unroll
    for (uint32_t u = 0; u < G; ++u) {
        const uint64_t i = first + (uint64_t)u * kPartBlock;
        const uint64_t j = i < n_ops ? i : 0ull;
        r[u] = a.keys[j];
        m[u] = a.meta[j];
    }
#pragma unroll
    for (uint32_t u = 0; u < G; ++u) {
        const bool live = first + (uint64_t)u * kPartBlock < n_ops;
        o[u] = decode_op(live ? r[u] : 0ull, live ? m[u] : 0u, a.rows, a.fields, a.max_scan);
    }
}

__global__ __launch_bounds__(kPartBlock) void kv_part_count_kernel(PartArgs a, bool zero_counts)
{
    __shared__ uint32_t s_hist[kPartMaxBuckets];
    if (zero_counts && blockIdx.x == 0) zero_epoch_counts(a.ctr, kPartBlock);
    for (uint32_t b = threadIdx.x; b < a.nb; b += kPartBlock) s_hist[b] = 0;
    __syncthreads();
    const uint64_t base = (uint64_t)blockIdx.x * kPartChunk + threadIdx.x;
    uint32_t bad = 0;
#pragma unroll 1
    for (uint32_t g = 0; g < kPartPer; g += kPartGroup) {
        Op o[kPartGroup];
        part_load(a, base + (uint64_t)g * kPartBlock, o);
#pragma unroll
        for (uint32_t u = 0; u < kPartGroup; ++u) {
            bad += (o[u].kind != LTPG_KV_NONE && !o[u].valid) ? 1u : 0u;
            if (!o[u].valid) continue;
            if (o[u].kind == LTPG_KV_WRITE) {
                if (o[u].row != a.hot) atomicAdd(&s_hist[o[u].row >> kPartShift], 1u);
            } else {
                for (uint32_t j = 0; j < o[u].len; ++j)
                    if (o[u].row + j != a.hot) atomicAdd(&s_hist[(o[u].row + j) >> kPartShift], 1u);
            }
        }
    }
    __syncthreads();
    for (uint32_t b = threadIdx.x; b < a.nb; b += kPartBlock) {
        const uint32_t c = s_hist[b];
        if (c) atomicAdd(&a.count[b], c);
    }
    if (bad) atomicAdd(&a.ctr->range_errors, bad);
}

// Exclusive scan of the bucket sizes into starts, cursors and slices (one
// workgroup; each thread owns a run of consecutive buckets).  Clears the
// sizes for the next epoch.
__global__ __launch_bounds__(kPartBlock) void kv_part_scan_kernel(PartArgs a)
{
    __shared__ uint32_t s_n[kPartBlock], s_sl[kPartBlock];
    const uint32_t per = (a.nb + kPartBlock - 1) / kPartBlock;
    const uint32_t b0 = threadIdx.x * per;
    uint32_t n = 0, ns = 0;
    for (uint32_t j = 0; j < per; ++j) {
        const uint32_t b = b0 + j;
        if (b < a.nb) {
            const uint32_t c = a.count[b];
            n += c;
            ns += (c + kPartSlice - 1) / kPartSlice;
        }
    }
    s_n[threadIdx.x] = n;
    s_sl[threadIdx.x] = ns;
    __syncthreads();
    // inclusive scans (Hillis-Steele over the block)
    for (uint32_t d = 1; d < kPartBlock; d <<= 1) {
        const uint32_t x = threadIdx.x >= d ? s_n[threadIdx.x - d] : 0u;
        const uint32_t y = threadIdx.x >= d ? s_sl[threadIdx.x - d] : 0u;
        __syncthreads();
        s_n[threadIdx.x] += x;
        s_sl[threadIdx.x] += y;
        __syncthreads();
    }
    uint32_t at = s_n[threadIdx.x] - n, sl = s_sl[threadIdx.x] - ns;
    for (uint32_t j = 0; j < per; ++j) {
        const uint32_t b = b0 + j;
        if (b >= a.nb) break;
        const uint32_t c = a.count[b];
        a.start[b] = at;
        a.cursor[b] = at;
        for (uint32_t k = 0; k * kPartSlice < c; ++k, ++sl) {
            if (sl >= a.cap_slices) continue;
            a.slices[3 * sl] = b;
            a.slices[3 * sl + 1] = at + k * kPartSlice;
            a.slices[3 * sl + 2] = at + min(c, (k + 1) * kPartSlice);
        }
        at += c;
        a.count[b] = 0;
    }
    if (threadIdx.x == kPartBlock - 1) {
        a.start[a.nb] = s_n[kPartBlock - 1];
        a.slices[3 * a.cap_slices] = min(s_sl[kPartBlock - 1], a.cap_slices);
    }
}

__global__ __launch_bounds__(kPartBlock) void kv_part_scatter_kernel(PartArgs a)
{
    __shared__ uint32_t s_at[kPartMaxBuckets];
    for (uint32_t b = threadIdx.x; b < a.nb; b += kPartBlock) s_at[b] = 0;
    __syncthreads();
    const uint64_t base = (uint64_t)blockIdx.x * kPartChunk + threadIdx.x;
#pragma unroll 1
    for (uint32_t g = 0; g < kPartPer; g += kPartGroup) {
        Op o[kPartGroup];
        part_load(a, base + (uint64_t)g * kPartBlock, o);
#pragma unroll
        for (uint32_t u = 0; u < kPartGroup; ++u) {
            if (!o[u].valid) continue;
            if (o[u].kind == LTPG_KV_WRITE) {
                if (o[u].row != a.hot) atomicAdd(&s_at[o[u].row >> kPartShift], 1u);
            } else {
                for (uint32_t j = 0; j < o[u].len; ++j)
                    if (o[u].row + j != a.hot) atomicAdd(&s_at[(o[u].row + j) >> kPartShift], 1u);
            }
        }
    }
    __syncthreads();
    // one run per bucket: the block's count becomes its run's start
    for (uint32_t b = threadIdx.x; b < a.nb; b += kPartBlock) {
        const uint32_t c = s_at[b];
        if (c) s_at[b] = atomicAdd(&a.cursor[b], c);
    }
    __syncthreads();
    const uint64_t n_ops = (uint64_t)a.S * a.B;
    constexpr uint32_t G = kPartGroup;
#pragma unroll 1
    for (uint32_t g = 0; g < kPartPer; g += G) {
        Op o[G];
        unsigned long long me[G];
        part_load(a, base + (uint64_t)g * kPartBlock, o);
#pragma unroll
        for (uint32_t u = 0; u < G; ++u) {
            // op indices stay below 2^32 (kv_part_prepare): 32-bit division
            const uint64_t i = base + (uint64_t)(g + u) * kPartBlock;
            const uint32_t i32 = i < n_ops ? (uint32_t)i : 0u;
            const uint32_t t = a.rm ? i32 / a.S : i32 % a.B;
            me[u] = priority(a.tag, a.tids[t], t);
        }
#pragma unroll
        for (uint32_t u = 0; u < G; ++u) {
            if (!o[u].valid) continue;
            if (o[u].kind == LTPG_KV_WRITE) {
                if (o[u].row == a.hot) continue;
                const uint32_t at = atomicAdd(&s_at[o[u].row >> kPartShift], 1u);
                a.ent_me[at] = me[u];
                a.ent_key[at] = ((uint32_t)(o[u].row & (kPartRows - 1)) << 1) | 1u;
            } else {
                for (uint32_t j = 0; j < o[u].len; ++j) {
                    const uint64_t r = o[u].row + j;
                    if (r == a.hot) continue;
                    const uint32_t at = atomicAdd(&s_at[r >> kPartShift], 1u);
                    a.ent_me[at] = me[u];
                    a.ent_key[at] = (uint32_t)(r & (kPartRows - 1)) << 1;
                }
            }
        }
    }
}

// The fast form's flags of one operation against its row's minimum W
// priority w (~0: no writer this epoch).
__device__ __forceinline__ void part_flag(const PartArgs &a, uint32_t key, unsigned long long me,
                                          unsigned long long w)
{
    const uint32_t pos = (uint32_t)(me & kPosMask);
    if (key & 1u) {
        if (w < me) a.doomed[pos] = a.epoch;
    } else if (w != ~0ull) {
        if (w < me)
            a.raw_flag[pos] = a.epoch;
        else if (w > me)
            a.war_flag[w & kPosMask] = a.epoch;
    }
}

__global__ __launch_bounds__(kPartBlock) void kv_part_process_kernel(PartArgs a)
{
    __shared__ unsigned long long s_w[kPartRows];
    if (blockIdx.x >= a.slices[3 * a.cap_slices]) return;
    const uint32_t b = a.slices[3 * blockIdx.x], beg = a.slices[3 * blockIdx.x + 1], end = a.slices[3 * blockIdx.x + 2];
    const bool multi = a.start[b + 1] - a.start[b] > kPartSlice;
    for (uint32_t r = threadIdx.x; r < kPartRows; r += kPartBlock) s_w[r] = ~0ull;
    __syncthreads();
    for (uint32_t e0 = beg + threadIdx.x; e0 < end; e0 += kPartGroup * kPartBlock) {
        uint32_t key[kPartGroup];
        unsigned long long me[kPartGroup];
#pragma unroll
        for (uint32_t u = 0; u < kPartGroup; ++u) {
            const uint32_t e = e0 + u * kPartBlock;
            key[u] = e < end ? a.ent_key[e] : 0u;
            me[u] = e < end ? a.ent_me[e] : ~0ull;
        }
#pragma unroll
        for (uint32_t u = 0; u < kPartGroup; ++u)
            if ((key[u] & 1u) && s_w[key[u] >> 1] > me[u]) atomicMin(&s_w[key[u] >> 1], me[u]);
    }
    __syncthreads();
    if (multi) {
        const uint64_t row0 = (uint64_t)b << kPartShift;
        for (uint32_t r = threadIdx.x; r < kPartRows; r += kPartBlock) {
            const unsigned long long v = s_w[r];
            if (v == ~0ull) continue;
            unsigned long long *p = &a.regs[a.rl.w(row0 + r)];
            if (probe(p) > v) atomicMin(p, v);
        }
        return;
    }
    for (uint32_t e0 = beg + threadIdx.x; e0 < end; e0 += kPartGroup * kPartBlock) {
        uint32_t key[kPartGroup];
        unsigned long long me[kPartGroup];
#pragma unroll
        for (uint32_t u = 0; u < kPartGroup; ++u) {
            const uint32_t e = e0 + u * kPartBlock;
            key[u] = e < end ? a.ent_key[e] : 0u;
            me[u] = e < end ? a.ent_me[e] : ~0ull;
        }
#pragma unroll
        for (uint32_t u = 0; u < kPartGroup; ++u)
            if (e0 + u * kPartBlock < end) part_flag(a, key[u], me[u], s_w[key[u] >> 1]);
    }
}

// The bucket's final W minima are read from the registers once, in row
// order, into LDS; each operation then finds its row's minimum there.
__global__ __launch_bounds__(kPartBlock) void kv_part_flags_kernel(PartArgs a)
{
    __shared__ unsigned long long s_w[kPartRows];
    if (blockIdx.x >= a.slices[3 * a.cap_slices]) return;
    const uint32_t b = a.slices[3 * blockIdx.x], beg = a.slices[3 * blockIdx.x + 1], end = a.slices[3 * blockIdx.x + 2];
    if (a.start[b + 1] - a.start[b] <= kPartSlice) return;  // decided in kv_part_process_kernel
    const uint64_t row0 = (uint64_t)b << kPartShift;
    for (uint32_t r = threadIdx.x; r < kPartRows; r += kPartBlock) {
        unsigned long long w = ~0ull;
        if (row0 + r < a.rows) {
            w = a.regs[a.rl.w(row0 + r)];
            if ((uint32_t)(w >> kTagShift) != a.tag) w = ~0ull;  // no writer this epoch
        }
        s_w[r] = w;
    }
    __syncthreads();
    for (uint32_t e0 = beg + threadIdx.x; e0 < end; e0 += kPartGroup * kPartBlock) {
        uint32_t key[kPartGroup];
        unsigned long long me[kPartGroup];
#pragma unroll
        for (uint32_t u = 0; u < kPartGroup; ++u) {
            const uint32_t e = e0 + u * kPartBlock;
            key[u] = e < end ? a.ent_key[e] : 0u;
            me[u] = e < end ? a.ent_me[e] : ~0ull;
        }
#pragma unroll
        for (uint32_t u = 0; u < kPartGroup; ++u)
            if (e0 + u * kPartBlock < end) part_flag(a, key[u], me[u], s_w[key[u] >> 1]);
    }
}

// ---- binned EXECUTE of point operations (LTPG_TUNE_PARTITIONED, or the
// ---- default shape of a large epoch; fast form, no scans; bin_execute.h) ---
struct KvBinSource {
    static constexpr bool kSmallTiles = false;
    const uint64_t *keys;
    const uint32_t *meta;
    uint64_t rows;
    uint32_t fields, max_scan;
    uint64_t hot;
    struct Raw {
        uint64_t row;
        uint32_t meta;
    };
    __device__ __forceinline__ Raw load(const BinArgs &, uint32_t i) const { return Raw{keys[i], meta[i]}; }
    __device__ __forceinline__ uint32_t decode(const BinArgs &, const Raw &r, uint32_t, bool live, bool *use,
                                               uint32_t *row, bool *write) const
    {
        const Op o = decode_op(r.row, live ? r.meta : 0u, rows, fields, max_scan);
        *use = o.valid && o.row != hot;
        *row = (uint32_t)o.row;
        *write = o.kind == LTPG_KV_WRITE;
        return (o.kind != LTPG_KV_NONE && !o.valid) ? 1u : 0u;
    }
};

// Read marking (fast form), one lane per op after every write has
// registered.  A read of row x by t against w = W[x] of this epoch:
//   w < me: t reads a row a higher-priority transaction writes -> raw(t);
//   w > me: the row's minimum writer (position bits of w) writes a row a
//           higher-priority transaction reads -> war for that writer.
// A writer with waw aborts anyway, so flagging only the minimum writer
// gives every transaction that can still commit its exact war bit; raw(t)
// is exact for every t.  Flags hold the epoch number, so equal stores race
// harmlessly and nothing is cleared between epochs.
template <uint32_t P>
__global__ __launch_bounds__(kBlock) void kv_mark_reads_kernel(
    const uint64_t *__restrict__ keys, const uint32_t *__restrict__ meta,
    const uint32_t *__restrict__ tids, uint32_t B, uint32_t S, uint64_t rows, uint32_t fields,
    const unsigned long long *__restrict__ regs, RegLayout rl, uint64_t hot, uint32_t tag,
    uint8_t *__restrict__ raw_flag, uint8_t *__restrict__ war_flag, uint8_t epoch, uint32_t max_scan, bool rm)
{
    // P ops per lane (1, or 2 with LTPG_TUNE_MORE_ITEMS), stride kBlock; all
    // their loads issued before any is used
    const uint64_t base = (uint64_t)blockIdx.x * (P * kBlock) + threadIdx.x;
    const uint64_t n_ops = (uint64_t)S * B;
    Op o[P];
    uint32_t t[P];
#pragma unroll
    for (uint32_t u = 0; u < P; ++u) {
        const uint64_t i = base + (uint64_t)u * kBlock;
        const bool live = i < n_ops;
        t[u] = live ? txn_of(i, B, S, rm) : 0u;
        o[u] = load_op(keys, meta, live ? i : 0, live, rows, fields, max_scan);
    }
#pragma unroll
    for (uint32_t u = 0; u < P; ++u) {
        if (o[u].len == 0) continue;  // writes, empty and invalid slots
        const unsigned long long me = priority(tag, tids[t[u]], t[u]);
        bool raw = false;
        constexpr uint32_t R = 8;  // a scan: every row of its range, eight registers in flight
        for (uint32_t k0 = 0; k0 < o[u].len; k0 += R) {
            unsigned long long w[R];
#pragma unroll
            for (uint32_t r = 0; r < R; ++r) {
                if (r && max_scan <= 1) break;
                w[r] = regs[rl.w(o[u].row + (k0 + r < o[u].len ? k0 + r : 0u))];
            }
#pragma unroll
            for (uint32_t r = 0; r < R; ++r) {
                if (r && max_scan <= 1) break;
                if (k0 + r >= o[u].len || o[u].row + k0 + r == hot) continue;
                if ((uint32_t)(w[r] >> kTagShift) != tag) continue;  // no writer this epoch
                if (w[r] < me)
                    raw = true;
                else if (w[r] > me)
                    war_flag[w[r] & kPosMask] = epoch;
            }
        }
        if (raw) raw_flag[t[u]] = epoch;
    }
}

// CHECK + COMMIT, counting form (check_r / check_w_0 / check_w_1 and
// __CHECK, YCSB/0/Execute.h:109-175, Genericfunction.h:101-144; writeback_0,
// Execute.h:184-191): every transaction counts raw (reads whose W register
// holds a higher priority), war (writes vs R) and waw (writes vs W) over all
// its ops -- the reference's counters, kept for parity checks of them --
// and commits iff waw == 0 && (raw == 0 || war == 0).
__global__ __launch_bounds__(kBlock) void kv_check_counting_kernel(
    const uint64_t *__restrict__ keys, const uint32_t *__restrict__ meta,
    const uint32_t *__restrict__ tids, uint32_t B, uint32_t S, uint64_t rows, uint32_t fields,
    const unsigned long long *__restrict__ regs, RegLayout rl, uint64_t hot, uint32_t tag,
    uint64_t *__restrict__ bitmap, uint32_t *__restrict__ conflicts, uint32_t max_scan,
    DeviceCounters *__restrict__ ctr, bool rm)
{
    const uint32_t t = blockIdx.x * kBlock + threadIdx.x;
    const int lane = lane_id();
    const bool live = t < B;
    const unsigned long long me = live ? priority(tag, tids[t], t) : 0ull;
    uint32_t raw = 0, war = 0, waw = 0;
    for (uint32_t s = 0; s < S; ++s) {
        const Op o = load_op(keys, meta, op_at(s, t, B, S, rm), live, rows, fields, max_scan);
        if (!o.valid) continue;
        if (o.kind != LTPG_KV_WRITE) {
            for (uint32_t k = 0; k < o.len; ++k)  // the hot row never conflicts
                raw += (o.row + k != hot && regs[rl.w(o.row + k)] < me) ? 1u : 0u;
        } else if (o.row != hot) {
            war += regs[rl.r(o.row)] < me ? 1u : 0u;
            waw += regs[rl.w(o.row)] < me ? 1u : 0u;
        }
    }
    const bool commit = live && waw == 0 && (raw == 0 || war == 0);
    if (live) conflicts[t] = raw | (war << 8) | (waw << 16);
    const unsigned long long word = __ballot(commit);
    const uint32_t wave_base = t - (uint32_t)lane;
    if (lane == 0 && wave_base < B) {
        bitmap[wave_base / 64] = word;
        const uint32_t n = (uint32_t)__popcll(word);
        const uint32_t live_n = (B - wave_base) < 64u ? (B - wave_base) : 64u;
        add_counts(ctr, (blockIdx.x * (kBlock / 64) + threadIdx.x / 64) % kCounterStripes, LTPG_TYPE_KV, n, live_n);
    }
}

// READOUT: committed transactions' read fields, gathered from the snapshot
// before any write-back of the epoch (read_1 / __READ, YCSB/0/Execute.h:
// 27-37, Genericfunction.h:31-45).  Reads of aborted transactions are never
// delivered, so they are not gathered.
template <int LP>
__global__ __launch_bounds__(kBlock) void kv_readout_kernel(
    const uint64_t *__restrict__ keys, const uint32_t *__restrict__ meta, uint32_t B, uint32_t S,
    uint64_t rows, uint32_t fields, uint32_t fw, uint32_t fsw, const uint32_t *__restrict__ table,
    const uint64_t *__restrict__ bitmap, uint32_t *__restrict__ read_values, uint32_t max_scan, uint32_t L,
    bool rm)
{
    const uint32_t t = blockIdx.x * kBlock + threadIdx.x;
    const int lane = lane_id();
    const uint32_t wave_base = t - (uint32_t)lane;
    if (wave_base >= B) return;
    const uint64_t word = bitmap[wave_base / 64];
    if (word == 0) return;
    const bool committed = t < B && ((word >> lane) & 1ull);
    for (uint32_t s = 0; s < S; ++s) {
        const uint64_t i = (uint64_t)s * B + t;  // slot-major: where its reads go
        const Op o = load_op(keys, meta, op_at(s, t, B, S, rm), committed, rows, fields, max_scan);
        for (uint32_t k = 0;; ++k) {  // row k of each read / scan
            const unsigned long long mask = __ballot(k < o.len);
            if (!mask) break;
            copy_fields<LP>(mask, ((o.row + k) * fields + o.field) * fsw, (i * L + k) * fw, 0u, table,
                            read_values, fw);
        }
    }
}

// Block-local compaction.  A chunk is CH consecutive transactions (CH =
// 256, or 64 as a launch shape); the transactions that still have work
// (committed ones, for the read-out of CHECK and for WRITEBACK) are gathered
// into an LDS list, then processed G lanes per transaction (one lane per
// slot), so lanes stay busy whatever the abort rate and every op load of a
// transaction is issued at once.  A wave walks the list in rounds of 64 / G
// transactions; for small batches gridDim.y blocks share one chunk's list
// (each builds the same list and takes every gridDim.y-th round), so that a
// small epoch runs as many short waves rather than a few long ones.
constexpr uint32_t kChunk = kBlock;

// Gathers the picked transactions (one per thread) into s_list in thread
// order, so that every block of a chunk builds the same list and can take
// its own share of it by index.  Every thread of the block calls it (it
// holds two barriers); s_cnt has one word per wave.  Returns the length.
__device__ __forceinline__ uint32_t list_build(bool pick, uint32_t t, uint32_t *s_list, uint32_t *s_cnt)
{
    const int lane = lane_id();
    const uint32_t wave = threadIdx.x / 64;
    const unsigned long long m = __ballot(pick);
    if (lane == 0) s_cnt[wave] = (uint32_t)__popcll(m);
    __syncthreads();
    uint32_t base = 0, n = 0;
#pragma unroll
    for (uint32_t w = 0; w < kBlock / 64; ++w) {
        const uint32_t c = s_cnt[w];
        base += w < wave ? c : 0u;
        n += c;
    }
    if (pick) s_list[base + (uint32_t)__popcll(m & ((1ull << lane) - 1ull))] = t;
    __syncthreads();
    return n;
}

// Per-wave staging of field copies.  A wave walks its transactions in
// rounds of 64 / G; a round of a low-contention batch flags only a few
// fields, and copying them right away leaves a wave with one round's fields
// in flight.  Instead each round appends its flagged fields (source,
// destination, delta) to the wave's own LDS list, and the list is copied
// once it holds 64 or more (or at the end), while rounds of op loads run back
// to back.  The list holds a round's worth more than the flush threshold.
// Only the wave that owns a list touches it, so a wavefront-scope fence
// orders its lanes' LDS accesses.
constexpr uint32_t kStage = 128;

struct StageList {
    unsigned long long src[kStage];
    unsigned long long dst[kStage];
    uint32_t delta[kStage];
};

__device__ __forceinline__ void wave_lds_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
}

// Append the flagged lanes' copies; returns the new (wave-uniform) length.
__device__ __forceinline__ uint32_t stage_push(StageList &l, uint32_t n, bool flag, uint64_t src_off,
                                               uint64_t dst_off, uint32_t delta)
{
    const unsigned long long m = __ballot(flag);
    if (flag) {
        const uint32_t at = n + (uint32_t)__popcll(m & ((1ull << lane_id()) - 1ull));
        l.src[at] = src_off;
        l.dst[at] = dst_off;
        l.delta[at] = delta;
    }
    return n + (uint32_t)__popcll(m);
}

// Four words at any word boundary: one 16-byte access.
struct __attribute__((packed, aligned(4))) Words4 {
    uint32_t w[4];
};

// How a wave copies fields of fw >= 4 words: 2^log_lanes adjacent lanes per
// field, lane k the words from 4k -- the last one the field's last four words,
// which overlap its neighbour's (both load them before either stores, and
// store equal values), so that no access leaves the field.
struct FieldLanes {
    uint32_t log_lanes, off;
    bool on;
    __device__ explicit FieldLanes(uint32_t fw)
    {
        const uint32_t need = (fw + 3) / 4;
        log_lanes = need <= 1 ? 0u : 32u - (uint32_t)__clz((int)(need - 1));
        const uint32_t k = (uint32_t)lane_id() & ((1u << log_lanes) - 1u);
        on = k < need;
        off = on ? min(4 * k, fw - 4) : 0u;
    }
};

// Copy the wave's n staged fields (fw >= 4): src[src_off + w] + delta ->
// dst[dst_off + w].  The staged fields never overlap: callers stage distinct
// destinations.  A 100-byte field takes 7 lanes of 8, so an instruction moves
// eight fields and four steps are in flight.  Bound by the random lines it
// touches; with 32 lanes of 4 bytes per field and each field's addresses
// looked up by ballot it was bound by instruction issue (318M vector
// instructions for the 7M reads of 2^20 transactions of 9 reads and a write).
__device__ __forceinline__ void stage_flush(StageList &l, uint32_t n, const FieldLanes &f, const uint32_t *src,
                                            uint32_t *dst)
{
    constexpr uint32_t U = 4;
    wave_lds_fence();
    const uint32_t mine = (uint32_t)lane_id() >> f.log_lanes, per = 64u >> f.log_lanes;
    for (uint32_t b = 0; b < n; b += U * per) {
        Words4 v[U];
        uint64_t d[U];
        uint32_t dl[U];
        bool ok[U];
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
            const uint32_t e = b + u * per + mine;
            ok[u] = f.on && e < n;
            const uint32_t at = ok[u] ? e : 0u;  // idle lanes load the first field, so no load is conditional
            d[u] = l.dst[at] + f.off;
            dl[u] = l.delta[at];
            v[u] = *reinterpret_cast<const Words4 *>(src + l.src[at] + f.off);
        }
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
            if (!ok[u]) continue;
            Words4 w;
#pragma unroll
            for (int k = 0; k < 4; ++k) w.w[k] = v[u].w[k] + dl[u];
            *reinterpret_cast<Words4 *>(dst + d[u]) = w;
        }
    }
    wave_lds_fence();
}

// Random-gather ceiling: n fields of fw words, each from a random slot
// (stride_w words apart) of src, copied to dst[i * fw ..] -- the access
// pattern of CHECK's read-out -- the way it copies them, 64 fields per wave
// step.
__global__ __launch_bounds__(kBlock) void calib_gather_kernel(const uint32_t *__restrict__ src, uint64_t slots,
                                                             uint32_t stride_w, uint32_t fw,
                                                             uint32_t *__restrict__ dst, uint64_t n, uint32_t per)
{
    __shared__ StageList s_stage[kBlock / 64];
    StageList &list = s_stage[threadIdx.x / 64];
    const FieldLanes lanes(fw);
    const uint64_t wave = ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) / 64;
    for (uint32_t k = 0; k < per; ++k) {
        const uint64_t i = (wave * per + k) * 64 + (uint64_t)lane_id();
        const bool has = i < n;
        const uint64_t so = has ? calib_index(i, slots) * stride_w : 0ull;
        if (fw >= 4) {
            const uint32_t pending = stage_push(list, 0, has, so, i * fw, 0u);
            if (pending) stage_flush(list, pending, lanes, src, dst);
        } else if (has) {
            for (uint32_t w = 0; w < fw; ++w) dst[i * fw + w] = src[so + w];
        }
    }
}

// One lane copies one field of fw <= 32 words (src_off a multiple of 4
// words): every 16-byte load of the field is issued before the first store,
// so a wave has all its fields in flight in one round.  Stores are 16 bytes
// wide where dst_off is a multiple of 4 words and the vector lies inside the
// field, else word by word, so nothing past word fw is written.
__device__ __forceinline__ void lane_copy(bool active, uint64_t src_off, uint64_t dst_off,
                                          uint32_t delta, const uint32_t *src, uint32_t *dst,
                                          uint32_t fw)
{
    if (!active) return;
    const uint4 *s4 = reinterpret_cast<const uint4 *>(src + src_off);
    uint4 v[8];
#pragma unroll
    for (uint32_t u = 0; u < 8; ++u)
        if (4 * u < fw) v[u] = s4[u];
    const bool vec = (dst_off & 3ull) == 0;
#pragma unroll
    for (uint32_t u = 0; u < 8; ++u) {
        if (4 * u >= fw) continue;
        const uint32_t w[4] = {v[u].x + delta, v[u].y + delta, v[u].z + delta, v[u].w + delta};
        if (vec && 4 * u + 4 <= fw) {
            *reinterpret_cast<uint4 *>(dst + dst_off + 4 * u) = make_uint4(w[0], w[1], w[2], w[3]);
        } else {
#pragma unroll
            for (uint32_t r = 0; r < 4; ++r)
                if (4 * u + r < fw) dst[dst_off + 4 * u + r] = w[r];
        }
    }
}

// Read-out of one op per lane on fields of FW < 4 words, each lane its own:
// one load if the wave has no scan, otherwise eight rows' loads in flight
// (bound by those random loads).  With four rows of three words each, whatever
// the fields and the ops, 2^20 transactions of 10 ops on 8-byte fields took 267
// us per epoch, 256 so; 10,000 of 10 scans of 100 rows 186, with the same in
// the read marking 134 so.
template <uint32_t FW>
__device__ __forceinline__ void read_narrow(const Op &o, uint64_t src, uint64_t step, uint64_t dst,
                                            const uint32_t *table, uint32_t *read_values)
{
    struct __attribute__((packed, aligned(4))) Words {
        uint32_t w[FW];
    };
    if (!__ballot(o.len > 1)) {
        const Words v = *reinterpret_cast<const Words *>(table + (o.len ? src : 0ull));
        if (o.len) *reinterpret_cast<Words *>(read_values + dst) = v;
        return;
    }
    constexpr uint32_t U = 8;
    for (uint32_t k0 = 0; k0 < o.len; k0 += U) {
        Words v[U];
#pragma unroll
        for (uint32_t u = 0; u < U; ++u)
            v[u] = *reinterpret_cast<const Words *>(table + (k0 + u < o.len ? src + (k0 + u) * step : 0ull));
#pragma unroll
        for (uint32_t u = 0; u < U; ++u)
            if (k0 + u < o.len) *reinterpret_cast<Words *>(read_values + dst + (k0 + u) * FW) = v[u];
    }
}

// Read-out of one op per lane (its rows' fields to the read values of slot
// position i): fields of 16 bytes and more through the wave's list, whose
// length it returns; narrower ones each lane its own.  Every lane of the wave
// calls it.
__device__ __forceinline__ uint32_t read_out(const Op &o, uint64_t i, StageList &list, uint32_t pending,
                                             const FieldLanes &lanes, const uint32_t *table, uint32_t *read_values,
                                             uint32_t fields, uint32_t fw, uint32_t fsw, uint32_t L)
{
    const uint64_t src0 = (o.row * fields + o.field) * fsw, step = (uint64_t)fields * fsw, dst0 = i * L * fw;
    if (fw < 4) {
        if (fw == 1) read_narrow<1>(o, src0, step, dst0, table, read_values);
        else if (fw == 2) read_narrow<2>(o, src0, step, dst0, table, read_values);
        else read_narrow<3>(o, src0, step, dst0, table, read_values);
        return 0;
    }
    for (uint32_t k = 0; __ballot(k < o.len); ++k) {  // row k of each read / scan: its own destination
        pending = stage_push(list, pending, k < o.len, src0 + k * step, dst0 + k * fw, 0u);
        if (pending >= 64) {
            stage_flush(list, pending, lanes, table, read_values);
            pending = 0;
        }
    }
    return pending;
}

// CHECK + COMMIT + read-out, fast form (rules as kv_check_counting_kernel).
// EXECUTE and the read marking have decided everything: a transaction
// commits iff it has no waw (doomed) and not both raw and war.  A block
// compacts its committed transactions into an LDS list and gathers their
// read fields right away, G lanes per transaction: no write-back has run
// yet, so the table is the snapshot (read_1 / __READ, YCSB/0/Execute.h:
// 27-37).  Commit bits collect in LDS and leave as whole bitmap words.
template <int G, int CH>
__global__ __launch_bounds__(kBlock) void kv_check_fast_kernel(
    const uint64_t *__restrict__ keys, const uint32_t *__restrict__ meta, uint32_t B, uint32_t S,
    uint64_t rows, uint32_t fields, uint32_t fw, uint32_t fsw, const uint8_t *__restrict__ doomed,
    const uint8_t *__restrict__ raw_flag, const uint8_t *__restrict__ war_flag, uint8_t epoch,
    const uint32_t *__restrict__ table, uint32_t *__restrict__ read_values, uint64_t *__restrict__ bitmap,
    uint32_t max_scan, uint32_t L, uint32_t per_lane, DeviceCounters *__restrict__ ctr, bool rm)
{
    __shared__ uint32_t s_list[CH];
    __shared__ unsigned long long s_bits[CH / 64];
    __shared__ uint32_t s_cnt[kBlock / 64];
    __shared__ StageList s_stage[kBlock / 64];
    const int lane = lane_id();
    const uint32_t chunk0 = blockIdx.x * CH;
    const uint32_t t0 = chunk0 + threadIdx.x;
    const bool commit = threadIdx.x < CH && t0 < B && doomed[t0] != epoch &&
                        !(raw_flag[t0] == epoch && war_flag[t0] == epoch);
    {
        const unsigned long long m = __ballot(commit);
        if (threadIdx.x < CH && lane == 0) s_bits[threadIdx.x / 64] = m;
    }
    const uint32_t n = list_build(commit, t0, s_list, s_cnt);
    constexpr uint32_t PER = 64 / G;  // transactions per wave per round
    const uint32_t grp = (uint32_t)lane / G, gl = (uint32_t)lane % G;
    StageList &list = s_stage[threadIdx.x / 64];
    const FieldLanes lanes(fw);
    uint32_t pending = 0;
    for (uint32_t j0 = (blockIdx.y * (kBlock / 64) + threadIdx.x / 64) * PER; j0 < n;
         j0 += gridDim.y * (kBlock / 64) * PER) {
        const uint32_t j = j0 + grp;
        const bool has = j < n;
        const uint32_t t = has ? s_list[j] : 0u;
        const uint64_t i = (uint64_t)gl * B + t;  // slot-major: where its reads go
        const Op o = load_op(keys, meta, op_at(gl, t, B, S, rm), has && gl < S, rows, fields, max_scan);
        if (per_lane) {
            // one lane per read op: all fields of a round in flight at once
            for (uint32_t k = 0; k < o.len; ++k)
                lane_copy(true, ((o.row + k) * fields + o.field) * fsw, (i * L + k) * fw, 0u, table,
                          read_values, fw);
        } else {
            pending = read_out(o, i, list, pending, lanes, table, read_values, fields, fw, fsw, L);
        }
    }
    if (pending) stage_flush(list, pending, lanes, table, read_values);
    if (blockIdx.y != 0) return;  // the chunk's other blocks only read out
    const uint32_t nwords = (B + 63) / 64;
    if (threadIdx.x < CH / 64 && chunk0 / 64 + threadIdx.x < nwords)
        bitmap[chunk0 / 64 + threadIdx.x] = s_bits[threadIdx.x];
    if (threadIdx.x == 0) {
        const uint32_t live_n = (B - chunk0) < (uint32_t)CH ? (B - chunk0) : (uint32_t)CH;
        add_counts(ctr, blockIdx.x % kCounterStripes, LTPG_TYPE_KV, n, live_n);
    }
}

// WRITEBACK: committed transactions apply their write slots (writeback_w /
// __WRITEBACK, YCSB/0/Execute.h:193-206, Genericfunction.h:145-158).
// Value: word + delta, delta = TID | 1 for RMW and 0 for copy-back, applied
// per write op in slot order.  The committed writer of a row is unique (the
// minimum W registrant), so reading the table here reads the snapshot.
// Several write ops of one transaction on one field are folded: the first
// in slot order writes word + count * delta, the others nothing -- the same
// result as applying them one by one, and it lets every store of a round go
// out without ordering between them.
struct WriteArgs {
    const uint64_t *keys;
    const uint32_t *meta;
    const uint32_t *tids;
    uint32_t B, S;
    uint64_t rows;
    uint32_t fields, fw, fsw;
    uint32_t *table;
    uint32_t values;
    uint64_t hot;
    uint32_t per_lane;
    bool rm;
    EpochEnd end;
};

// The end of an epoch that keeps no state: its commit count and range errors
// (final before WRITEBACK, whose first wave this is), and the TID order flag
// starts over.  As a kernel of its own 2 us and a launch.
__device__ __forceinline__ void end_epoch(const EpochEnd &e)
{
    static_assert(kCounterStripes == 64, "one lane per stripe");
    if (!e.ctr || blockIdx.x != 0 || blockIdx.y != 0 || threadIdx.x >= 64) return;
    uint32_t c = e.ctr->commits[threadIdx.x][LTPG_TYPE_KV];
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) c += __shfl_xor(c, d);
    if (threadIdx.x != 0) return;
    e.marks[kMarkUnsorted] = e.marks[kMarkWritten] = 0;
    if (!e.result) return;
    e.result[0] = c;
    e.result[1] = e.ctr->range_errors;
}

// One round of 64 / G transactions, t the lane group's (if has).
template <int G>
__device__ __forceinline__ uint32_t write_round(const WriteArgs &a, bool has, uint32_t t, StageList &list,
                                                uint32_t pending, const FieldLanes &lanes)
{
    const uint32_t grp = (uint32_t)lane_id() / G, gl = (uint32_t)lane_id() % G;
    const uint32_t step = (has && a.values == LTPG_VALUES_RMW) ? (a.tids[t] | 1u) : 0u;
    const Op o = load_op(a.keys, a.meta, op_at(gl, t, a.B, a.S, a.rm), has && gl < a.S, a.rows, a.fields);
    // writes to the hot row go through kv_hot_sum_kernel
    const bool wr = o.valid && o.kind == LTPG_KV_WRITE && o.row != a.hot;
    const unsigned long long wm = __ballot(wr);
    if (!wm) return pending;
    const uint64_t off = (o.row * a.fields + o.field) * a.fsw;
    // fold duplicates: count this field among the group's write slots
    uint32_t count = 0;
    bool first = true;
    for (uint32_t k = 0; k < a.S && k < (uint32_t)G; ++k) {
        const int from = (int)(grp * G + k);
        const uint64_t ok = __shfl(off, from);
        if (((wm >> from) & 1ull) && ok == off) {
            ++count;
            first &= k >= gl;
        }
    }
    if (a.per_lane) {
        lane_copy(wr && first, off, off, step * count, a.table, a.table, a.fw);
        return pending;
    }
    if (a.fw < 4) {
        if (wr && first)
            for (uint32_t w = 0; w < a.fw; ++w) a.table[off + w] += step * count;
        return pending;
    }
    // a row's committed writer is unique and its duplicate writes are
    // folded: staged fields never overlap
    pending = stage_push(list, pending, wr && first, off, off, step * count);
    if (pending >= 64) {
        stage_flush(list, pending, lanes, a.table, a.table);
        pending = 0;
    }
    return pending;
}

template <int G, int CH>
__global__ __launch_bounds__(kBlock) void kv_writeback_kernel(WriteArgs a, const uint64_t *__restrict__ bitmap)
{
    __shared__ uint32_t s_list[CH];
    __shared__ uint32_t s_cnt[kBlock / 64];
    __shared__ StageList s_stage[kBlock / 64];
    end_epoch(a.end);
    const uint32_t t0 = blockIdx.x * CH + threadIdx.x;
    // t0 < B also guards a bitmap word left by an earlier, larger batch
    // when this phase runs without a fresh CHECK
    const uint32_t n = list_build(threadIdx.x < CH && t0 < a.B && ((bitmap[t0 / 64] >> (t0 % 64)) & 1ull), t0,
                                  s_list, s_cnt);
    constexpr uint32_t PER = 64 / G;
    const uint32_t grp = (uint32_t)lane_id() / G;
    StageList &list = s_stage[threadIdx.x / 64];
    const FieldLanes lanes(a.fw);
    uint32_t pending = 0;
    for (uint32_t j0 = (blockIdx.y * (kBlock / 64) + threadIdx.x / 64) * PER; j0 < n;
         j0 += gridDim.y * (kBlock / 64) * PER) {
        const bool has = j0 + grp < n;
        pending = write_round<G>(a, has, has ? s_list[j0 + grp] : 0u, list, pending, lanes);
    }
    if (pending) stage_flush(list, pending, lanes, a.table, a.table);
}

// ---- the committed transactions of a large batch as one list ---------------
//
// Commits crowd among the lowest priorities, so with a block per 256
// transactions a few blocks do nearly all of an epoch's field copies.  For
// large batches (kv_check_lists) CHECK decides every transaction
// first and lists the committed ones (kv_commit_list_kernel); the read-out and
// WRITEBACK then share that list evenly over the whole chip.  2^20
// transactions x 16 ops on 100-byte fields, 3.5 % committed: CHECK 64 -> 7 + 29
// us, WRITEBACK 74 -> 27 us.  With 81 % committed (9 reads, 1 write): CHECK 662
// -> 7 + 441 us, which is the rate of random 128-byte reads and whole writes
// (3.6 TB/s; the gather alone reaches 4.2), WRITEBACK 148 -> 76 us.
constexpr uint32_t kListBlock = 1024, kListPer = 4;  // transactions per block and thread

__global__ __launch_bounds__(kListBlock) void kv_commit_list_kernel(
    uint32_t B, const uint8_t *__restrict__ doomed, const uint8_t *__restrict__ raw_flag,
    const uint8_t *__restrict__ war_flag, uint8_t epoch, uint64_t *__restrict__ bitmap, uint32_t *__restrict__ list,
    DeviceCounters *__restrict__ ctr)
{
    constexpr uint32_t kWaves = kListBlock / 64;
    __shared__ uint32_t s_cnt[kListPer * kWaves], s_base;
    const uint32_t first = blockIdx.x * (kListPer * kListBlock), wave = threadIdx.x / 64;
    unsigned long long m[kListPer];
#pragma unroll
    for (uint32_t r = 0; r < kListPer; ++r) {
        const uint32_t t = first + r * kListBlock + threadIdx.x, j = t < B ? t : 0u;
        const uint8_t d = doomed[j], ra = raw_flag[j], wa = war_flag[j];
        m[r] = __ballot(t < B && d != epoch && !(ra == epoch && wa == epoch));
    }
#pragma unroll
    for (uint32_t r = 0; r < kListPer; ++r) {
        if (lane_id() != 0) continue;
        const uint32_t t = first + r * kListBlock + wave * 64;
        if (t < B) bitmap[t / 64] = m[r];
        s_cnt[r * kWaves + wave] = (uint32_t)__popcll(m[r]);
    }
    __syncthreads();
    if (wave == 0) {
        const uint32_t c = s_cnt[lane_id()];
        uint32_t inc = c;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const uint32_t x = __shfl_up(inc, d);
            if (lane_id() >= d) inc += x;
        }
        s_cnt[lane_id()] = inc - c;
        if (lane_id() == 63) {
            const uint32_t left = B - first, live = left < kListPer * kListBlock ? left : kListPer * kListBlock;
            s_base = inc ? atomicAdd(&ctr->kv_list_n, inc) : 0u;
            add_counts(ctr, blockIdx.x % kCounterStripes, LTPG_TYPE_KV, inc, live);
        }
    }
    __syncthreads();
#pragma unroll
    for (uint32_t r = 0; r < kListPer; ++r)
        if ((m[r] >> lane_id()) & 1ull)
            list[s_base + s_cnt[r * kWaves + wave] + (uint32_t)__popcll(m[r] & ((1ull << lane_id()) - 1ull))] =
                first + r * kListBlock + threadIdx.x;
}
static_assert(kListPer * kListBlock / 64 == 64, "one wave scans the counts");

// Read-out of the listed transactions.  Slot-major batches: a wave takes one
// slot of 64 consecutive entries, whose op loads and read values are nearly
// consecutive; request-major ones: 64 consecutive op slots.
__global__ __launch_bounds__(kBlock) void kv_readout_list_kernel(
    const uint64_t *__restrict__ keys, const uint32_t *__restrict__ meta, uint32_t B, uint32_t S, uint64_t rows,
    uint32_t fields, uint32_t fw, uint32_t fsw, const uint32_t *__restrict__ table, uint32_t *__restrict__ read_values,
    const uint32_t *__restrict__ commits, const DeviceCounters *__restrict__ ctr, uint32_t max_scan, uint32_t L, bool rm)
{
    __shared__ StageList s_stage[kBlock / 64];
    StageList &list = s_stage[threadIdx.x / 64];
    const FieldLanes lanes(fw);
    const uint32_t n = ctr->kv_list_n;
    const uint32_t chunks = (n + 63) / 64;
    const uint32_t units = rm ? (n * S + 63) / 64 : chunks * S;  // n * S <= 2^30
    uint32_t pending = 0;
    for (uint32_t u = blockIdx.x * (kBlock / 64) + __builtin_amdgcn_readfirstlane(threadIdx.x / 64); u < units;
         u += gridDim.x * (kBlock / 64)) {
        uint32_t j, s;
        if (rm) {
            const uint32_t f = u * 64 + (uint32_t)lane_id();
            j = f / S;
            s = f - j * S;
        } else {
            s = u / chunks;
            j = (u - s * chunks) * 64 + (uint32_t)lane_id();
        }
        const uint32_t t = commits[j < n ? j : 0u];
        const Op o = load_op(keys, meta, op_at(s, t, B, S, rm), j < n, rows, fields, max_scan);
        pending = read_out(o, (uint64_t)s * B + t, list, pending, lanes, table, read_values, fields, fw, fsw, L);
    }
    if (pending) stage_flush(list, pending, lanes, table, read_values);
}

// One round of 64 listed transactions, a lane each, whose slots are runs of 64.
// The meta words of all slots come first and say which keys to load; a lane's
// write fields wait in LDS, `fields` [slot][lane], to be folded.
__device__ __forceinline__ uint32_t write_slots(const WriteArgs &a, uint32_t t, uint32_t (*fields)[64],
                                                StageList &list, uint32_t pending, const FieldLanes &lanes)
{
    const uint32_t lane = (uint32_t)lane_id(), at = t < a.B ? t : 0u;
    uint32_t writes = 0;
#pragma unroll 4
    for (uint32_t s = 0; s < a.S; ++s)
        writes |= (uint32_t)((a.meta[(uint64_t)s * a.B + at] & 3u) == LTPG_KV_WRITE) << s;
    if (t >= a.B) writes = 0;
    const uint32_t step = a.values == LTPG_VALUES_RMW ? (a.tids[at] | 1u) : 0u;
    uint32_t n = 0;
    while (__ballot(writes != 0)) {
        Op o[4];
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) {
            const bool has = writes != 0;
            const uint32_t s = has ? (uint32_t)__ffs(writes) - 1u : 0u;
            writes &= writes - 1u;
            o[u] = load_op(a.keys, a.meta, (uint64_t)s * a.B + at, has, a.rows, a.fields);
        }
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u)  // writes to the hot row go through kv_hot_sum_kernel
            if (o[u].valid && o[u].row != a.hot) fields[n++][lane] = (uint32_t)(o[u].row * a.fields) + o[u].field;
    }
    for (uint32_t k = 0; __ballot(k < n); k += 4) {
        // fold duplicates: the first write of a field counts them all
        uint32_t mine[4], count[4] = {0, 0, 0, 0};
        bool first[4];
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) {
            first[u] = k + u < n;
            const uint32_t f = fields[first[u] ? k + u : 0u][lane];
            mine[u] = first[u] ? f : 0u;  // a lane without one holds a field of the table all the same
        }
#pragma unroll 2
        for (uint32_t i = 0; __ballot(i < n); ++i) {
            const uint32_t f = fields[i < n ? i : 0u][lane];
#pragma unroll
            for (uint32_t u = 0; u < 4; ++u) {
                const bool same = i < n && f == mine[u];
                count[u] += same;
                first[u] &= !(same && i < k + u);
            }
        }
        if (a.fw < 4) {
            for (uint32_t w = 0; w < a.fw; ++w) {
                uint32_t v[4];
#pragma unroll
                for (uint32_t u = 0; u < 4; ++u) v[u] = a.table[(uint64_t)mine[u] * a.fsw + w];
#pragma unroll
                for (uint32_t u = 0; u < 4; ++u)
                    if (first[u]) a.table[(uint64_t)mine[u] * a.fsw + w] = v[u] + step * count[u];
            }
            continue;
        }
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) {
            const uint64_t off = (uint64_t)mine[u] * a.fsw;
            pending = stage_push(list, pending, first[u], off, off, step * count[u]);
            if (pending >= 64) {
                stage_flush(list, pending, lanes, a.table, a.table);
                pending = 0;
            }
        }
    }
    return pending;
}

// WRITEBACK of the listed transactions: 64 / G per round, or of a long list 64
// (write_slots); entries beyond a smaller current batch (the phase without a
// fresh CHECK) are left out.  Listed transactions lie close together, so their
// slots come in runs, while lane groups read a line per slot and transaction,
// and the keys of reads too: 1,013,000 commits of 1 to 10 ops, a tenth of them
// writes, 142 us in groups, 45 so (100-byte fields), 131,000 24 / 11; of 1 to 16 ops, half of
// them writes, 456,000 commits 160 / 112, 203,000 70 / 56, 115,000 40 / 38.  A
// lane's chain is longer, though, and few waves do not hide it: 62,000 of the
// latter 24 / 33, 254,000 of one or two writes 21 / 22 (935,000: 89 / 81).
constexpr uint32_t kSlotCommits = 1u << 17, kSlotOps = 1u << 20;
template <int G>
__global__ __launch_bounds__(kBlock) void kv_writeback_list_kernel(WriteArgs a, const uint32_t *__restrict__ commits,
                                                                  const DeviceCounters *__restrict__ ctr, bool slots)
{
    constexpr bool kSlots = G <= 16;  // op slots that fit LDS
    __shared__ StageList s_stage[kBlock / 64];
    __shared__ uint32_t s_fields[kSlots ? kBlock / 64 : 1][kSlots ? G : 1][64];
    end_epoch(a.end);
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    StageList &list = s_stage[wave];
    const FieldLanes lanes(a.fw);
    const uint32_t n = ctr->kv_list_n;
    uint32_t pending = 0;
    if (kSlots && slots && n >= kSlotCommits && n * a.S >= kSlotOps) {
        for (uint32_t j0 = (blockIdx.x * (kBlock / 64) + wave) * 64; j0 < n; j0 += gridDim.x * kBlock) {
            const uint32_t j = j0 + (uint32_t)lane_id();
            pending = write_slots(a, j < n ? commits[j] : a.B, s_fields[kSlots ? wave : 0], list, pending, lanes);
        }
    } else {
        constexpr uint32_t PER = 64 / G;
        const uint32_t grp = (uint32_t)lane_id() / G;
        for (uint32_t j0 = (blockIdx.x * (kBlock / 64) + wave) * PER; j0 < n; j0 += gridDim.x * (kBlock / 64) * PER) {
            const uint32_t t = j0 + grp < n ? commits[j0 + grp] : a.B;
            pending = write_round<G>(a, t < a.B, t < a.B ? t : 0u, list, pending, lanes);
        }
    }
    if (pending) stage_flush(list, pending, lanes, a.table, a.table);
}

// One small epoch in one workgroup (LTPG_TUNE_SMALL_EPOCH, and the served
// form's epochs): EXECUTE, read marking, CHECK with the read-out, and
// WRITEBACK back to back, separated by workgroup barriers instead of kernel
// boundaries.  The rules are those of the fast form (kv_execute_dedup_kernel,
// kv_mark_reads_kernel, kv_check_fast_kernel, kv_writeback_kernel) with the
// whole epoch in one workgroup: the ops, TIDs and conflict flags sit in LDS,
// and the W registrations go to an LDS hash of the written rows (row + 1 ->
// minimum TID << 24 | position) instead of the per-row registers in HBM,
// which this path never touches.  The batch may sit in pinned host memory
// (read once).  With seq_out the commit bitmap is also written to host_bits
// and then seq is stored there with a system-scope release, as
// publish_kernel does after a multi-kernel epoch.  With result the commit count
// and the range errors go there instead of the counters.  A hot row (at most
// kSmallHotFields fields) never registers or conflicts, and its committed
// deltas are summed per field in LDS and added to the row with the other
// writes; rows < 2^32 - 1.
constexpr uint32_t kSmallBlock = 1024;
constexpr uint32_t kSmallOps = LTPG_SMALL_EPOCH_OPS;
constexpr uint32_t kSmallPer = kSmallOps / kSmallBlock;  // op slots per thread
constexpr uint32_t kSmallSlots = 2 * kSmallOps;          // hash load <= 1/2: probing always ends
constexpr uint32_t kSmallUnroll = 4;                     // 16-byte pieces in flight per thread
constexpr uint32_t kSmallMerge = 8;                      // the same in the one-round copy
constexpr uint32_t kSmallHotFields = 1024;               // fields of a table with a hot row
constexpr uint32_t kSmallCopies = kSmallOps + kSmallHotFields;

__device__ __forceinline__ uint32_t small_hash(uint64_t row)
{
    return (uint32_t)((row * 0x9E3779B97F4A7C15ull) >> 40) & (kSmallSlots - 1);
}

// Slot of a written row in the hash, or -1 if no op of the epoch writes it.
__device__ __forceinline__ int small_find(const uint32_t *s_key, uint64_t row)
{
    const uint32_t key = (uint32_t)row + 1u;
    for (uint32_t h = small_hash(row);; h = (h + 1) & (kSmallSlots - 1)) {
        const uint32_t k = s_key[h];
        if (k == key) return (int)h;
        if (k == 0u) return -1;
    }
}

__global__ __launch_bounds__(kSmallBlock) void kv_small_epoch_kernel(
    const uint64_t *__restrict__ keys, const uint32_t *__restrict__ meta, const uint32_t *__restrict__ tids,
    uint32_t B, uint32_t S, bool rm, uint64_t rows, uint32_t fields, uint32_t fw, uint32_t fsw, uint32_t rsw,
    uint32_t max_scan, uint32_t L, uint32_t values, uint64_t hot, uint32_t *__restrict__ table,
    uint32_t *__restrict__ read_values, uint64_t *__restrict__ bitmap, uint64_t *__restrict__ host_bits,
    uint64_t *seq_out, uint64_t seq, uint32_t *__restrict__ result, DeviceCounters *__restrict__ ctr)
{
    __shared__ uint64_t s_row[kSmallOps];
    __shared__ uint32_t s_meta[kSmallOps];
    __shared__ uint32_t s_tid[kSmallOps];
    __shared__ uint32_t s_key[kSmallSlots];            // row + 1 of a written row, 0 = empty
    __shared__ unsigned long long s_min[kSmallSlots];  // its writers' minimum TID << 24 | position
    __shared__ uint8_t s_waw[kSmallOps], s_raw[kSmallOps], s_war[kSmallOps];
    __shared__ uint32_t s_list[kSmallOps];             // committed transactions
    __shared__ uint32_t s_add[kSmallCopies];           // of a copy: a write's delta, a read's rows
    __shared__ unsigned long long s_bits[kSmallOps / 64];  // the commit bitmap
    __shared__ uint32_t s_hot[kSmallHotFields];        // committed hot-row deltas per field
    __shared__ uint32_t s_n, s_bad, s_reads, s_writes;
    // the copies, in the hash's place: committed reads from the front, folded
    // writes from the back
    unsigned long long *s_field = s_min;  // the table's field
    uint32_t *s_slot = s_key;             // a read's op slot
    static_assert(kSmallCopies <= kSmallSlots, "the copies fit the hash");
    const uint32_t n = B * S;
    // the batch: every load issued before the first use
    uint64_t r[kSmallPer];
    uint32_t m[kSmallPer], tv[kSmallPer];
#pragma unroll
    for (uint32_t k = 0; k < kSmallPer; ++k) {
        const uint32_t i = k * kSmallBlock + threadIdx.x;
        r[k] = keys[i < n ? i : 0u];
        m[k] = meta[i < n ? i : 0u];
        tv[k] = tids[i < B ? i : 0u];
    }
    for (uint32_t k = threadIdx.x; k < kSmallSlots; k += kSmallBlock) {
        s_key[k] = 0u;
        s_min[k] = ~0ull;
    }
    const bool has_hot = hot < rows;
    if (has_hot)
        for (uint32_t f = threadIdx.x; f < fields; f += kSmallBlock) s_hot[f] = 0u;
    // the epoch's commit counts start at zero (thread 0 adds to them last)
    if (!result)
        for (uint32_t c = threadIdx.x; c < kCounterStripes * kCountedTypes; c += kSmallBlock)
            ctr->commits[c / kCountedTypes][c % kCountedTypes] = 0;
    if (threadIdx.x == 0) {
        s_n = 0;
        s_bad = 0;
        s_reads = 0;
        s_writes = 0;
    }
#pragma unroll
    for (uint32_t k = 0; k < kSmallPer; ++k) {
        const uint32_t i = k * kSmallBlock + threadIdx.x;
        if (i < n) {
            s_row[i] = r[k];
            s_meta[i] = m[k];
        }
        if (i < B) {
            s_tid[i] = tv[k];
            s_waw[i] = 0;
            s_raw[i] = 0;
            s_war[i] = 0;
        }
    }
    // (the counter stores and thread 0's later atomics meet in one L2; the
    // barriers order them)
    __syncthreads();
    // EXECUTE: W registrations into the hash
    uint32_t bad = 0;
#pragma unroll
    for (uint32_t k = 0; k < kSmallPer; ++k) {
        const uint32_t i = k * kSmallBlock + threadIdx.x;
        if (i >= n) continue;
        const Op o = decode_op(r[k], m[k], rows, fields, max_scan);
        bad += (o.kind != LTPG_KV_NONE && !o.valid) ? 1u : 0u;
        if (!o.valid || o.kind != LTPG_KV_WRITE || o.row == hot) continue;  // hot-row writes never register
        const uint32_t t = txn_of(i, B, S, rm);
        const uint32_t key = (uint32_t)o.row + 1u;
        uint32_t h = small_hash(o.row);
        while (true) {
            const uint32_t prev = atomicCAS(&s_key[h], 0u, key);
            if (prev == 0u || prev == key) break;
            h = (h + 1) & (kSmallSlots - 1);
        }
        atomicMin(&s_min[h], ((unsigned long long)s_tid[t] << kTidShift) | t);
    }
    if (bad) atomicAdd(&s_bad, bad);
    __syncthreads();
    // waw of every write; raw of every read, war of the row's minimum writer
    // when a higher-priority transaction reads it
#pragma unroll
    for (uint32_t k = 0; k < kSmallPer; ++k) {
        const uint32_t i = k * kSmallBlock + threadIdx.x;
        if (i >= n) continue;
        const Op o = decode_op(r[k], m[k], rows, fields, max_scan);
        if (!o.valid) continue;
        const uint32_t t = txn_of(i, B, S, rm);
        const unsigned long long me = ((unsigned long long)s_tid[t] << kTidShift) | t;
        if (o.kind == LTPG_KV_WRITE) {
            if (o.row != hot && s_min[small_find(s_key, o.row)] < me) s_waw[t] = 1;
            continue;
        }
        bool raw = false;
        for (uint32_t q = 0; q < o.len; ++q) {  // a scan: every row of its range
            if (o.row + q == hot) continue;  // the hot row never conflicts
            const int h = small_find(s_key, o.row + q);
            if (h < 0) continue;
            const unsigned long long w = s_min[h];
            if (w < me)
                raw = true;
            else if (w > me)
                s_war[w & kPosMask] = 1;
        }
        if (raw) s_raw[t] = 1;
    }
    __syncthreads();
    // CHECK: commit bits, the bitmap and the list of committed transactions
    const uint32_t nw = (B + 63) / 64;
    for (uint32_t t0 = 0; t0 < B; t0 += kSmallBlock) {
        const uint32_t t = t0 + threadIdx.x;
        const bool c = t < B && !s_waw[t] && !(s_raw[t] && s_war[t]);
        const unsigned long long bits = __ballot(c);
        if (c) s_list[atomicAdd(&s_n, 1u)] = t;
        if (lane_id() == 0 && t / 64 < nw) {
            bitmap[t / 64] = bits;
            s_bits[t / 64] = bits;
        }
    }
    __syncthreads();
    const uint32_t nc = s_n;
    // list the copies, G lanes per committed transaction (lane = slot): each
    // read, and the first write slot of a transaction on a field, which writes
    // word + count * delta, the others nothing.  Hot-row writes add their
    // delta to the field's sum instead (kv_hot_sum_kernel's reduce).
    const bool rmw = values == LTPG_VALUES_RMW;  // copy-back changes nothing
    const uint32_t G = S <= 1 ? 1u : 1u << (32 - __clz((int)(S - 1)));
    const uint32_t sl = (uint32_t)lane_id() % G, grp = (uint32_t)lane_id() / G, txns = 64 / G;
    for (uint32_t j0 = (threadIdx.x / 64) * txns; j0 < nc; j0 += kSmallBlock / G) {
        const bool has = j0 + grp < nc && sl < S;
        const uint32_t t = has ? s_list[j0 + grp] : 0u;
        const uint32_t i = has ? (rm ? t * S + sl : sl * B + t) : 0u;
        const Op o = decode_op(s_row[i], s_meta[i], rows, fields, max_scan);
        const bool any_wr = has && rmw && o.valid && o.kind == LTPG_KV_WRITE;
        if (any_wr && o.row == hot) atomicAdd(&s_hot[o.field], s_tid[t] | 1u);
        const bool wr = any_wr && o.row != hot, rd = has && o.valid && o.kind != LTPG_KV_WRITE;
        const unsigned long long wm = __ballot(wr), rdm = __ballot(rd);
        const uint64_t key = o.row * fields + o.field;
        uint32_t count = 0;
        bool first = wr;
        for (uint32_t k = 0; wm && k < S; ++k) {
            const uint64_t kk = __shfl(key, (int)(grp * G + k));
            if (((wm >> (grp * G + k)) & 1ull) && kk == key) {
                ++count;
                first &= k >= sl;
            }
        }
        const unsigned long long fm = __ballot(first), below = (1ull << lane_id()) - 1ull;
        uint32_t r0 = 0, w0 = 0;
        if (lane_id() == 0) {
            if (rdm) r0 = atomicAdd(&s_reads, (uint32_t)__popcll(rdm));
            if (fm) w0 = atomicAdd(&s_writes, (uint32_t)__popcll(fm));
        }
        r0 = __shfl(r0, 0);
        w0 = __shfl(w0, 0);
        const uint32_t at = rd ? r0 + (uint32_t)__popcll(rdm & below)
                               : kSmallCopies - 1 - (w0 + (uint32_t)__popcll(fm & below));
        if (rd || first) {
            s_field[at] = key;
            s_slot[at] = sl * B + t;
            s_add[at] = rd ? o.len : count * (s_tid[t] | 1u);
        }
    }
    __syncthreads();
    if (has_hot && rmw) {
        for (uint32_t f = threadIdx.x; f < fields; f += kSmallBlock) {
            if (s_hot[f] == 0) continue;
            const uint32_t at = kSmallCopies - 1 - atomicAdd(&s_writes, 1u);
            s_field[at] = hot * fields + f;
            s_add[at] = s_hot[f];
        }
        __syncthreads();
    }
    // read-out of the committed reads and write-back of the committed
    // writes, 16 bytes per lane (FieldLanes).  Reads see the snapshot: when
    // all fit one round, every load is issued before a barrier and every store
    // after it; otherwise the read-out runs in rounds, then a barrier, then the
    // write-back.  1,024 transactions of two ops on 100-byte fields, whole
    // epoch: 102 us word by word with each word's op decoded again, 33 so;
    // on 1 KB fields 623 and 165.
    const uint32_t total_r = s_reads * L, total = total_r + s_writes;
    const FieldLanes lanes(max(fw, 4u));
    const uint32_t mine = threadIdx.x >> lanes.log_lanes, per = kSmallBlock >> lanes.log_lanes;
    struct Copy {
        uint64_t src, dst;
        uint32_t add;
        bool ok, read;
        Words4 v;
    };
    const auto look = [&](uint32_t x, uint32_t end, Copy &c) {
        c.ok = lanes.on && x < end;
        c.read = x < total_r;
        c.src = c.dst = c.add = 0;
        if (!c.ok) return;
        if (c.read) {
            const uint32_t e = L == 1 ? x : x / L, q = x - e * L;  // row q of a scan
            c.ok = q < s_add[e];
            if (c.ok) c.src = (s_field[e] + (uint64_t)q * fields) * fsw;
            c.dst = ((uint64_t)s_slot[e] * L + q) * rsw;
        } else {
            const uint32_t e = kSmallCopies - 1 - (x - total_r);
            c.src = c.dst = s_field[e] * fsw;
            c.add = s_add[e];
        }
    };
    const auto load = [&](Copy &c) {  // a lane without a copy loads from field 0
        const uint32_t *p = table + c.src + lanes.off;
        if (fw >= 4) {
            c.v = *reinterpret_cast<const Words4 *>(p);
            return;
        }
#pragma unroll
        for (uint32_t w = 0; w < 3; ++w) c.v.w[w] = p[min(w, fw - 1)];
    };
    const auto store = [&](const Copy &c) {
        if (!c.ok) return;
        uint32_t *p = (c.read ? read_values : table) + c.dst + lanes.off;
        Words4 v = c.v;
#pragma unroll
        for (uint32_t w = 0; w < 4; ++w) v.w[w] += c.add;
        if (fw >= 4) {
            *reinterpret_cast<Words4 *>(p) = v;
            return;
        }
#pragma unroll
        for (uint32_t w = 0; w < 3; ++w)
            if (w < fw) p[w] = v.w[w];
    };
    if (total <= kSmallMerge * per) {
        Copy c[kSmallMerge];
#pragma unroll
        for (uint32_t u = 0; u < kSmallMerge; ++u) look(u * per + mine, total, c[u]);
#pragma unroll
        for (uint32_t u = 0; u < kSmallMerge; ++u) load(c[u]);
        __syncthreads();
#pragma unroll
        for (uint32_t u = 0; u < kSmallMerge; ++u) store(c[u]);
    } else {
        for (uint32_t part = 0; part < 2; ++part) {
            const uint32_t end = part ? total : total_r;
            for (uint32_t x0 = part ? total_r : 0u; x0 < end; x0 += kSmallUnroll * per) {
                Copy c[kSmallUnroll];
#pragma unroll
                for (uint32_t u = 0; u < kSmallUnroll; ++u) look(x0 + u * per + mine, end, c[u]);
#pragma unroll
                for (uint32_t u = 0; u < kSmallUnroll; ++u) load(c[u]);
#pragma unroll
                for (uint32_t u = 0; u < kSmallUnroll; ++u) store(c[u]);
            }
            __syncthreads();
        }
    }
    if (threadIdx.x == 0 && result) {
        result[0] = nc;
        result[1] = s_bad;
    } else if (threadIdx.x == 0) {
        add_counts(ctr, 0, LTPG_TYPE_KV, nc, B);
        if (s_bad) atomicAdd(&ctr->range_errors, s_bad);
    }
    if (seq_out) {
        // one wave copies the bitmap to host memory, then releases seq at
        // system scope: a host that reads seq with an acquire load reads the
        // bitmap too
        __syncthreads();
        if (threadIdx.x < 64) {
            for (uint32_t w = threadIdx.x; w < nw; w += 64) host_bits[w] = s_bits[w];
            __threadfence_system();
            if (threadIdx.x == 0) __hip_atomic_store(seq_out, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    }
}

// Hot row: committed writes to it add their delta (TID | 1 per word) in any
// order.  A block sums its transactions' deltas per field in LDS and adds
// each non-zero sum to one of kCounterStripes accumulator rows; then
// kv_hot_apply_kernel folds the stripes into the row and clears them.  Bound by
// latency: 16,000 transactions of 8 ops 4.7 + 6.6 us one slot and one stripe
// after the other, 3.5 + 4.6 with their loads in flight together.  (As one
// kernel whose last block folds: 9.7 us, and 260 more for 3,000 fields.)
constexpr uint32_t kHotLdsFields = 1024;

__global__ __launch_bounds__(kBlock) void kv_hot_sum_kernel(
    const uint64_t *__restrict__ keys, const uint32_t *__restrict__ meta,
    const uint32_t *__restrict__ tids, uint32_t B, uint32_t S, uint64_t rows, uint32_t fields, uint64_t hot,
    const uint64_t *__restrict__ bitmap, uint32_t *__restrict__ acc, bool rm)
{
    __shared__ uint32_t bins[kHotLdsFields];
    const bool lds = fields <= kHotLdsFields;
    if (lds)
        for (uint32_t f = threadIdx.x; f < fields; f += kBlock) bins[f] = 0;
    __syncthreads();
    uint32_t *stripe = acc + (uint64_t)(blockIdx.x % kCounterStripes) * fields;
    const uint32_t t = blockIdx.x * kBlock + threadIdx.x;
    const bool committed = t < B && ((bitmap[t / 64] >> (t % 64)) & 1ull);
    if (committed) {
        const uint32_t delta = tids[t] | 1u;
        constexpr uint32_t U = 8;
        for (uint32_t s0 = 0; s0 < S; s0 += U) {
            Op o[U];
#pragma unroll
            for (uint32_t u = 0; u < U; ++u)
                o[u] = load_op(keys, meta, op_at(s0 + u, t, B, S, rm), s0 + u < S, rows, fields);
#pragma unroll
            for (uint32_t u = 0; u < U; ++u) {
                if (!o[u].valid || o[u].kind != LTPG_KV_WRITE || o[u].row != hot) continue;
                if (lds) atomicAdd(&bins[o[u].field], delta);
                else atomicAdd(&stripe[o[u].field], delta);
            }
        }
    }
    __syncthreads();
    if (lds)
        for (uint32_t f = threadIdx.x; f < fields; f += kBlock)
            if (bins[f]) atomicAdd(&stripe[f], bins[f]);
}

__global__ __launch_bounds__(kBlock) void kv_hot_apply_kernel(uint32_t *__restrict__ table, uint64_t hot,
                                                             uint32_t fields, uint32_t fw, uint32_t fsw,
                                                             uint32_t *__restrict__ acc)
{
    const uint32_t f = blockIdx.x * kBlock + threadIdx.x;
    if (f >= fields) return;
    // every load before the first store, which might be to the next one's place
    uint32_t v[kCounterStripes], total = 0;
#pragma unroll
    for (int k = 0; k < kCounterStripes; ++k) v[k] = acc[(uint64_t)k * fields + f];
#pragma unroll
    for (int k = 0; k < kCounterStripes; ++k) {
        total += v[k];
        if (v[k]) acc[(uint64_t)k * fields + f] = 0;
    }
    if (total == 0) return;
    uint32_t *w = table + (hot * fields + f) * (uint64_t)fsw;
    for (uint32_t k = 0; k < fw; ++k) w[k] += total;
}

// Rows `idx` of the table, every field, packed (row i of the output holds
// fields * fw words); one thread per output word.  The caller has checked
// every index against the table.
__global__ __launch_bounds__(kBlock) void kv_gather_rows_kernel(const uint32_t *__restrict__ table,
                                                                const uint64_t *__restrict__ idx, uint64_t n,
                                                                uint32_t fields, uint32_t fw, uint32_t fsw,
                                                                uint32_t *__restrict__ out)
{
    const uint64_t per = (uint64_t)fields * fw;
    for (uint64_t x = (uint64_t)blockIdx.x * kBlock + threadIdx.x; x < n * per; x += (uint64_t)gridDim.x * kBlock) {
        const uint64_t i = x / per, r = x % per, f = r / fw, w = r % fw;
        out[x] = table[(idx[i] * fields + f) * fsw + w];
    }
}

// ---- served key-value epochs in one persistent workgroup ------------------
//
// The device loop's op decode and write hash in 32-bit row arithmetic (its
// tables have fewer than 2^32 - 1 rows): the same fields, validity and
// scan length as decode_op, with a multiplicative hash on 32 bits.
struct Op32 {
    uint32_t row, kind, field, len;
    bool valid;
};

__device__ __forceinline__ Op32 decode_op32(uint64_t key, uint32_t m, uint32_t rows, uint32_t fields,
                                            uint32_t max_scan)
{
    Op32 o;
    o.kind = m & 3u;
    o.field = (m >> 8) & 0xffffu;
    const uint32_t sl = (m >> 24) + 1u;
    o.row = (uint32_t)key;
    o.valid = o.kind != LTPG_KV_NONE && (key >> 32) == 0ull && o.row < rows && o.field < fields &&
              (o.kind != LTPG_KV_SCAN || sl <= max_scan);
    const uint32_t left = o.row < rows ? rows - o.row : 0u;
    o.len = !o.valid || o.kind == LTPG_KV_WRITE ? 0u : o.kind == LTPG_KV_READ ? 1u : (sl < left ? sl : left);
    return o;
}

// The loop keeps an op as (row, meta) in 32 bits each, validated once when
// the request is admitted: meta bit 2 (never set in an op's meta by its
// layout: kind in bits 0-1, field in 8-23, scan length in 24-31) records that
// the op is valid.
constexpr uint32_t kLoopValid = 4u;

__device__ __forceinline__ uint32_t loop_pack_meta(uint64_t key, uint32_t m, uint32_t rows, uint32_t fields,
                                                   uint32_t max_scan)
{
    const Op32 o = decode_op32(key, m, rows, fields, max_scan);
    return (m & ~kLoopValid) | (o.valid ? kLoopValid : 0u);
}

__device__ __forceinline__ Op32 loop_decode(uint32_t row, uint32_t m, uint32_t rows)
{
    Op32 o;
    o.kind = m & 3u;
    o.field = (m >> 8) & 0xffffu;
    o.row = row;
    o.valid = (m & kLoopValid) != 0u;
    const uint32_t sl = (m >> 24) + 1u, left = rows - row;  // (row < rows when valid)
    o.len = !o.valid || o.kind == LTPG_KV_WRITE ? 0u : o.kind == LTPG_KV_READ ? 1u : (sl < left ? sl : left);
    return o;
}

static_assert(kSmallSlots == 4096, "loop_hash yields 12 bits");
__device__ __forceinline__ uint32_t loop_hash(uint32_t row) { return (row * 0x9E3779B1u) >> 20; }

__device__ __forceinline__ int loop_find(const uint32_t *s_key, uint32_t row)
{
    const uint32_t key = row + 1u;
    for (uint32_t h = loop_hash(row);; h = (h + 1) & (kSmallSlots - 1)) {
        const uint32_t k = s_key[h];
        if (k == key) return (int)h;
        if (k == 0u) return -1;
    }
}

// kv_serve_loop_kernel runs the served form's key-value epochs back to back
// in one 1024-thread workgroup, without a kernel launch or a host round trip
// between them:
//
//   admission  the requests aborted by the last epoch (kept in LDS, in
//              priority order) head the next epoch, followed by arrivals
//              taken from the request ring in arrival order, up to the epoch
//              cap.  Priority inside an epoch is batch position, which is
//              arrival order: every carried request arrived before every new
//              one, and carried requests keep their relative order.  The
//              next epoch is decided and admitted right after an epoch's
//              CHECK, from arrivals prefetched during the epoch, into the
//              other halves of the double-buffered LDS arrays, so one
//              barrier separates two epochs; after an idle or stalled turn
//              (or an exit test) the loop's top admits from the ring;
//   phases     those of kv_small_epoch_kernel: W registrations in an LDS
//              hash of the written rows, read marking, Aria's commit rule,
//              read-out of committed reads (when the host keeps them) and
//              write-back of committed writes, the RMW delta being the low
//              32 bits of the arrival sequence number | 1;
//   results    one record per epoch in the done ring (pinned host memory),
//              written by wave 0 right after CHECK (wave 0 takes no part in
//              the write-back) and published by a system-scope release of
//              ctl->done_tail after it;
//   requeue    the aborted requests are compacted, in position order, to the
//              front of the other half of the double-buffered LDS op and
//              sequence arrays and head the next epoch.  Without kept reads
//              no barrier separates the write-back, the publish and the
//              requeue: wave 0 publishes while waves 1.. issue write-back
//              atomics.
//
// Every wait is bounded: the loop ends when the host sets ctl->stop, after
// idle_ticks without work, after stall_ticks with the done ring full and
// after slice_ticks in all; the kernel then saves the carried requests to
// device memory and clears ctl->running.  Control decisions are taken from
// values thread 0 broadcasts through LDS, so every wave leaves the loop at
// the same iteration.
constexpr uint32_t kLoopMaxT = kSmallOps;  // transactions per epoch at one op slot each
// s_waitcnt vmcnt(0) expcnt(7) lgkmcnt(15): wait for the wave's vector memory
// accesses only (gfx9 encoding: vmcnt in bits 3:0 and 15:14)
constexpr int kWaitVmcnt0 = 0x0F70;

__device__ __forceinline__ uint64_t sys_load(const uint64_t *p)
{
    return __hip_atomic_load(p, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_SYSTEM);
}

__device__ __forceinline__ void sys_store(uint64_t *p, uint64_t v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// A request-ring entry, written by the host: a system-scope load, which
// bypasses the GPU caches, so an entry of a ring slot the host has reused is
// never served from a line cached on an earlier lap.
template <typename T>
__device__ __forceinline__ T ring_load(const T *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Workgroup barrier for LDS only: it orders LDS accesses like __syncthreads
// but does not wait for the wave's global loads, which stay in flight across
// it (the served loop keeps PCIe reads in flight over several phases).
__device__ __forceinline__ void lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Exclusive prefix count of the flags of items k * kSmallBlock + threadIdx.x
// (k < kSmallPer, in item order): per-wave ballots, then one pass over the
// wave totals in LDS.  Returns the total; s_w holds 16 * kSmallPer + 1 words.
__device__ __forceinline__ uint32_t block_count_before(const bool (&f)[kSmallPer], uint32_t (&before)[kSmallPer],
                                                       uint32_t *s_w)
{
    constexpr uint32_t kWaves = kSmallBlock / 64;
    const uint32_t lane = (uint32_t)lane_id(), wave = threadIdx.x / 64;
    const unsigned long long lt = lane ? (~0ull >> (64 - lane)) : 0ull;
    uint32_t pre[kSmallPer];
#pragma unroll
    for (uint32_t k = 0; k < kSmallPer; ++k) {
        const unsigned long long m = __ballot(f[k]);
        pre[k] = (uint32_t)__popcll(m & lt);
        if (lane == 0) s_w[k * kWaves + wave] = (uint32_t)__popcll(m);
    }
    lds_sync();
    if (threadIdx.x == 0) {
        uint32_t run = 0;
        for (uint32_t j = 0; j < kSmallPer * kWaves; ++j) {
            const uint32_t c = s_w[j];
            s_w[j] = run;
            run += c;
        }
        s_w[kSmallPer * kWaves] = run;
    }
    lds_sync();
#pragma unroll
    for (uint32_t k = 0; k < kSmallPer; ++k) before[k] = s_w[k * kWaves + wave] + pre[k];
    const uint32_t total = s_w[kSmallPer * kWaves];
    lds_sync();
    return total;
}

// Unsigned division by a divisor fixed for the kernel's life (ops per
// request, field words): q = high 64 bits of n * M with M = floor(2^64 / d)
// + 1 (exactly 2^64 / d for a power of two), exact for every 32-bit n because
// n * d < 2^64 (Granlund and Montgomery, "Division by invariant integers
// using multiplication", 1994).  Two 32x32->64 multiplies instead of the
// ~25-instruction division sequence.
struct FastDiv {
    uint64_t m;
    uint32_t d;
    __device__ explicit FastDiv(uint32_t d_) : m(d_ > 1 ? ~0ull / d_ + 1ull : 0ull), d(d_) {}
    __device__ __forceinline__ uint32_t div(uint32_t n) const
    {
        if (d == 1) return n;
        const uint64_t hi = (uint64_t)n * (uint32_t)(m >> 32);
        const uint64_t lo = ((uint64_t)n * (uint32_t)m) >> 32;
        return (uint32_t)((hi + lo) >> 32);
    }
};

__global__ __launch_bounds__(kSmallBlock) void kv_serve_loop_kernel(ServeLoopArgs a)
{
    // op arrays, double-buffered: the requeue writes the carried requests
    // into the half the next epoch reads while this epoch's half is read
    // (rows and validated metas: loop_pack_meta)
    __shared__ uint32_t s_rowb[2][kSmallOps];
    __shared__ uint32_t s_metab[2][kSmallOps];
    __shared__ uint64_t s_seqb[2][kLoopMaxT];        // arrival sequence number by position, double-buffered
    __shared__ uint32_t s_key[kSmallSlots];          // row + 1 of a written row, 0 = empty
    __shared__ uint32_t s_min[kSmallSlots];          // its writers' minimum position
    // conflict flags by position, double-buffered: the next epoch's are
    // cleared while waves may still read this epoch's
    __shared__ uint8_t s_wawb[2][kLoopMaxT], s_rawb[2][kLoopMaxT], s_warb[2][kLoopMaxT];
    __shared__ uint32_t s_list[kLoopMaxT];           // committed transactions, in position order
    __shared__ uint32_t s_dst[kLoopMaxT];            // an aborted position's place in the next epoch, ~0 if committed
    // the same, one copy per wave, for epochs of at most 64 transactions
    // (each wave counts the commits itself)
    __shared__ uint32_t s_listw[kSmallBlock / 64][64], s_dstw[kSmallBlock / 64][64];
    __shared__ uint32_t s_w[16 * kSmallPer + 1];
    __shared__ uint64_t s_busy;  // wall-clock ticks inside epochs
    // control words, double-buffered: thread 0 fills the half the loop is
    // not reading, and every wave switches halves after the next barrier,
    // so reading them needs no barrier of its own
    __shared__ uint64_t s_ctl[2][4];
    __shared__ uint32_t s_bad;

    // kernel arguments as locals: the lambdas below capture by reference,
    // and a reference to the argument struct would force it into scratch
    const uint32_t S = a.S, fields = a.fields, fw = a.fw, fsw = a.fsw, L = a.L, max_scan = a.max_scan;
    const uint32_t values = a.values;
    const FastDiv dS(S), dfw(fw), dper(L * fw);
    const uint64_t rows = a.rows, hot = a.hot, done_mask = a.done_mask;
    // rows < 2^32 - 1 here (kv_serve_loop_ok): 32-bit rows; a hot row
    // outside the table becomes a value no row takes
    const uint32_t rows32 = (uint32_t)rows, hot32 = hot < rows ? (uint32_t)hot : 0xFFFFFFFFu;
    ServeCtl *ctl = a.ctl;
    uint32_t *table = a.table;
    uint32_t *reads = a.reads;
    uint64_t *done = a.done;
    // where the previous launch stopped (fields only the kernel writes)
    // (the start time too comes from thread 0: every exit test below must
    // give the same answer in every wave)
    __shared__ uint64_t s_start;
    if (threadIdx.x == 0) {
        s_ctl[0][0] = sys_load(&ctl->head);
        s_ctl[0][1] = sys_load(&ctl->done_tail);
        s_ctl[0][2] = sys_load(&ctl->epochs);
        s_ctl[0][3] = (sys_load(&ctl->n_carry) & 0xffffffffull) | (sys_load(&ctl->cap) << 32);
        s_start = wall_clock64();
    }
    __syncthreads();
    uint64_t head = s_ctl[0][0], done_tail = s_ctl[0][1], epoch = s_ctl[0][2];
    uint32_t n_carry = (uint32_t)(s_ctl[0][3] & 0xffffffffull), cap = (uint32_t)(s_ctl[0][3] >> 32);
    uint32_t cp = 0;  // the half of s_ctl being read
    uint32_t op = 0;  // the half of s_rowb / s_metab being read
    const uint64_t t_start = s_start;
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < n_carry * S; i += kSmallBlock) {
        s_rowb[0][i] = (uint32_t)a.carry_keys[i];  // saved by the last launch, already validated
        s_metab[0][i] = a.carry_meta[i];
    }
    for (uint32_t t = threadIdx.x; t < n_carry; t += kSmallBlock) s_seqb[0][t] = a.carry_seq[t];
    // the write hash starts empty; each epoch empties the slots its writes
    // took once its marking is done
    for (uint32_t h = threadIdx.x; h < kSmallSlots; h += kSmallBlock) {
        s_key[h] = 0u;
        s_min[h] = ~0u;
    }
    uint64_t t_work = t_start, code = 0;
    // profile: thread 0 stamps the end of each part (after its barrier)
    // (sums in LDS: a register array would be spilled)
    const bool prof = a.profile != 0;
    __shared__ uint64_t s_prof[kServeProfParts + 2];  // sums, then the last stamp and the epoch count
    if (prof && threadIdx.x == 0) {
        for (int k = 0; k < kServeProfParts; ++k) s_prof[k] = 0;
        s_prof[kServeProfParts] = t_start;
        s_prof[kServeProfParts + 1] = 0;
    }
    const auto stamp = [&](int part) {
        if (prof && threadIdx.x == 0) {
            const uint64_t t = wall_clock64();
            s_prof[part] += t - s_prof[kServeProfParts];
            s_prof[kServeProfParts] = t;
        }
    };
    // The host's control words (tail, stop, done_head) cross PCIe: during an
    // epoch thread 0 issues their loads after admission and stores the
    // values at the end of the epoch, so the next admission decides on
    // values at most one epoch old without waiting for them; only an idle or
    // stalled loop waits for a fresh read.  Ring entries are read only below
    // the tail so read (the host writes them before it advances the tail),
    // with ring_load, after the tail's load has returned.  poll() fills the
    // other half of s_ctl; the caller switches halves after a barrier.
    const auto poll = [&]() {
        if (threadIdx.x == 0) {
            uint64_t *c = s_ctl[cp ^ 1u];
            c[0] = __hip_atomic_load(&ctl->tail, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            c[1] = __hip_atomic_load(&ctl->stop, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            c[2] = __hip_atomic_load(&ctl->done_head, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            c[3] = wall_clock64();
        }
    };
    // Releases the records written so far: every lane of wave 0 (the lanes
    // that store records) issues a system-scope release fence, then lane 0
    // stores done_tail (with kept reads, every wave fenced its stores before
    // the barrier that precedes this).  A release-only fence: the acquire
    // half of __threadfence_system would also invalidate the L2.
    const auto publish = [&](uint64_t tail_value) {
        if (threadIdx.x < 64) {
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "");
            if (threadIdx.x == 0)
                __hip_atomic_store(&ctl->done_tail, tail_value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    };
    poll();
    if (threadIdx.x == 0) {
        s_busy = 0;
        s_bad = 0;
    }
    __syncthreads();
    cp ^= 1u;
    // The epoch about to run, uniform in every wave: admitted (its ops,
    // sequence numbers and zeroed flags already in half op, admitted by the
    // last epoch right after its CHECK), B transactions of which n_new new
    // arrivals, now its start time and tail_seen the ring tail it knows.
    bool admitted = false;
    uint32_t B = 0, n_new = 0;
    uint64_t now = 0, tail_seen = 0;
    while (true) {
        uint32_t *const s_row = s_rowb[op];
        uint32_t *const s_meta = s_metab[op];
        uint64_t *const s_seq = s_seqb[op];
        uint8_t *const s_waw = s_wawb[op], *const s_raw = s_rawb[op], *const s_war = s_warb[op];
        if (!admitted) {
        const uint64_t tail = s_ctl[cp][0], stop = s_ctl[cp][1], done_head = s_ctl[cp][2];
        now = s_ctl[cp][3];
        tail_seen = tail;
        if (stop) {
            code = kServeExitStop;
            break;
        }
        if (now - t_start > a.slice_ticks) {
            code = kServeExitSlice;
            break;
        }
        const uint64_t avail = tail > head ? tail - head : 0ull;
        const uint32_t room = cap > n_carry ? cap - n_carry : 0u;
        n_new = (uint32_t)(avail < room ? avail : (uint64_t)room);
        B = n_carry + n_new;
        if (B == 0) {
            if (now - t_work > a.idle_ticks) {
                code = kServeExitIdle;
                break;
            }
            __builtin_amdgcn_s_sleep(32);
            poll();
            lds_sync();
            cp ^= 1u;
            stamp(9);
            continue;
        }
        if (done_tail + 1 + B - done_head > done_mask + 1) {
            if (now - t_work > a.stall_ticks) {
                code = kServeExitStall;
                break;
            }
            __builtin_amdgcn_s_sleep(32);
            poll();
            lds_sync();
            cp ^= 1u;
            stamp(9);
            continue;
        }
        stamp(0);
        // admission after an idle turn, an exit test or a full done ring:
        // arrivals head .. head + n_new - 1 behind the carried requests, read
        // from the ring (every ring load issued before the first LDS store)
        {
            const uint32_t n = B * S, c0 = n_carry * S;
            uint64_t r[kSmallPer] = {};
            uint32_t m[kSmallPer] = {};
#pragma unroll
            for (uint32_t k = 0; k < kSmallPer; ++k) {
                const uint32_t i = k * kSmallBlock + threadIdx.x;
                const bool live = i >= c0 && i < n;
                const uint32_t jn = live ? dS.div(i - c0) : 0u;
                const uint64_t at = live ? ((head + jn) & a.ring_mask) * S + (i - c0 - jn * S) : 0ull;
                if (n_new) {  // uniform: no PCIe read for an epoch of carried requests
                    r[k] = ring_load(&a.ring_keys[at]);
                    m[k] = ring_load(&a.ring_meta[at]);
                }
            }
#pragma unroll
            for (uint32_t k = 0; k < kSmallPer; ++k) {
                const uint32_t i = k * kSmallBlock + threadIdx.x;
                if (i >= c0 && i < n) {
                    s_row[i] = (uint32_t)r[k];
                    s_meta[i] = loop_pack_meta(r[k], m[k], rows32, fields, max_scan);
                }
            }
        }
        for (uint32_t t = n_carry + threadIdx.x; t < B; t += kSmallBlock) s_seq[t] = head + (t - n_carry);
        for (uint32_t t = threadIdx.x; t < B; t += kSmallBlock) {
            s_waw[t] = 0;
            s_raw[t] = 0;
            s_war[t] = 0;
        }
        head += n_new;
        lds_sync();
        stamp(1);
        }  // !admitted
        const uint32_t n = B * S;
        // the arrivals this epoch took are in LDS (in every wave, before the
        // barrier above): their ring slots may be reused by the host
        if (threadIdx.x == 0 && n_new) __hip_atomic_store(&ctl->head, head, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        // the next admission's control words: loads in flight during the epoch
        uint64_t c_tail = 0, c_stop = 0, c_dh = 0;
        if (threadIdx.x == 0) {
            c_tail = __hip_atomic_load(&ctl->tail, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            c_stop = __hip_atomic_load(&ctl->stop, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            c_dh = __hip_atomic_load(&ctl->done_head, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
        // and its arrivals: the published requests after this admission, up
        // to a full epoch, loaded now and admitted into the next epoch right
        // after this one's CHECK
        const uint32_t pf_n = (uint32_t)(tail_seen - head < a.cap_max ? tail_seen - head : (uint64_t)a.cap_max);
        uint64_t pf_r[kSmallPer] = {};
        uint32_t pf_m[kSmallPer] = {};
#pragma unroll
        for (uint32_t k = 0; k < kSmallPer; ++k) {
            const uint32_t i = k * kSmallBlock + threadIdx.x;
            const uint32_t q = dS.div(i);
            if (i < pf_n * S) {
                const uint64_t at = ((head + q) & a.ring_mask) * S + (i - q * S);
                pf_r[k] = ring_load(&a.ring_keys[at]);
                pf_m[k] = ring_load(&a.ring_meta[at]);
            }
        }
        uint32_t r[kSmallPer];
        uint32_t m[kSmallPer];
#pragma unroll
        for (uint32_t k = 0; k < kSmallPer; ++k) {
            const uint32_t i = k * kSmallBlock + threadIdx.x;
            r[k] = i < n ? s_row[i] : 0u;
            m[k] = i < n ? s_meta[i] : 0u;
        }
        // EXECUTE: W registrations into the hash (priority = position).  A
        // single-row read takes a slot for its row as well (its minimum
        // stays ~0 unless a write registers there), so that the marking
        // below reads the row's minimum without probing; every slot taken is
        // kept for the marking.
        uint32_t bad = 0;
        uint32_t wslot[kSmallPer];  // ~0: no slot
#pragma unroll
        for (uint32_t k = 0; k < kSmallPer; ++k) {
            wslot[k] = ~0u;
            const uint32_t i = k * kSmallBlock + threadIdx.x;
            if (i >= n) continue;
            const Op32 o = loop_decode(r[k], m[k], rows32);
            bad += (o.kind != LTPG_KV_NONE && !o.valid) ? 1u : 0u;
            if (!o.valid || o.kind == LTPG_KV_SCAN || o.row == hot32) continue;
            const uint32_t key = o.row + 1u;
            uint32_t h = loop_hash(o.row);
            while (true) {
                const uint32_t prev = atomicCAS(&s_key[h], 0u, key);
                if (prev == 0u || prev == key) break;
                h = (h + 1) & (kSmallSlots - 1);
            }
            wslot[k] = h;
            if (o.kind == LTPG_KV_WRITE) atomicMin(&s_min[h], dS.div(i));
        }
        if (bad) atomicAdd(&s_bad, bad);
        lds_sync();
        stamp(2);
        // waw of every write; raw of every read, war of the row's minimum
        // writer when a higher-priority transaction reads it
#pragma unroll
        for (uint32_t k = 0; k < kSmallPer; ++k) {
            const uint32_t i = k * kSmallBlock + threadIdx.x;
            if (i >= n) continue;
            const Op32 o = loop_decode(r[k], m[k], rows32);
            if (!o.valid) continue;
            const uint32_t t = dS.div(i);
            if (o.kind == LTPG_KV_WRITE) {
                if (o.row != hot32 && s_min[wslot[k]] < t) s_waw[t] = 1;
                continue;
            }
            // (a minimum of ~0: no write registered the row)
            bool raw = false;
            if (o.kind == LTPG_KV_READ) {
                if (wslot[k] != ~0u) {
                    const uint32_t w = s_min[wslot[k]];
                    if (w < t)
                        raw = true;
                    else if (w > t && w != ~0u)
                        s_war[w] = 1;
                }
            } else {
                for (uint32_t q = 0; q < o.len; ++q) {
                    if (o.row + q == hot32) continue;
                    const int h = loop_find(s_key, o.row + q);
                    if (h < 0) continue;
                    const uint32_t w = s_min[h];
                    if (w < t)
                        raw = true;
                    else if (w > t && w != ~0u)
                        s_war[w] = 1;
                }
            }
            if (raw) s_raw[t] = 1;
        }
        // the control words loaded during the epoch, and the time, to LDS
        // before the barrier: every wave decides on them after CHECK
        if (threadIdx.x == 0) {
            uint64_t *cn = s_ctl[cp ^ 1u];
            cn[0] = c_tail;
            cn[1] = c_stop;
            cn[2] = c_dh;
            cn[3] = wall_clock64();
            s_busy += cn[3] - now;
        }
        lds_sync();
        stamp(3);
        // CHECK: commit bits and the committed list in position order.  An
        // epoch of at most 64 transactions (the common case under the
        // commit-based cap) is counted with one ballot: by every wave into
        // its own copies of the arrays, with no barrier after it, when the
        // host keeps no reads; else by wave 0 alone.
        uint32_t nc;
        const uint32_t *dstv = s_dst, *listv = s_list;  // the arrays this wave reads below
        if (B <= 64 && !reads) {
            const uint32_t t = (uint32_t)lane_id(), wave = threadIdx.x / 64;
            const bool ct = t < B && !s_waw[t] && !(s_raw[t] && s_war[t]);
            const unsigned long long m = __ballot(ct);
            const uint32_t bf = (uint32_t)__popcll(m & (t ? (~0ull >> (64 - t)) : 0ull));
            uint32_t *const dw = s_dstw[wave], *const lw = s_listw[wave];
            if (t < B) dw[t] = ct ? ~0u : t - bf;
            if (ct) lw[bf] = t;
            nc = (uint32_t)__popcll(m);
            dstv = dw;
            listv = lw;
            // the wave's lanes read each other's entries below: LDS accesses
            // of one wave complete in order; keep the compiler's order too
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            __builtin_amdgcn_wave_barrier();
            stamp(4);
        } else {
        if (B <= 64) {
            if (threadIdx.x < 64) {
                const uint32_t t = threadIdx.x;
                const bool ct = t < B && !s_waw[t] && !(s_raw[t] && s_war[t]);
                const unsigned long long m = __ballot(ct);
                const uint32_t bf = (uint32_t)__popcll(m & (t ? (~0ull >> (64 - t)) : 0ull));
                if (t < B) s_dst[t] = ct ? ~0u : t - bf;
                if (ct) s_list[bf] = t;
                if (t == 0) s_w[0] = (uint32_t)__popcll(m);
            }
        } else {
            bool c[kSmallPer];
            uint32_t before[kSmallPer];
#pragma unroll
            for (uint32_t k = 0; k < kSmallPer; ++k) {
                const uint32_t t = k * kSmallBlock + threadIdx.x;
                c[k] = t < B && !s_waw[t] && !(s_raw[t] && s_war[t]);
            }
            const uint32_t total = block_count_before(c, before, s_w);
#pragma unroll
            for (uint32_t k = 0; k < kSmallPer; ++k) {
                const uint32_t t = k * kSmallBlock + threadIdx.x;
                if (t < B) s_dst[t] = c[k] ? ~0u : t - before[k];
                if (c[k]) s_list[before[k]] = t;
            }
            if (threadIdx.x == 0) s_w[0] = total;
        }
        // With kept reads the read-out below loads the table, so the last
        // epoch's write-back atomics must be ordered before it: a barrier
        // with workgroup-scope release / acquire of global memory.  Without,
        // nothing in the loop reads the table and an LDS barrier suffices.
        if (reads)
            __syncthreads();
        else
            lds_sync();
        nc = s_w[0];
        stamp(4);
        }
        // The next epoch, decided now in every wave alike: the aborted
        // requests head it (the requeue below moves them), followed by the
        // prefetched arrivals up to its cap.  It is admitted now, into the
        // other halves, unless the host asked to stop, the slice is over, it
        // would be empty or the done ring has no room for its record; the
        // loop's top then decides again on fresh values.  The arrivals go to
        // LDS before the write-back: their loads returned during the phases
        // above, and no load result is then left pending behind the
        // write-back atomics (its first use would wait for those as well).
        const uint32_t carry_n = B - nc;
        uint32_t cap_n = a.cap_max;
        if (a.growth) {
            const uint64_t g = (uint64_t)a.growth * nc;
            cap_n = (uint32_t)(g < a.floor ? a.floor : (g > a.cap_max ? a.cap_max : g));
        }
        const uint64_t n_tail = s_ctl[cp ^ 1u][0], n_stop = s_ctl[cp ^ 1u][1], n_dh = s_ctl[cp ^ 1u][2],
                       n_now = s_ctl[cp ^ 1u][3];
        uint32_t new_n;
        {
            const uint64_t avail = n_tail > head ? n_tail - head : 0ull;
            const uint32_t room = cap_n > carry_n ? cap_n - carry_n : 0u;
            new_n = (uint32_t)(avail < room ? avail : (uint64_t)room);
            new_n = new_n < pf_n ? new_n : pf_n;
        }
        const uint32_t B_n = carry_n + new_n;
        const bool go = !n_stop && n_now - t_start <= a.slice_ticks && B_n > 0 &&
                        done_tail + 1 + B + 1 + B_n - n_dh <= done_mask + 1;
        if (go) {
            uint32_t *const nx_row = s_rowb[op ^ 1u] + (uint64_t)carry_n * S;
            uint32_t *const nx_meta = s_metab[op ^ 1u] + (uint64_t)carry_n * S;
#pragma unroll
            for (uint32_t k = 0; k < kSmallPer; ++k) {
                const uint32_t i = k * kSmallBlock + threadIdx.x;
                if (i < new_n * S) {
                    nx_row[i] = (uint32_t)pf_r[k];
                    nx_meta[i] = loop_pack_meta(pf_r[k], pf_m[k], rows32, fields, max_scan);
                }
            }
            for (uint32_t t = threadIdx.x; t < new_n; t += kSmallBlock) s_seqb[op ^ 1u][carry_n + t] = head + t;
            for (uint32_t t = threadIdx.x; t < B_n; t += kSmallBlock) {
                s_wawb[op ^ 1u][t] = 0;
                s_rawb[op ^ 1u][t] = 0;
                s_warb[op ^ 1u][t] = 0;
            }
        }
        // the marking is done: empty the hash slots this epoch's writes took
#pragma unroll
        for (uint32_t k = 0; k < kSmallPer; ++k)
            if (wslot[k] != ~0u) {
                s_key[wslot[k]] = 0u;
                s_min[wslot[k]] = ~0u;
            }
        // the epoch's record, stored now by wave 0 (which takes no part in
        // the write-back below) so that its PCIe writes are done by the
        // time done_tail is released
        if (threadIdx.x < 64) {
            if (threadIdx.x == 0)
                done[done_tail & done_mask] = (uint64_t)B | ((uint64_t)nc << 16) | (epoch << 32);
            for (uint32_t t = threadIdx.x; t < B; t += 64)
                done[(done_tail + 1 + t) & done_mask] = s_seq[t] | (dstv[t] == ~0u ? kDoneCommitted : 0ull);
        }
        // read-out (when kept) and write-back; reads see the snapshot, so
        // every read completes before the first write-back store
        const uint32_t per = L * fw;
        const uint32_t total_r = reads ? nc * S * per : 0u;
        const uint32_t total_w = values == LTPG_VALUES_RMW ? nc * S * fw : 0u;
        const uint64_t entry_words = (uint64_t)S * per;
        const auto read_item = [&](uint32_t x, uint64_t &src, uint64_t &dst) -> bool {
            const uint32_t j = dper.div(x), rem = x - j * per, q = dfw.div(rem), w = rem - q * fw;
            const uint32_t jt = dS.div(j), t = listv[jt], sl = j - jt * S;
            const uint32_t i = t * S + sl;
            const Op32 o = loop_decode(s_row[i], s_meta[i], rows32);
            const bool ok = q < o.len;
            src = ok ? ((uint64_t)(o.row + q) * fields + o.field) * fsw + w : 0ull;
            dst = ((done_tail + 1 + t) & done_mask) * entry_words + ((uint64_t)sl * L + q) * fw + w;
            return ok;
        };
        // a committed write adds its delta to every word of its field with
        // an atomic add: several writes of one transaction to one field (and
        // the writes to the hot row, which never conflict) then need no
        // folding, and the sum is the sequential one (modular addition)
        const auto write_item = [&](uint32_t x, uint64_t &off, uint32_t &add) -> bool {
            const uint32_t j = dfw.div(x), w = x - j * fw;
            const uint32_t jt = dS.div(j), t = listv[jt], sl = j - jt * S;
            const uint32_t i = t * S + sl;
            const Op32 o = loop_decode(s_row[i], s_meta[i], rows32);
            const bool wr = o.valid && o.kind == LTPG_KV_WRITE;
            add = (uint32_t)s_seq[t] | 1u;
            off = wr ? ((uint64_t)o.row * fields + o.field) * fsw + w : 0ull;
            return wr;
        };
        // the read-out (kept reads only) in rounds, then a barrier, then the
        // write-back; without kept reads an epoch's writes are one round.
        // (The barrier closes every path through the read-out, so no table
        // load is left pending after it.)
        if (total_r) {
            for (uint32_t b0 = 0; b0 < total_r; b0 += kSmallUnroll * kSmallBlock) {
                uint64_t src[kSmallUnroll], dst[kSmallUnroll];
                bool ok[kSmallUnroll];
                uint32_t v[kSmallUnroll];
#pragma unroll
                for (uint32_t u = 0; u < kSmallUnroll; ++u) {
                    const uint32_t x = b0 + u * kSmallBlock + threadIdx.x;
                    ok[u] = x < total_r && read_item(x, src[u], dst[u]);
                    if (!ok[u]) src[u] = 0ull;
                }
#pragma unroll
                for (uint32_t u = 0; u < kSmallUnroll; ++u)
                    v[u] = __hip_atomic_load(&table[src[u]], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
                for (uint32_t u = 0; u < kSmallUnroll; ++u)
                    if (ok[u]) reads[dst[u]] = v[u];
            }
            // every table load has returned (a load whose value is not kept
            // is otherwise never waited for, and the first later write of
            // its register would wait for every access issued after it,
            // the write-back atomics included), then every read of the
            // snapshot is done before the first write
            __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);
            __syncthreads();
        }
        {
            // waves 1.. issue the write-back atomics and never wait for
            // them inside the loop (no later load result is pending behind
            // them); the next epoch's read-out is ordered after them by its
            // barrier (kept reads), and the launch ends after them
            if (threadIdx.x >= 64)
                for (uint32_t x = threadIdx.x - 64; x < total_w; x += kSmallBlock - 64) {
                    uint64_t off;
                    uint32_t add;
                    if (write_item(x, off, add)) atomicAdd(&table[off], add);
                }
        }
        // committed reads went to host memory from every wave
        if (reads && total_r) __threadfence_system();
        if (threadIdx.x == 64) {
            add_counts(a.ctr, (uint32_t)(epoch % kCounterStripes), LTPG_TYPE_KV, nc, B);
            const uint32_t bad_ops = s_bad;
            s_bad = 0;  // (the next EXECUTE adds to it after the barrier below)
            if (bad_ops) atomicAdd(&a.ctr->range_errors, bad_ops);
        }
        // Kept reads: every wave fenced its stores above, and the barrier
        // orders those fences before the release below.  Without, the record
        // is wave 0's alone and wave 0 publishes it while waves 1.. are still
        // issuing the write-back (nothing after this point reads what they
        // write: the requeue reads this epoch's LDS halves and writes the
        // other ones).
        if (reads) lds_sync();
        stamp(6);
        publish(done_tail + 1 + B);
        done_tail += 1 + B;
        stamp(7);
        // requeue: the aborted requests move to the front, in position order
        // (everything is re-read from LDS: nothing of the phases above stays
        // in registers across the read-out and write-back)
        uint64_t sq[kSmallPer];
        uint32_t ro[kSmallPer], mo[kSmallPer], dst_t[kSmallPer], dst_i[kSmallPer];
        bool ab[kSmallPer], abop[kSmallPer];
#pragma unroll
        for (uint32_t k = 0; k < kSmallPer; ++k) {
            const uint32_t t = k * kSmallBlock + threadIdx.x;
            dst_t[k] = t < B ? dstv[t] : ~0u;
            ab[k] = dst_t[k] != ~0u;
            sq[k] = ab[k] ? s_seq[t] : 0ull;
            const uint32_t i = t;
            const uint32_t ti = i < n ? dS.div(i) : 0u;
            const uint32_t di = i < n ? dstv[ti] : ~0u;
            abop[k] = di != ~0u;
            dst_i[k] = di * S + (i - ti * S);
            ro[k] = abop[k] ? s_row[i] : 0u;
            mo[k] = abop[k] ? s_meta[i] : 0u;
        }
        // everything goes to the other halves, which no wave reads in this
        // epoch: no barrier between the reads above and the stores below
#pragma unroll
        for (uint32_t k = 0; k < kSmallPer; ++k) {
            if (ab[k]) s_seqb[op ^ 1u][dst_t[k]] = sq[k];
            if (abop[k]) {
                s_rowb[op ^ 1u][dst_i[k]] = ro[k];
                s_metab[op ^ 1u][dst_i[k]] = mo[k];
            }
        }
        n_carry = carry_n;
        cap = cap_n;
        ++epoch;
        t_work = now;
        admitted = go;
        if (go) {
            B = B_n;
            n_new = new_n;
            head += new_n;
            now = n_now;
            tail_seen = n_tail;
        }
        lds_sync();
        cp ^= 1u;
        op ^= 1u;
        stamp(8);
        if (prof && threadIdx.x == 0) s_prof[kServeProfParts + 1] += 1;
    }
    // save the carried requests for the next launch (same stream: ordered)
    for (uint32_t i = threadIdx.x; i < n_carry * S; i += kSmallBlock) {
        a.carry_keys[i] = s_rowb[op][i];  // (the packed form; only this kernel reads it back)
        a.carry_meta[i] = s_metab[op][i];
    }
    for (uint32_t t = threadIdx.x; t < n_carry; t += kSmallBlock) a.carry_seq[t] = s_seqb[op][t];
    __syncthreads();
    if (threadIdx.x == 0) {
        if (prof) {
            for (int k = 0; k < kServeProfParts; ++k) ctl->prof[k] += s_prof[k];
            ctl->prof_epochs += s_prof[kServeProfParts + 1];
        }
        ctl->busy_ticks += s_busy;
        sys_store(&ctl->n_carry, n_carry);
        sys_store(&ctl->cap, cap);
        sys_store(&ctl->epochs, epoch);
        sys_store(&ctl->head, head);
        sys_store(&ctl->exit_code, code);
        sys_store(&ctl->running, 0ull);
    }
}

// Latencies of the steps an epoch of the device loop chains (the terms of
// its dependent-chain roofline), in wall-clock ticks per step, measured by
// thread 0 of one 1024-thread workgroup while every lane runs the same chain:
//   [0] an LDS-only workgroup barrier (lds_sync) over 16 waves;
//   [1] a dependent LDS load (each lane chases its own index chain);
//   [2] a dependent LDS atomic with return (a compare-and-swap that never
//       swaps, along the chain);
//   [3] a dependent system-scope load of pinned host memory (a PCIe round
//       trip), thread 0 alone;
//   [4] a publish -- a system-scope release fence, then a relaxed
//       system-scope store to pinned host memory -- back to back, thread 0
//       alone (each fence also waits for the previous store).
// Every index stays inside its array: LDS chain values are masked to 4096,
// host chain values are masked to chain_words (a power of two).
__global__ __launch_bounds__(kSmallBlock) void latency_probe_kernel(uint64_t *host, uint32_t chain_words,
                                                                   unsigned long long *out, uint32_t reps,
                                                                   uint32_t host_reps, uint32_t mask,
                                                                   uint64_t sentinel)
{
    // mask (4095) and sentinel (never reached) come from the host, so the
    // compiler can neither drop the chains nor the waits for their ends
    __shared__ uint32_t s_chain[4096];
    for (uint32_t i = threadIdx.x; i < 4096; i += kSmallBlock) s_chain[i] = (i * 2053u + 1u) & 4095u;
    __syncthreads();
    unsigned long long t0 = 0;
    // [0] barriers
    if (threadIdx.x == 0) t0 = wall_clock64();
    for (uint32_t r = 0; r < reps; ++r) lds_sync();
    if (threadIdx.x == 0) out[0] = wall_clock64() - t0;
    __syncthreads();
    // [1] dependent LDS loads
    uint32_t idx = (threadIdx.x * 4u) & mask;
    if (threadIdx.x == 0) t0 = wall_clock64();
    for (uint32_t r = 0; r < reps; ++r) idx = s_chain[idx] & mask;
    if (idx == (uint32_t)sentinel) out[5] = idx;  // waits for the last load
    if (threadIdx.x == 0) out[1] = wall_clock64() - t0;
    __syncthreads();
    // [2] dependent LDS atomics with return
    idx = (threadIdx.x * 4u) & mask;
    if (threadIdx.x == 0) t0 = wall_clock64();
    // a compare-and-swap whose compare value is never stored: it returns the
    // slot unchanged (an add of 0 would be turned into a plain load)
    for (uint32_t r = 0; r < reps; ++r) idx = atomicCAS(&s_chain[idx], (uint32_t)sentinel, 0u) & mask;
    if (idx == (uint32_t)sentinel) out[5] = idx;
    if (threadIdx.x == 0) out[2] = wall_clock64() - t0;
    __syncthreads();
    if (threadIdx.x == 0) {
        // [3] PCIe round trips
        uint64_t j = 0;
        t0 = wall_clock64();
        for (uint32_t r = 0; r < host_reps; ++r) j = ring_load(&host[j]) & (chain_words - 1);
        if (j == sentinel) out[5] = j;
        out[3] = wall_clock64() - t0;
        // [4] publishes
        t0 = wall_clock64();
        for (uint32_t r = 0; r < host_reps; ++r) {
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "");
            __hip_atomic_store(&host[chain_words], (uint64_t)r, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "");
        out[4] = wall_clock64() - t0;
    }
}

int lanes_for(uint32_t fw)
{
    if (fw > 64) return 0;
    int lp = 1;
    while ((uint32_t)lp < fw) lp <<= 1;
    return lp;
}

inline dim3 grid_for(uint64_t n_threads)
{
    return dim3((unsigned)((n_threads + kBlock - 1) / kBlock));
}

inline dim3 grid_stride(uint64_t n)
{
    uint64_t g = (n + kBlock - 1) / kBlock;
    if (g > 65536) g = 65536;
    if (g == 0) g = 1;
    return dim3((unsigned)g);
}

#define LTPG_LP_SWITCH(lp, CALL) \
    switch (lp) {                \
    case 1: CALL(1); break;      \
    case 2: CALL(2); break;      \
    case 4: CALL(4); break;      \
    case 8: CALL(8); break;      \
    case 16: CALL(16); break;    \
    case 32: CALL(32); break;    \
    case 64: CALL(64); break;    \
    default: CALL(0); break;     \
    }

}  // namespace

hipError_t launch_reset_epoch_counters(DeviceCounters *ctr, hipStream_t s)
{
    hipLaunchKernelGGL(reset_epoch_counters_kernel, dim3(1), dim3(kBlock), 0, s, ctr);
    return hipGetLastError();
}

hipError_t launch_copy_u128(void *dst, const void *src, uint64_t n16, hipStream_t s)
{
    uint64_t g = (n16 + kBlock - 1) / kBlock;
    if (g > 8192) g = 8192;
    if (g == 0) g = 1;
    hipLaunchKernelGGL(copy_u128_kernel, dim3((unsigned)g), dim3(kBlock), 0, s, static_cast<uint4 *>(dst),
                       static_cast<const uint4 *>(src), n16);
    return hipGetLastError();
}

hipError_t launch_fill_set(const FillSet &f, hipStream_t s)
{
    uint64_t most = 1;
    for (uint32_t k = 0; k < f.n; k++) most = std::max(most, f.bytes[k]);
    // Few blocks start sooner, many keep the stores of one block together: 160 MB
    // 26 us with 8192, 28 with 65,536, 1.6 GB 319 and 271.
    const uint64_t cap = most > (1ull << 29) ? 65536 : 8192;
    const uint64_t blocks = std::min<uint64_t>((most + 16 * 256 - 1) / (16 * 256), cap);
    hipLaunchKernelGGL(fill_set_kernel, dim3((unsigned)blocks), dim3(256), 0, s, f);
    return hipGetLastError();
}

hipError_t launch_fill_u64(unsigned long long *p, uint64_t n, unsigned long long v, hipStream_t s)
{
    hipLaunchKernelGGL(fill_u64_kernel, grid_stride(n), dim3(kBlock), 0, s, p, n, v);
    return hipGetLastError();
}

hipError_t launch_copy_u32(uint32_t *dst, const uint32_t *src, uint64_t n, hipStream_t s)
{
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(copy_u32_kernel, grid_stride(n), dim3(kBlock), 0, s, dst, src, n);
    return hipGetLastError();
}

hipError_t launch_readback(uint32_t *dst, const uint32_t *src, uint32_t words, uint32_t *blocks, uint64_t *seq_out,
                           uint64_t seq, hipStream_t s)
{
    hipLaunchKernelGGL(readback_kernel, dim3((words + kReadbackWords - 1) / kReadbackWords), dim3(256), 0, s, dst, src,
                       words, blocks, seq_out, seq);
    return hipGetLastError();
}

hipError_t launch_publish(const PublishSet &p, uint64_t *seq_out, uint64_t seq, hipStream_t s)
{
    hipLaunchKernelGGL(publish_kernel, dim3(1), dim3(kBlock), 0, s, p, seq_out, seq);
    return hipGetLastError();
}

hipError_t launch_archive(const PublishSet &p, unsigned long long *stamp, DeviceCounters *reset, hipStream_t s)
{
    uint32_t most = 1;
    for (int k = 0; k < 5; k++) most = std::max(most, p.n[k]);
    const uint32_t blocks = std::min((most + kBlock - 1) / kBlock, 64u);
    hipLaunchKernelGGL(archive_kernel, dim3(blocks), dim3(kBlock), 0, s, p, stamp, reset);
    return hipGetLastError();
}

hipError_t launch_calibration(unsigned long long *a, uint64_t len, uint64_t n, int atomics,
                              unsigned long long *sink, hipStream_t s)
{
    constexpr uint32_t per = 16;
    const uint64_t threads = (n + per - 1) / per;
    const dim3 grid((unsigned)((threads + kBlock - 1) / kBlock));
    if (atomics)
        hipLaunchKernelGGL(calib_atomic_kernel, grid, dim3(kBlock), 0, s, a, len, n, per, sink);
    else
        hipLaunchKernelGGL(calib_load_kernel, grid, dim3(kBlock), 0, s, a, len, n, per, sink);
    return hipGetLastError();
}

hipError_t launch_gather_calibration(const uint32_t *src, uint64_t slots, uint32_t stride_w, uint32_t fw,
                                     uint32_t *dst, uint64_t n, hipStream_t s)
{
    constexpr uint32_t per = 4;
    const uint64_t waves = (n + 64ull * per - 1) / (64ull * per);
    const dim3 grid((unsigned)((waves * 64 + kBlock - 1) / kBlock));
    hipLaunchKernelGGL(calib_gather_kernel, grid, dim3(kBlock), 0, s, src, slots, stride_w, fw, dst, n, per);
    return hipGetLastError();
}

hipError_t launch_grid_barrier(uint32_t blocks, unsigned int *count, unsigned int *gen, uint32_t reps,
                               uint32_t spin_limit, unsigned int *err, hipStream_t s)
{
    void *args[] = {&count, &gen, &reps, &spin_limit, &err};
    return hipLaunchCooperativeKernel(reinterpret_cast<const void *>(grid_barrier_kernel), dim3(blocks), dim3(kBlock),
                                      args, 0, s);
}

hipError_t launch_boundary(uint32_t blocks, unsigned int *p, hipStream_t s)
{
    hipLaunchKernelGGL(boundary_kernel, dim3(blocks), dim3(kBlock), 0, s, p);
    return hipGetLastError();
}

hipError_t launch_stamp(unsigned long long *out, hipStream_t s)
{
    hipLaunchKernelGGL(stamp_kernel, dim3(1), dim3(1), 0, s, out);
    return hipGetLastError();
}

hipError_t launch_fill_u8(uint8_t *p, uint64_t n, uint8_t v, hipStream_t s)
{
    hipLaunchKernelGGL(fill_u8_kernel, grid_stride(n), dim3(kBlock), 0, s, p, n, v);
    return hipGetLastError();
}

hipError_t launch_kv_fill_reference(const KvState &kv, hipStream_t s)
{
    const uint64_t n = kv.rows * kv.fields * kv.field_stride;
    hipLaunchKernelGGL(kv_fill_reference_kernel, grid_stride(n), dim3(kBlock), 0, s, kv.table, n,
                       kv.fields, kv.field_words, kv.field_stride);
    return hipGetLastError();
}

hipError_t launch_repack(const uint32_t *src, uint32_t *dst, uint64_t n_fields, uint32_t fw,
                         uint32_t fsw, int to_strided, hipStream_t s)
{
    hipLaunchKernelGGL(repack_kernel, grid_stride(n_fields * fw), dim3(kBlock), 0, s, src, dst, n_fields, fw,
                       fsw, to_strided);
    return hipGetLastError();
}

hipError_t launch_kv_transpose(const uint32_t *src, uint32_t *dst, uint64_t rows, uint32_t cols,
                               int to_row_major, hipStream_t s)
{
    hipLaunchKernelGGL(transpose_kernel<uint32_t>, grid_stride(rows * cols), dim3(kBlock), 0, s, src, dst, rows,
                       cols, to_row_major);
    return hipGetLastError();
}

RegLayout reg_layout(const KvState &kv)
{
    RegLayout rl;
    rl.row_mul = kv.split_regs ? 1 : 2;
    rl.w_off = kv.split_regs ? kv.rows : 1;
    return rl;
}

// Default EXECUTE shapes, from a sweep of rows x ops x Zipf x reads; times in
// us, per-transaction registers / per-op registers / binned.
//
// Binned: its cost besides streaming is one short run per tile and bucket, so
// it needs about 1024 ops per bucket.  TIDs in order, Zipf 0.9, 50 % reads:
//   1M rows (256 buckets):    160K ops 23 / 17 / 15, 320K 28 / 27 / 17,
//                             1.3M 76 / 61 / 27, 16M 394 / 295 / 152
//   10M rows (64 to 512 hashed, 1024 from 2^22 ops):
//                             160K ops 21 / 17 / 17, 320K 25 / 27 / 19,
//                             650K 43 / 46 / 24, 4M 191 / 121 / 58,
//                             16M 442 / 374 / 153
//   100M rows (1024, 2048 hashed): 1.3M ops 64 / 64 / 38, 16M 505 / 446 / 217
// (with 90 % reads at Zipf 0.99 the line is crossed at about twice the ops).
// All reads take the bins without their flags: 10M rows, Zipf 0.99, 320K ops 10
// / - / 11, 4M 55 / - / 34, 16M 196 / - / 83.
//
// Whether TIDs are in order, and what is read, the host does not know.  The
// same with TIDs shuffled, per-transaction registers / binned (Zipf 0.99, 50 %
// reads in brackets):
//   50K rows: 320K ops 31 / 19 (39 / 21), 4M 217 / 78 (293 / 77), 16M 389 / 280
//   1M rows:  320K ops 28 / 21 (35 / 18), 4M 206 / 85 (299 / 78), 16M 413 / 345
//   10M rows: 320K ops 26 / 24 (33 / 27), 4M 190 / 105 (280 / 98), 16M 464 / 398
// The registers are the faster ones, and ltpg_kv_set_tuning(0) keeps a context on
// them, where the TIDs are shuffled and nearly all operations write rows of their
// own (10M rows, Zipf 0, 650K ops 33 / 89, 16M on 50K rows 240 / 268), and where
// a few writes meet reads that crowd on few rows (Zipf 0.99, 99 % reads, in order
// 50K rows 1.3M ops 24 / 37, 16M 125 / 177; 10M rows 1.3M 33 / 49, 4M 73 / 75,
// 16M 237 / 168; shuffled 16M 126 / 408 and 238 / 425): there each read has a
// flag byte to store.
// Below 32K rows there are too few buckets to fill the chip (20K rows, 16M ops,
// Zipf 0: 186 / 191 / 212).
bool kv_bin_auto(uint64_t rows, uint64_t ops)
{
    if (rows <= (1ull << 15) || rows > (1ull << 28) || ops >= (1ull << 31)) return false;
    return ops >= (1ull << 18) && ops >= 1024ull * bin_shape(rows, ops).buckets;
}

bool kv_execute_bins(const KvState &kv, const KvBatchDev &b)
{
    const uint64_t ops = (uint64_t)b.n_txns * b.n_slots;
    if (!kv.bin.ent || kv.max_scan > 1 || !(kv.partitioned || (kv.auto_shape && kv_bin_auto(kv.rows, ops))) ||
        ops >= 0xFFFF0000ull)
        return false;
    return bin_fits(kv.bin, bin_shape(kv.rows, ops));
}

namespace {

// Per-op registration where the binned path is not taken: small epochs are a
// chain of dependent misses per transaction otherwise (80K ops on 1M rows 19
// / 10 us, 160K 22 / 16), and the largest ones gain from its row folding
// (100M rows: 4M ops 180 / 143, 16M 504 / 447); in between it loses where
// most rows are distinct (1.3M ops on 10M rows, Zipf 0: 48 / 53).
inline bool kv_per_op_auto(uint64_t ops) { return ops < (1ull << 18) || ops >= (1ull << 21); }

hipError_t launch_kv_bin(const KvState &kv, const KvBatchDev &b, const EpochTag &e, DeviceCounters *ctr,
                         hipStream_t s, bool zero_counts)
{
    const KvBinSource src = {b.keys, b.meta, kv.rows, kv.fields, kv.max_scan, kv.hot_row};
    BinArgs a;
    a.width = b.request_major ? b.n_slots : b.n_txns;
    a.n_ops = b.n_txns * b.n_slots;
    a.rm = b.request_major;
    a.tids = b.tids;
    a.B = b.n_txns;
    a.doomed = kv.doomed;
    a.raw_flag = kv.raw_flag;
    a.war_flag = kv.war_flag;
    return launch_bin(src, a, bin_shape(kv.rows, a.n_ops), kv.bin, e, ctr, zero_counts, kv.clear_flags, true, s);
}

}  // namespace

hipError_t launch_kv_execute(const KvState &kv, const KvBatchDev &b, const EpochTag &e, bool counts,
                             DeviceCounters *ctr, hipStream_t s, bool zero_counts)
{
    // an empty epoch still starts its commit counts at zero
    if (b.n_txns == 0) return zero_counts ? launch_reset_epoch_counters(ctr, s) : hipSuccess;
    const uint64_t ops = (uint64_t)b.n_txns * b.n_slots;
    const dim3 op_grid((unsigned)((ops + kBlock - 1) / kBlock));
    if (!counts && kv_execute_bins(kv, b)) return launch_kv_bin(kv, b, e, ctr, s, zero_counts);
    if (kv.partitioned && !counts && kv.part.ent_me) {
        PartArgs a;
        a.keys = b.keys;
        a.meta = b.meta;
        a.tids = b.tids;
        a.B = b.n_txns;
        a.S = b.n_slots;
        a.rows = kv.rows;
        a.fields = kv.fields;
        a.max_scan = kv.max_scan;
        a.hot = kv.hot_row;
        a.nb = kv.part.n_buckets;
        a.cap_slices = kv.part.cap_slices;
        a.count = kv.part.count;
        a.start = kv.part.start;
        a.cursor = kv.part.cursor;
        a.slices = kv.part.slices;
        a.ent_me = kv.part.ent_me;
        a.ent_key = kv.part.ent_key;
        a.regs = kv.regs;
        a.rl = reg_layout(kv);
        a.tag = e.tag;
        a.epoch = e.epoch;
        a.rm = b.request_major;
        a.doomed = kv.doomed;
        a.raw_flag = kv.raw_flag;
        a.war_flag = kv.war_flag;
        a.ctr = ctr;
        const dim3 chunks((unsigned)((ops + kPartChunk - 1) / kPartChunk));
        // slices: one per non-empty bucket, plus one per kPartSlice operations
        const uint64_t entries = ops * (kv.max_scan > 1 ? kv.max_scan : 1);
        uint64_t slices = a.nb + entries / kPartSlice + 1;
        if (slices > kv.part.cap_slices) slices = kv.part.cap_slices;
        hipLaunchKernelGGL(kv_part_count_kernel, chunks, dim3(kPartBlock), 0, s, a, zero_counts);
        hipLaunchKernelGGL(kv_part_scan_kernel, dim3(1), dim3(kPartBlock), 0, s, a);
        hipLaunchKernelGGL(kv_part_scatter_kernel, chunks, dim3(kPartBlock), 0, s, a);
        hipLaunchKernelGGL(kv_part_process_kernel, dim3((unsigned)slices), dim3(kPartBlock), 0, s, a);
        hipLaunchKernelGGL(kv_part_flags_kernel, dim3((unsigned)slices), dim3(kPartBlock), 0, s, a);
        return hipGetLastError();
    }
    const bool per_op = kv.exec_per_op || (kv.auto_shape && !counts && kv_per_op_auto(ops));
    if (per_op && !counts) {
        if (kv.more_items)
            hipLaunchKernelGGL(kv_execute_dedup_kernel<4>, dim3((unsigned)((ops + 4 * kBlock - 1) / (4 * kBlock))),
                               dim3(kBlock), 0, s, b.keys, b.meta, b.tids, b.n_txns, b.n_slots, kv.rows, kv.fields,
                               kv.regs, reg_layout(kv), kv.hot_row, e.tag, kv.doomed, e.epoch, zero_counts,
                               kv.max_scan, ctr, b.request_major);
        else
            hipLaunchKernelGGL(kv_execute_dedup_kernel<2>, dim3((unsigned)((ops + 2 * kBlock - 1) / (2 * kBlock))),
                               dim3(kBlock), 0, s, b.keys, b.meta, b.tids, b.n_txns, b.n_slots, kv.rows, kv.fields,
                               kv.regs, reg_layout(kv), kv.hot_row, e.tag, kv.doomed, e.epoch, zero_counts,
                               kv.max_scan, ctr, b.request_major);
    } else if (per_op) {
        hipLaunchKernelGGL(kv_execute_ops_kernel, op_grid, dim3(kBlock), 0, s, b.keys, b.meta, b.tids, b.n_txns,
                           b.n_slots, kv.rows, kv.fields, kv.regs, reg_layout(kv), kv.hot_row, e.tag, kv.doomed,
                           e.epoch, counts, zero_counts, kv.max_scan, ctr, b.request_major);
    } else {
        hipLaunchKernelGGL(kv_execute_kernel, grid_for(b.n_txns), dim3(kBlock), 0, s, b.keys, b.meta, b.tids,
                           b.n_txns, b.n_slots, kv.rows, kv.fields, kv.regs, reg_layout(kv), kv.hot_row, e.tag,
                           kv.doomed, e.epoch, counts, zero_counts, kv.max_scan, ctr, b.request_major);
    }
    if (!counts) {
        if (kv.more_items)
            hipLaunchKernelGGL(kv_mark_reads_kernel<2>, dim3((unsigned)((ops + 2 * kBlock - 1) / (2 * kBlock))),
                               dim3(kBlock), 0, s, b.keys, b.meta, b.tids, b.n_txns, b.n_slots, kv.rows, kv.fields,
                               kv.regs, reg_layout(kv), kv.hot_row, e.tag, kv.raw_flag, kv.war_flag, e.epoch,
                               kv.max_scan, b.request_major);
        else
            hipLaunchKernelGGL(kv_mark_reads_kernel<1>, op_grid, dim3(kBlock), 0, s, b.keys, b.meta, b.tids,
                               b.n_txns, b.n_slots, kv.rows, kv.fields, kv.regs, reg_layout(kv), kv.hot_row, e.tag,
                               kv.raw_flag, kv.war_flag, e.epoch, kv.max_scan, b.request_major);
    }
    return hipGetLastError();
}

int group_for(uint32_t S)
{
    int g = 1;
    while ((uint32_t)g < S) g <<= 1;
    return g;
}

#define LTPG_G_SWITCH(g, CALL)   \
    switch (g) {                \
    case 1: CALL(1); break;     \
    case 2: CALL(2); break;     \
    case 4: CALL(4); break;     \
    case 8: CALL(8); break;     \
    case 16: CALL(16); break;   \
    case 32: CALL(32); break;   \
    default: CALL(64); break;   \
    }

// A chunk's committed transactions are shared out over gridDim.y blocks,
// each of which rebuilds the chunk's list (CH flag reads), until the grid
// has about 2048 blocks or every wave of the chunk copies a single round of
// transactions: a small epoch's read-out and write-back then run as many
// short waves instead of a few long ones.
inline dim3 grid_chunks(uint32_t B, uint32_t ch, uint32_t g)
{
    const uint32_t chunks = (B + ch - 1) / ch;
    const uint32_t per_block = (kBlock / 64) * (64 / g);  // transactions per block and round
    const uint32_t max_split = (ch + per_block - 1) / per_block;
    uint32_t split = (2048 + chunks - 1) / chunks;
    if (split > max_split) split = max_split;
    return dim3(chunks, split < 1 ? 1 : split);
}

// The per-lane copy needs fields that start on 16-byte boundaries and fit
// eight 16-byte loads.
static uint32_t lane_copy_ok(const KvState &kv)
{
    return kv.lane_copy && kv.field_stride % 4 == 0 && kv.field_words <= 32 ? 1u : 0u;
}

// The list costs one more kernel, which an even share of the copies makes up
// for in large batches that commit unevenly.  CHECK and WRITEBACK with the list
// and by chunks, uniform rows (Zipf 0.9 in brackets), 100-byte fields: 10,000
// transactions of 10 ops 19 us against 15 (17 / 13), 98,304 61 / 60 (36 / 34),
// 196,608 89 / 100 (61 / 60); 32,768 of 16 22 / 21 (16 / 14), 65,536 23 / 28
// (16 / 15), 262,144 24 / 56 (17 / 17); of 4 ops 262,144 40 / 37 (24 / 20).
constexpr uint64_t kListOps = 1u << 20, kListOpsFewSlots = 1u << 21;
// 8 per CU, what the read-out's registers and LDS allow to be resident.  Of
// WRITEBACK 7 are (with up to 8 slots or more than 16; 1792 blocks take the same
// time), but with 9 to 16 slots the lanes' fields leave LDS for 6, and the last
// 512 blocks would be a second round: 2^20 transactions of 16 ops at Zipf 0.6
// 28.4 us with 2048, 26.2 with 1536 (1792 cost 9 us more at 1.01M commits).
constexpr uint32_t kListBlocks = 2048, kListBlocks16 = 1536;

bool kv_check_lists(const KvState &kv, const KvBatchDev &b)
{
    return kv.commit_list && (uint64_t)b.n_txns * b.n_slots >= (b.n_slots >= 8 ? kListOps : kListOpsFewSlots) &&
           !kv.small_chunks && !kv.lane_copy;
}

// Read values and written fields are moved whole, padding included: fields of
// 64 bytes and more then leave as whole 64-byte segments of memory, where a
// partly written segment costs a read at the memory side (8.1M reads of 100
// bytes with every seventh slot left out: 597 us packed, 432 us for 7.7M
// fields of 128 bytes).  Nothing reads the padding.  (Read values of a context
// short of memory are packed, read_stride = field_words.)
hipError_t launch_kv_check(const KvState &kv, const KvBatchDev &b, const EpochTag &e, bool counts,
                           DeviceCounters *ctr, hipStream_t s)
{
    if (b.n_txns == 0) return hipSuccess;
    if (counts) {
        hipLaunchKernelGGL(kv_check_counting_kernel, grid_for(b.n_txns), dim3(kBlock), 0, s, b.keys,
                           b.meta, b.tids, b.n_txns, b.n_slots, kv.rows, kv.fields, kv.regs, reg_layout(kv),
                           kv.hot_row, e.tag, kv.bitmap, kv.conflicts, kv.max_scan, ctr, b.request_major);
        return hipGetLastError();
    }
    if (kv_check_lists(kv, b)) {
        hipLaunchKernelGGL(kv_commit_list_kernel,
                           dim3((b.n_txns + kListPer * kListBlock - 1) / (kListPer * kListBlock)), dim3(kListBlock), 0,
                           s, b.n_txns, kv.doomed, kv.raw_flag, kv.war_flag, e.epoch, kv.bitmap, kv.commit_list, ctr);
        const uint64_t units = ((uint64_t)b.n_txns + 63) / 64 * b.n_slots, per = kBlock / 64;
        const uint64_t blocks = std::min<uint64_t>(kListBlocks, (units + per - 1) / per);
        hipLaunchKernelGGL(kv_readout_list_kernel, dim3((unsigned)blocks), dim3(kBlock), 0, s, b.keys, b.meta, b.n_txns,
                           b.n_slots, kv.rows, kv.fields, kv.read_stride, kv.field_stride, kv.table, kv.read_values,
                           kv.commit_list, ctr, kv.max_scan, kv.read_slot, b.request_major);
        return hipGetLastError();
    }
#define CALL1(GV, CHV)                                                                               \
    hipLaunchKernelGGL((kv_check_fast_kernel<GV, CHV>), grid_chunks(b.n_txns, CHV, GV), dim3(kBlock), 0, s, b.keys, \
                       b.meta, b.n_txns, b.n_slots, kv.rows, kv.fields, kv.read_stride, kv.field_stride,    \
                       kv.doomed, kv.raw_flag, kv.war_flag, e.epoch, kv.table, kv.read_values, kv.bitmap,  \
                       kv.max_scan, kv.read_slot, lane_copy_ok(kv), ctr, b.request_major)
#define CALL(GV)                    \
    if (kv.small_chunks)            \
        CALL1(GV, 64);              \
    else                            \
        CALL1(GV, kChunk)
    LTPG_G_SWITCH(group_for(b.n_slots), CALL)
#undef CALL
#undef CALL1
    return hipGetLastError();
}

hipError_t launch_kv_readout(const KvState &kv, const KvBatchDev &b, hipStream_t s)
{
    if (b.n_txns == 0) return hipSuccess;
    const int lp = lanes_for(kv.read_stride);
#define CALL(LPV)                                                                          \
    hipLaunchKernelGGL(kv_readout_kernel<LPV>, grid_for(b.n_txns), dim3(kBlock), 0, s,    \
                       b.keys, b.meta, b.n_txns, b.n_slots, kv.rows, kv.fields,           \
                       kv.read_stride, kv.field_stride, kv.table, kv.bitmap, kv.read_values, kv.max_scan, \
                       kv.read_slot, b.request_major)
    LTPG_LP_SWITCH(lp, CALL)
#undef CALL
    return hipGetLastError();
}

hipError_t launch_kv_writeback(const KvState &kv, const KvBatchDev &b, uint32_t values, DeviceCounters *ctr,
                               hipStream_t s, const EpochEnd &end)
{
    if (b.n_txns == 0) return hipSuccess;
    const WriteArgs a = {b.keys,          b.meta,          b.tids,   b.n_txns,   b.n_slots, kv.rows,
                         kv.fields,       kv.field_stride, kv.field_stride, kv.table,   values,    kv.hot_row,
                         lane_copy_ok(kv), b.request_major, end};
    const int g = group_for(b.n_slots);
    if (kv.list_valid && kv_check_lists(kv, b)) {
        const uint64_t per = (kBlock / 64) * (64 / g);  // transactions per block and round
        const uint32_t most = g == 16 ? kListBlocks16 : kListBlocks;
        const dim3 grid((unsigned)std::min<uint64_t>(most, (b.n_txns + per - 1) / per));
        const bool slots = !a.rm && kv.rows * kv.fields <= 1ull << 32;  // a field's index fits 32 bits
#define CALL(GV) \
    hipLaunchKernelGGL(kv_writeback_list_kernel<GV>, grid, dim3(kBlock), 0, s, a, kv.commit_list, ctr, slots)
        LTPG_G_SWITCH(g, CALL)
#undef CALL
    } else {
#define CALL1(GV, CHV)                                                                                      \
    hipLaunchKernelGGL((kv_writeback_kernel<GV, CHV>), grid_chunks(b.n_txns, CHV, GV), dim3(kBlock), 0, s, a, kv.bitmap)
#define CALL(GV)         \
    if (kv.small_chunks) \
        CALL1(GV, 64);   \
    else                 \
        CALL1(GV, kChunk)
        LTPG_G_SWITCH(g, CALL)
#undef CALL
#undef CALL1
    }
    if (kv.hot_row != LTPG_NO_HOT_ROW && values == LTPG_VALUES_RMW) {
        hipLaunchKernelGGL(kv_hot_sum_kernel, grid_for(b.n_txns), dim3(kBlock), 0, s, b.keys, b.meta, b.tids,
                           b.n_txns, b.n_slots, kv.rows, kv.fields, kv.hot_row, kv.bitmap, kv.hot_acc,
                           b.request_major);
        hipLaunchKernelGGL(kv_hot_apply_kernel, grid_for(kv.fields), dim3(kBlock), 0, s, kv.table, kv.hot_row,
                           kv.fields, kv.field_words, kv.field_stride, kv.hot_acc);
    }
    return hipGetLastError();
}

bool kv_small_epoch_ok(const KvState &kv, const KvBatchDev &b)
{
    return b.n_txns > 0 && b.n_slots > 0 && (uint64_t)b.n_txns * b.n_slots <= kSmallOps &&
           (kv.hot_row == LTPG_NO_HOT_ROW || kv.fields <= kSmallHotFields) && kv.rows < 0xFFFFFFFFull;
}

// Words a small epoch copies at most.
uint64_t kv_small_words(const KvState &kv, const KvBatchDev &b)
{
    return (uint64_t)b.n_txns * b.n_slots * kv.read_slot * kv.field_words;
}

// The single-workgroup epoch by default: one workgroup copies fields at a
// fraction of the chip's rate, so it is taken while what it saves in launches
// is more (one kernel against four, back to back, uniform rows: 64 ops on
// 4-byte fields 7 us against 17, 1,024 12 / 18, of 64 slots each 2,048 26 / 22;
// 100-byte fields 256 ops 12 / 17, 512 15 / 18, 1,024 20 / 19; 1 KB fields 64
// ops 15 / 22, 256 30 / 25).
bool kv_small_auto(const KvState &kv, const KvBatchDev &b)
{
    return kv.auto_shape && kv_small_epoch_ok(kv, b) && (uint64_t)b.n_txns * b.n_slots <= kSmallOps / 2 &&
           kv_small_words(kv, b) <= 1u << 14;
}

hipError_t launch_kv_small_epoch(const KvState &kv, const KvBatchDev &b, uint32_t values, DeviceCounters *ctr,
                                 uint64_t *host_bits, uint64_t *seq_out, uint64_t seq, hipStream_t s,
                                 uint32_t *result)
{
    if (!kv_small_epoch_ok(kv, b)) return hipErrorInvalidValue;
    hipLaunchKernelGGL(kv_small_epoch_kernel, dim3(1), dim3(kSmallBlock), 0, s, b.keys, b.meta, b.tids, b.n_txns,
                       b.n_slots, b.request_major, kv.rows, kv.fields, kv.field_words, kv.field_stride, kv.read_stride,
                       kv.max_scan, kv.read_slot, values, kv.hot_row, kv.table, kv.read_values, kv.bitmap, host_bits, seq_out, seq,
                       result, ctr);
    return hipGetLastError();
}

hipError_t launch_kv_gather_rows(const KvState &kv, const uint64_t *idx, uint64_t n, uint32_t *out, hipStream_t s)
{
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(kv_gather_rows_kernel, grid_stride(n * kv.fields * kv.field_words), dim3(kBlock), 0, s,
                       kv.table, idx, n, kv.fields, kv.field_words, kv.field_stride, out);
    return hipGetLastError();
}

bool kv_serve_loop_ok(const KvState &kv, uint32_t S)
{
    return S >= 1 && S <= 64 && S <= kSmallOps && (kv.hot_row == LTPG_NO_HOT_ROW || kv.fields <= kSmallHotFields) &&
           kv.rows < 0xFFFFFFFFull;
}

hipError_t launch_latency_probe(uint64_t *host, uint32_t chain_words, unsigned long long *out, uint32_t reps,
                                uint32_t host_reps, hipStream_t s)
{
    if (chain_words == 0 || (chain_words & (chain_words - 1))) return hipErrorInvalidValue;
    hipLaunchKernelGGL(latency_probe_kernel, dim3(1), dim3(kSmallBlock), 0, s, host, chain_words, out, reps, host_reps,
                       4095u, ~0ull);
    return hipGetLastError();
}

hipError_t launch_kv_serve_loop(const ServeLoopArgs &a, hipStream_t s)
{
    if (a.S < 1 || a.S > 64 || (uint64_t)a.cap_max * a.S > kSmallOps || a.cap_max == 0 || a.floor == 0)
        return hipErrorInvalidValue;
    hipLaunchKernelGGL(kv_serve_loop_kernel, dim3(1), dim3(kSmallBlock), 0, s, a);
    return hipGetLastError();
}

}  // namespace ltpg
