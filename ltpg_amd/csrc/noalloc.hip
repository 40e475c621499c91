// noalloc.hip - a key-value epoch that allocates nothing.
//
// ltpg_kv_epoch_noalloc runs the same EXECUTE / CHECK / WRITEBACK kernels as
// ltpg_epoch_run on a key-value context, but over a table and batch the
// caller owns, with every per-row register, per-transaction flag, binned
// operation and counter in `scratch`: a file-scope device array of fixed size that each GPU holds
// from module load to process end.  For callers that cannot call hipMalloc
// (code under graph capture, tight serving loops).
//
// Host code never passes `scratch` itself to a kernel (in host code the name
// is a host-side stand-in, not a device address): the first call on each
// device looks its address up with hipGetSymbolAddress, with that device
// current, and every later call on the device uses that address.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>
#include <string>
#include <vector>

#include "ltpg_internal.h"

namespace ltpg {
namespace {

constexpr uint64_t kRegsBytes = 2ull * LTPG_NOALLOC_MAX_ROWS * 8;  // interleaved R / W per row
constexpr uint64_t kFlagsAt = kRegsBytes;                         // doomed, raw, war: one byte per txn each
constexpr uint64_t kCountersAt = kFlagsAt + 3ull * LTPG_NOALLOC_MAX_TXNS;
constexpr uint64_t kListAt = kCountersAt + (sizeof(DeviceCounters) + 255) / 256 * 256;
// Binned EXECUTE of up to kBinOps op slots: at most 1024 buckets (2^20 rows)
// and one tile per 2^kBinSlotBits slots (larger batches use the registers).
constexpr uint64_t kBinOps = 1ull << 24;
constexpr uint64_t kBinEnts = kBinOps + (1ull << kBinSlotBits);
constexpr uint64_t kBinOffs = (kBinOps >> kBinSlotBits) * 1025 + 1025;
constexpr uint64_t kMarksAt = kListAt + 4ull * LTPG_NOALLOC_MAX_TXNS;
constexpr uint64_t kEntsAt = kMarksAt + (4 * kBinMarks + 255) / 256 * 256;
constexpr uint64_t kOffsAt = kEntsAt + 4 * kBinEnts;
constexpr uint64_t kScratchBytes = kOffsAt + (4 * kBinOffs + 255) / 256 * 256;

static __device__ __align__(256) uint8_t scratch[kScratchBytes];

// The last call's contents are still there: registers back to "no
// registrant", the batch's flags and the counters to zero.
__global__ void noalloc_init_kernel(unsigned long long *regs, uint64_t n_regs, uint8_t *flags, uint32_t B,
                                    DeviceCounters *ctr)
{
    const uint64_t first = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x, step = (uint64_t)gridDim.x * blockDim.x;
    ulonglong2 *r2 = reinterpret_cast<ulonglong2 *>(regs);
    for (uint64_t i = first; i < n_regs / 2; i += step) r2[i] = make_ulonglong2(~0ull, ~0ull);
    for (uint64_t i = first; i < B; i += step)
        flags[i] = flags[LTPG_NOALLOC_MAX_TXNS + i] = flags[2ull * LTPG_NOALLOC_MAX_TXNS + i] = 0;
    uint32_t *c = reinterpret_cast<uint32_t *>(ctr);
    for (uint64_t i = first; i < sizeof(DeviceCounters) / 4; i += step) c[i] = 0;
}

// The result of an empty epoch.
__global__ void noalloc_empty_kernel(uint32_t *result) { result[threadIdx.x] = 0; }

// scratch's device address, per device (looked up once each)
std::mutex g_mu;
std::vector<uint8_t *> g_scratch;

int scratch_of(int device, uint8_t **out)
{
    std::lock_guard<std::mutex> lk(g_mu);
    if ((size_t)device >= g_scratch.size()) g_scratch.resize(device + 1, nullptr);
    if (!g_scratch[device]) {
        void *p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            LTPG_FAIL(LTPG_ERR_DEVICE, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
        g_scratch[device] = static_cast<uint8_t *>(p);
    }
    *out = g_scratch[device];
    return LTPG_OK;
}

// Words of fields that one workgroup may copy before the other path's six
// kernels are faster (uniform rows, back to back: 1,024 ops on 100-byte fields
// 18 us against 27, 2,048 34 / 27; on 400-byte fields 512 ops 28 / 30, 1,024
// 46 / 30; on 1 KB fields 256 ops 29 / 35, 512 48 / 34).
constexpr uint64_t kAloneWords = 3u << 14;

}  // namespace
}  // namespace ltpg

using namespace ltpg;

extern "C" int ltpg_kv_epoch_noalloc(uint32_t *table, uint64_t rows, uint32_t fields, uint32_t field_bytes,
                                     const ltpg_kv_batch *batch, uint32_t values, uint64_t *bitmap,
                                     uint32_t *read_values, uint32_t *result, void *hip_stream)
{
    if (!table || !batch) LTPG_FAIL(LTPG_ERR_INVALID, "null table or batch");
    if (rows == 0 || rows > LTPG_NOALLOC_MAX_ROWS)
        LTPG_FAIL(LTPG_ERR_INVALID, "rows must be in [1, LTPG_NOALLOC_MAX_ROWS]");
    if (fields == 0 || field_bytes == 0 || field_bytes % 4 || field_bytes > 1024)
        LTPG_FAIL(LTPG_ERR_INVALID, "fields >= 1 and field_bytes a multiple of 4 in [4, 1024]");
    if (values != LTPG_VALUES_COPYBACK && values != LTPG_VALUES_RMW) LTPG_FAIL(LTPG_ERR_INVALID, "unknown values");
    const uint32_t B = batch->n_txns, S = batch->n_slots;
    if (B > LTPG_NOALLOC_MAX_TXNS) LTPG_FAIL(LTPG_ERR_INVALID, "n_txns exceeds LTPG_NOALLOC_MAX_TXNS");
    if (B && (S == 0 || S > 64)) LTPG_FAIL(LTPG_ERR_INVALID, "n_slots must be in [1, 64]");
    if (B && (!batch->keys || !batch->meta || !batch->tids || !bitmap || !read_values))
        LTPG_FAIL(LTPG_ERR_INVALID, "null batch array, bitmap or read values");
    int device = 0;
    LTPG_HIP_TRY(hipGetDevice(&device));
    uint8_t *p = nullptr;
    int rc = scratch_of(device, &p);
    if (rc) return rc;
    hipStream_t s = static_cast<hipStream_t>(hip_stream);
    KvState kv;
    kv.rows = rows;
    kv.fields = fields;
    kv.field_words = field_bytes / 4;
    kv.field_stride = kv.read_stride = kv.field_words;  // the caller's table and read values are packed
    kv.max_slots = S;
    kv.table = table;
    kv.regs = reinterpret_cast<unsigned long long *>(p);
    kv.doomed = p + kFlagsAt;
    kv.raw_flag = kv.doomed + LTPG_NOALLOC_MAX_TXNS;
    kv.war_flag = kv.raw_flag + LTPG_NOALLOC_MAX_TXNS;
    kv.read_values = read_values;
    kv.bitmap = bitmap;
    DeviceCounters *ctr = reinterpret_cast<DeviceCounters *>(p + kCountersAt);
    KvBatchDev b;
    b.n_txns = B;
    b.n_slots = S;
    b.keys = batch->keys;
    b.meta = batch->meta;
    b.tids = batch->tids;
    uint32_t *marks = reinterpret_cast<uint32_t *>(p + kMarksAt);
    if (kv_small_epoch_ok(kv, b) && kv_small_words(kv, b) <= kAloneWords) {
        // one kernel; the registers and flags stay in its LDS (64 x 4 ops: ten
        // launches 36 us, this one 8 us, most of it the launch)
        uint32_t *res = result ? result : reinterpret_cast<uint32_t *>(ctr->pad0);
        LTPG_HIP_TRY(launch_kv_small_epoch(kv, b, values, ctr, nullptr, nullptr, 0, s, res));
        return LTPG_OK;
    }
    if (B) {
        // kernels only, so that a caller may capture the call into a graph
        kv.commit_list = reinterpret_cast<uint32_t *>(p + kListAt);
        kv.bin.ent = reinterpret_cast<uint32_t *>(p + kEntsAt);
        kv.bin.cap_ent = kBinEnts;
        kv.bin.off = reinterpret_cast<uint32_t *>(p + kOffsAt);
        kv.bin.cap_off = kBinOffs;
        kv.bin.marks = marks;
        // binning needs no registers, whose refill costs 16 bytes per row:
        // taken wherever there are rows enough for its buckets (1M rows: 80K
        // ops take 13 us binned, 9 on the registers and 9 for their refill;
        // 65,536 x 10 ops, whole call: 81 -> 33 us)
        kv.partitioned = rows > (1ull << 15);
        kv.clear_flags = true;
        if (!kv_execute_bins(kv, b)) {
            const uint64_t n = std::max<uint64_t>(rows, B / 4);
            hipLaunchKernelGGL(noalloc_init_kernel, dim3((unsigned)std::min<uint64_t>(4096, (n + 255) / 256)), dim3(256),
                               0, s, kv.regs, 2 * rows, kv.doomed, B, ctr);
            LTPG_HIP_TRY(hipGetLastError());
        }
        EpochTag e;
        e.epoch = 1;
        e.tag = 254;
        LTPG_HIP_TRY(launch_kv_execute(kv, b, e, false, ctr, s));
        LTPG_HIP_TRY(launch_kv_check(kv, b, e, false, ctr, s));
        kv.list_valid = true;  // of the CHECK above
        EpochEnd end;
        end.ctr = ctr;
        end.marks = marks;
        end.result = result;
        LTPG_HIP_TRY(launch_kv_writeback(kv, b, values, ctr, s, end));
    } else if (result) {
        hipLaunchKernelGGL(noalloc_empty_kernel, dim3(1), dim3(2), 0, s, result);
        LTPG_HIP_TRY(hipGetLastError());
    }
    return LTPG_OK;
}
