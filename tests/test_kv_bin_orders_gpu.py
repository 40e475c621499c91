"""Binned EXECUTE of batches that are not in TID order, or whose reads crowd on
a few rows: against the oracle where its buckets change their ways (hot buckets
shared by many blocks, TIDs compared in the tiles and in 64-bit hash tables of
one or several shares, ties, no write at all), and in time against the
registers."""
import ctypes
import time

import numpy as np
import pytest

import ltpg_amd as L
from oracle import oracle

pytestmark = pytest.mark.gpu


def batch(rows, B, S, hot_rows, hot_share, writes, seed):
    """`hot_share` of the operations on the first `hot_rows` rows, the others
    anywhere; a share of `writes` of all operations, or that many."""
    rng = np.random.default_rng(seed)
    n = B * S
    keys = rng.integers(0, rows, n).astype(np.uint64)
    pick = rng.random(n) < hot_share
    keys[pick] = rng.integers(0, hot_rows, int(pick.sum()))
    meta = np.full(n, L.kv_meta(L.KV_READ, 0), np.uint32)
    if isinstance(writes, int):
        w = rng.choice(n, writes, replace=False)
        keys[w] = rng.integers(0, hot_rows, writes)
    else:
        w = rng.random(n) < writes
    meta[w] = L.kv_meta(L.KV_WRITE, 0)
    return keys, meta


def order(kind, B, seed):
    t = np.arange(B, dtype=np.uint32) * 3 + 5
    if kind == "shuffled":
        return np.random.default_rng(seed).permutation(t).astype(np.uint32)
    if kind == "ties":  # two TIDs in turn
        return (np.arange(B) % 2 == 0).astype(np.uint32)
    return t


@pytest.mark.parametrize("rows,B,S,hot_rows,hot_share,writes", [
    (300_000, 65_536, 19, 3, 0.6, 0.001),    # hot buckets, tiles of 4096, few writers
    (300_000, 65_536, 19, 3, 0.6, 1),        # one write in all
    (300_000, 65_536, 19, 3, 0.6, 0),        # none
    (9_000_000, 70_001, 16, 2, 0.5, 0.002),  # hot hashed buckets
    (300_000, 300_001, 15, 2, 0.5, 0.002),   # tiles of 16384, a ragged last one
    (300_000, 65_536, 19, 2, 0.7, 1.0),      # writers only
    (9_000_000, 40_000, 16, 1, 0.0, 1.0),    # hashed, one share of distinct writes
    (9_000_000, 81_920, 8, 1, 0.0, 0.97),    # as many writes as the 64-bit table has slots
    (120_000_000, 1_000_003, 16, 1, 0.0, 1.0),  # two shares; 2048 buckets, tiles of 16384
    (400_000, 1_048_577, 17, 2, 0.3, 0.01),  # more than 1024 tiles, hot
    (60_000_000, 1_048_577, 17, 2, 0.2, 0.5),  # the same, hashed
], ids=lambda v: str(v))
@pytest.mark.parametrize("tids", ["ordered", "shuffled", "ties"])
def test_orders_and_crowds_match_oracle(gpu, rows, B, S, hot_rows, hot_share, writes, tids):
    keys, meta = batch(rows, B, S, hot_rows, hot_share, writes, B + S)
    t = order(tids, B, S)
    table = np.zeros(rows, np.uint32)
    ora = oracle.kv_epoch(table, rows, 1, 1, keys, meta, t, S, values=L.VALUES_COPYBACK, want_reads=False, inplace=True)
    with L.Context(workload=L.WORKLOAD_KV, kv_rows=rows, kv_fields=1, kv_field_bytes=4, max_txns=B,
                   kv_max_slots=S) as ctx:
        for request_major in (False, True):
            k, m = keys, meta
            if request_major:
                k, m = (np.ascontiguousarray(a.reshape(S, B).T).reshape(-1) for a in (keys, meta))
            ctx.kv_submit(k, m, t, S, request_major=request_major)
            ctx.epoch_run(L.PHASE_EXECUTE | L.PHASE_CHECK)
            ctx.sync()
            np.testing.assert_array_equal(ctx.commit_bitmap(), ora.bitmap)


def test_one_call_after_another_on_the_library_scratch(gpu):
    """The allocation-free epoch keeps nothing of the call before: whether TIDs
    were in order, a row was written or a bucket was hot."""
    rows, B, S = 400_000, 40_000, 16
    hip = ctypes.CDLL("libamdhip64.so")
    with L.Context(workload=L.WORKLOAD_KV, kv_rows=64, kv_fields=1, max_txns=64, kv_max_slots=1) as ctx:
        table, bits, reads = (L.DeviceBuffer(ctx, n) for n in (4 * rows, (B + 63) // 64 * 8, 4 * B * S))
        table.upload(np.zeros(rows, np.uint32))
        calls = [(0.0, 0.5, "ordered"), (0.7, 0.002, "ordered"), (0.0, 0, "ordered"), (0.7, 0.002, "shuffled"),
                 (0.7, 0, "shuffled"), (0.0, 0.5, "ties"), (0.0, 0.5, "ordered"), (0.7, 1.0, "ties"),
                 (0.0, 1, "ordered")]
        for seed, (share, writes, tids) in enumerate(calls):
            keys, meta = batch(rows, B, S, 2, share, writes, seed)
            t = order(tids, B, seed)
            dev = L.DeviceKvBatch(ctx, keys, meta, t, S)
            struct = dev.struct()
            rc = L.lib.ltpg_kv_epoch_noalloc(ctypes.c_void_p(table.ptr), rows, 1, 4, ctypes.byref(struct),
                                             L.VALUES_COPYBACK, ctypes.c_void_p(bits.ptr), ctypes.c_void_p(reads.ptr),
                                             None, None)
            assert rc == L.OK and hip.hipDeviceSynchronize() == 0
            got = np.empty((B + 63) // 64, np.uint64)
            bits.download(got)
            ora = oracle.kv_epoch(np.zeros(rows, np.uint32), rows, 1, 1, keys, meta, t, S, values=L.VALUES_COPYBACK,
                                  want_reads=False, inplace=True)
            np.testing.assert_array_equal(got, ora.bitmap, err_msg=str((share, writes, tids)))
            dev.free()
        for b in (table, bits, reads):
            b.free()


def execute_us(ctx, dev, n=20):
    for _ in range(3):
        ctx.kv_submit_device(dev)
        ctx.epoch_run(L.PHASE_EXECUTE)
    best = 1e9
    for _ in range(3):
        ctx.sync()
        t = time.perf_counter()
        for _ in range(n):
            ctx.kv_submit_device(dev)
            ctx.epoch_run(L.PHASE_EXECUTE)
        ctx.sync()
        best = min(best, (time.perf_counter() - t) / n * 1e6)
    return best


@pytest.mark.parametrize("rows,theta,read_pct,shuffled", [
    (50_000, 0.99, 90, True), (1_000_000, 0.99, 50, True), (10_000_000, 0.99, 50, True), (10_000_000, 0.99, 90, True),
    (50_000, 0.99, 100, False), (1_000_000, 0.99, 100, True), (10_000_000, 0.99, 100, False),
])
def test_default_shape_keeps_up_with_the_registers(gpu, rows, theta, read_pct, shuffled):
    """EXECUTE of 2^18 x 16 operations by default takes no longer than on the
    registers with one lane per transaction, half as long again allowed for
    noise (it was 4 to 10 times as long)."""
    B, S = 1 << 18, 16
    k, m, t = L.kv_generate(seed=3, rows=rows, fields=1, n_txns=B, n_slots=S, theta=theta, read_pct=read_pct,
                            distinct_keys=False)
    if shuffled:
        t = np.random.default_rng(1).permutation(t).astype(np.uint32)
    with L.Context(workload=L.WORKLOAD_KV, kv_rows=rows, kv_fields=1, kv_field_bytes=4, max_txns=B,
                   kv_max_slots=S) as ctx:
        dev = L.DeviceKvBatch(ctx, k, m, t, S)
        default = execute_us(ctx, dev)
        ctx.kv_set_tuning(0)
        registers = execute_us(ctx, dev)
        dev.free()
    print(f"default {default:.0f} us, registers {registers:.0f} us")
    assert default < 1.5 * registers
