"""Host batches and results on both sides of the sizes where their transport
changes: batches that fit the pinned part of a slot and ones that do not,
mixed, on an idle and on a busy stream, with the caller's buffers overwritten
after each submit; results read back through pinned memory and directly; and
a run's archive in pinned and in device memory."""
import numpy as np
import pytest

import ltpg_amd as L
from oracle import oracle
from tests import kvcases as kc

pytestmark = pytest.mark.gpu

STAGE = 2 << 20  # bytes of a slot's pinned part


def committed(bits, n):
    return np.unpackbits(bits.view(np.uint8), count=n, bitorder="little").astype(bool)


@pytest.mark.parametrize("idle", [True, False], ids=["idle", "busy"])
def test_host_batches_of_mixed_sizes_match_oracle(gpu, idle):
    rows, fields, fw, S = 50_000, 3, 1, 7
    edge = (STAGE - 600) // (S * 12 + 4)  # the most transactions that fit the pinned part, or one less
    sizes = [1, edge, edge + 12, 40_000, 63, 30_000, edge - 1, 2]
    with L.Context(workload=L.WORKLOAD_KV, kv_rows=rows, kv_fields=fields, kv_field_bytes=4 * fw,
                   max_txns=max(sizes), kv_max_slots=S) as ctx:
        table = kc.initial_table(rows, fields, fw)
        ctx.kv_table_load(table)
        for i, B in enumerate(sizes):
            k, m, t = L.kv_generate(seed=i, rows=rows, fields=fields, n_txns=B, n_slots=S, min_ops=1, max_ops=S,
                                    theta=0.9)
            host = k.copy(), m.copy(), t.copy()
            ctx.kv_submit(*host, S)
            for a in host:
                a[:] = 0
            ctx.epoch_run()
            ora = oracle.kv_epoch(table, rows, fields, fw, k, m, t, S, inplace=True)
            if idle:
                np.testing.assert_array_equal(ctx.commit_bitmap(), ora.bitmap)
                assert ctx.commit_count() == ora.commit_count
                read = ((m & 3) == L.KV_READ) & np.tile(committed(ora.bitmap, B), S)
                np.testing.assert_array_equal(ctx.kv_read_values().reshape(-1)[read], ora.read_values.reshape(-1)[read])
        ctx.sync()
        np.testing.assert_array_equal(ctx.kv_table_read(), table)


@pytest.mark.parametrize("n", [1, 31, 2047, 2048, 65_535, 65_537])
def test_counters_read_back_at_the_edges(gpu, n):
    # 65,536 counters are the most that go through pinned memory
    with L.Context(workload=L.WORKLOAD_KV, kv_rows=500, kv_fields=1, kv_field_bytes=4, max_txns=n, kv_max_slots=2,
                   flags=L.FLAG_CONFLICT_COUNTS) as ctx:
        table = kc.initial_table(500, 1, 1)
        ctx.kv_table_load(table)
        for seed in (1, 2):
            k, m, t = L.kv_generate(seed=seed, rows=500, fields=1, n_txns=n, n_slots=2, min_ops=1, max_ops=2, theta=0.5)
            ctx.kv_submit(k, m, t, 2)
            ctx.epoch_run()
            ora = oracle.kv_epoch(table, 500, 1, 1, k, m, t, 2, inplace=True)
            np.testing.assert_array_equal(ctx.conflict_counters(), ora.conflicts)
            np.testing.assert_array_equal(ctx.commit_bitmap(), ora.bitmap)


@pytest.mark.parametrize("n_no,n_pay", [(1, 0), (0, 3), (700, 801), (20_000, 4000), (40, 50_000)])
def test_order_entry_host_batches_match_device_batches(gpu, n_no, n_pay):
    W, n = 2, n_no + n_pay + 90
    got = []
    for mem in (L.MEM_HOST, L.MEM_DEVICE):
        with L.Context(workload=L.WORKLOAD_TPCC, tpcc_warehouses=W, max_txns=n) as ctx:
            ctx.tpcc_populate(3)
            gen = L.TpccGenerator(warehouses=W, seed=9)
            for e in range(3):
                b = gen.next(3 * max(n_no, n_pay) + 50, tid_base=e << 20)  # about half of each type
                assert b.n_no >= n_no and b.n_pay >= n_pay
                b.n_no, b.n_pay = n_no, n_pay
                ro, dl = L.readonly_batch(b, W, 40, 40, 5), L.delivery_batch(b, W, 10, 5)
                bufs = []
                if mem == L.MEM_DEVICE:
                    b, bufs = L.upload_tpcc_batch(ctx, b)
                    ro, more = L.upload_readonly_batch(ctx, ro)
                    dl, more2 = L.upload_delivery_batch(ctx, dl)
                    bufs = bufs + more + more2
                ctx.tpcc_submit(b, mem)
                ctx.tpcc_submit_readonly(ro, mem)
                ctx.tpcc_submit_delivery(dl, mem)
                ctx.epoch_run()
                for ty in (L.TYPE_NEWORDER, L.TYPE_PAYMENT, L.TYPE_ORDERSTATUS, L.TYPE_STOCKLEVEL, L.TYPE_DELIVERY):
                    got.append(ctx.tpcc_bitmap(ty))
                if n_pay:  # only committed transactions' reads are written
                    reads = ctx.tpcc_read_values(L.TYPE_PAYMENT).reshape(-1, n_pay)
                    got.append(reads * committed(ctx.tpcc_bitmap(L.TYPE_PAYMENT), n_pay))
                for x in bufs:
                    x.free()
    half = len(got) // 2
    for a, b in zip(got[:half], got[half:]):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("batches,B", [(3, 1000), (33, 1 << 20)])
def test_archive_of_a_run_matches_oracle(gpu, batches, B):
    # 33 x 2^20 transactions are more than the archive in pinned memory holds
    rows = 100_000
    with L.Context(workload=L.WORKLOAD_KV, kv_rows=rows, kv_fields=1, kv_field_bytes=4, max_txns=B,
                   kv_max_slots=1) as ctx:
        k, m, t = L.kv_generate(seed=1, rows=rows, fields=1, n_txns=B, n_slots=1, min_ops=1, max_ops=1, theta=0.6)
        ora = oracle.kv_epoch(kc.initial_table(rows, 1, 1), rows, 1, 1, k, m, t, 1, want_reads=False)
        dev = L.DeviceKvBatch(ctx, k, m, t, 1)
        runner = L.Batched(ctx, None, [L.kv_desc(dev)] * batches)
        for mode in (L.RUN_GRAPH, L.RUN_PLAIN, L.RUN_GRAPH):
            runner.run(mode)
            for i in range(batches):
                np.testing.assert_array_equal(runner.bitmap(i, L.TYPE_KV), ora.bitmap)
        runner.close()
        dev.free()
