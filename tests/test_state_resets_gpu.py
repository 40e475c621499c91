"""Registers, flags and commit counts start over where they should: past the
last epoch number, with flag arrays of odd length, and between the batches of
a replayed run."""
import numpy as np
import pytest

import ltpg_amd as L
from oracle import oracle
from tests import kvcases as kc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B", [1, 15, 17, 333])
def test_epochs_past_the_wrap_match_oracle(gpu, B):
    rows, S = 3 * B + 1, 3
    with L.Context(workload=L.WORKLOAD_KV, kv_rows=rows, kv_fields=1, kv_field_bytes=4, max_txns=B,
                   kv_max_slots=S) as ctx:
        table = kc.initial_table(rows, 1, 1)
        ctx.kv_table_load(table)
        for e in range(520):
            k, m, t = L.kv_generate(seed=e, rows=rows, fields=1, n_txns=B, n_slots=S, min_ops=1, max_ops=S, theta=0.5,
                                    distinct_keys=False)
            ctx.kv_submit(k, m, t, S)
            ctx.epoch_run()
            ora = oracle.kv_epoch(table, rows, 1, 1, k, m, t, S, inplace=True, want_reads=False)
            np.testing.assert_array_equal(ctx.commit_bitmap(), ora.bitmap)
        np.testing.assert_array_equal(ctx.kv_table_read(), table)


@pytest.mark.parametrize("sizes", [(700,), (3, 5000, 40_000, 1), (0, 4000, 0), (50,) * 300], ids=["1", "4", "empty", "300"])
def test_commit_counts_of_a_replayed_run(gpu, sizes):
    rows, S = 20_000, 8
    with L.Context(workload=L.WORKLOAD_KV, kv_rows=rows, kv_fields=1, kv_field_bytes=4, max_txns=max(sizes),
                   kv_max_slots=S) as ctx:
        table = kc.initial_table(rows, 1, 1)
        ctx.kv_table_load(table)
        batches = [L.kv_generate(seed=i, rows=rows, fields=1, n_txns=n, n_slots=S, min_ops=1, max_ops=S, theta=0.8,
                                 distinct_keys=False) for i, n in enumerate(sizes)]
        devs = [L.DeviceKvBatch(ctx, *b, S) for b in batches]
        runner = L.Batched(ctx, None, [L.kv_desc(d) for d in devs])
        ctx.commit_totals(reset=True)
        total = 0
        for _ in range(3):
            runner.run(L.RUN_GRAPH)
            for i, b in enumerate(batches):
                if sizes[i] == 0:
                    count = 0
                    continue
                ora = oracle.kv_epoch(table, rows, 1, 1, *b, S, inplace=True, want_reads=False)
                np.testing.assert_array_equal(runner.bitmap(i, L.TYPE_KV), ora.bitmap)
                count = ora.commit_count
                total += count
            assert ctx.commit_count() == count
            assert ctx.commit_totals()[0] == total
        runner.close()
        for d in devs:
            d.free()
