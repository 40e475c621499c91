"""The single-workgroup epoch against the oracle: where a context takes it by
default and just past that, where a caller chose it, fields below, at and above
four words, scans, a hot row with as many fields as there may be, duplicate
writes, both layouts, copy-back and invalid ops."""
import numpy as np
import pytest

import ltpg_amd as L
from oracle import oracle
from tests import kvcases as kc

pytestmark = pytest.mark.gpu


def check(rows, fields, fw, B, S, tuning=None, theta=0.9, read_pct=50, hot=False, scan=0, copyback=False, epochs=3):
    hot_row = 2 if hot else L.NO_HOT_ROW
    values = L.VALUES_COPYBACK if copyback else L.VALUES_RMW
    with L.Context(workload=L.WORKLOAD_KV, kv_rows=rows, kv_fields=fields, kv_field_bytes=4 * fw, max_txns=B,
                   kv_max_slots=S, kv_max_scan=scan, kv_hot_row=hot_row, values=values) as ctx:
        if tuning is not None:
            ctx.kv_set_tuning(tuning)
        table = kc.initial_table(rows, fields, fw)
        ctx.kv_table_load(table)
        for e in range(epochs):
            keys, meta, t = L.kv_generate(seed=e, rows=rows, fields=fields, n_txns=B, n_slots=S, min_ops=1, max_ops=S,
                                          theta=theta, read_pct=read_pct, distinct_keys=False)
            rng = np.random.default_rng(e)
            if hot:
                keys[rng.random(keys.size) < 0.3] = hot_row
            if scan:
                pick = (meta & 3) == L.KV_READ
                length = rng.integers(1, scan + 1, keys.size).astype(np.uint32)
                meta[pick] = (meta[pick] & ~np.uint32(3)) | L.KV_SCAN | (length[pick] - 1) << 24
            if e == 1:
                t = rng.permutation(t).astype(np.uint32)
                keys[rng.integers(0, keys.size)] = rows
            rm = e == 2
            k, m = keys, meta
            if rm:
                k, m = (np.ascontiguousarray(a.reshape(S, B).T).reshape(-1) for a in (keys, meta))
            ctx.kv_submit(k, m, t, S, request_major=rm)
            ctx.epoch_run()
            ora = oracle.kv_epoch(table, rows, fields, fw, keys, meta, t, S, inplace=True, hot_row=hot_row,
                                  values=values, max_scan=scan)
            np.testing.assert_array_equal(ctx.commit_bitmap(), ora.bitmap)
            assert ctx.commit_count() == ora.commit_count
            com = np.unpackbits(ora.bitmap.view(np.uint8), bitorder="little")[:B].astype(bool)
            kind, per = meta & 3, max(1, scan)
            n = np.where(kind == L.KV_READ, 1, np.where(kind == L.KV_SCAN, (meta >> 24) + 1, 0))
            n = np.where((keys < rows) & np.tile(com, S), np.minimum(n, rows - keys.astype(np.int64)), 0)
            read = np.arange(per)[None, :] < n[:, None]
            got, want = (v.reshape(B * S, per, fw)[read] for v in (ctx.kv_read_values(), ora.read_values))
            np.testing.assert_array_equal(got, want)
        np.testing.assert_array_equal(ctx.kv_table_read().reshape(-1), table.reshape(-1))


@pytest.mark.parametrize("B,S,fw", [
    (1, 1, 1), (64, 1, 3), (16, 64, 1), (64, 16, 16), (1024, 1, 2), (341, 3, 5), (655, 1, 25),  # one workgroup
    (1025, 1, 2), (512, 3, 1), (656, 1, 25), (64, 16, 17),                                      # past it
])
@pytest.mark.parametrize("more", [{}, dict(hot=True), dict(copyback=True)], ids=["", "hot", "copyback"])
def test_default_small_epochs_match_oracle(gpu, B, S, fw, more):
    check(5000, 3, fw, B, S, **more)


@pytest.mark.parametrize("fw", [1, 3, 4, 5, 25, 64, 65, 256])
@pytest.mark.parametrize("B,S,read_pct", [(2048, 1, 0), (1024, 2, 50), (128, 16, 100), (37, 33, 50)])
def test_chosen_small_epochs_match_oracle(gpu, fw, B, S, read_pct):
    check(50_000, 2, fw, B, S, tuning=L.TUNE_SMALL_EPOCH, theta=0.3, read_pct=read_pct)


@pytest.mark.parametrize("B,S,scan", [(100, 4, 5), (20, 16, 3), (512, 4, 7)])
def test_small_epochs_with_scans_match_oracle(gpu, B, S, scan):
    check(3000, 2, 3, B, S, tuning=L.TUNE_SMALL_EPOCH if B > 500 else None, scan=scan)


def test_small_epoch_with_the_widest_hot_row_matches_oracle(gpu):
    check(60, 1024, 1, 2048, 1, tuning=L.TUNE_SMALL_EPOCH, theta=0.0, read_pct=20, hot=True)


@pytest.mark.parametrize("fw", [1, 2, 3, 4])
@pytest.mark.parametrize("scan,hot", [(0, True), (1, False), (8, False), (9, True), (19, False)])
def test_larger_epochs_with_scans_and_a_hot_row_match_oracle(gpu, fw, scan, hot):
    # several kernels: reads of narrow fields alone and eight rows at a time
    check(4000, 3, fw, 1500, 9, theta=0.5, scan=scan, hot=hot)


@pytest.mark.parametrize("tuning", [None, L.TUNE_SMALL_EPOCH])
def test_check_again_after_a_small_epoch(gpu, tuning):
    rows, B, S = 300, 200, 4
    with L.Context(workload=L.WORKLOAD_KV, kv_rows=rows, kv_fields=1, kv_field_bytes=4, max_txns=B,
                   kv_max_slots=S) as ctx:
        if tuning is not None:
            ctx.kv_set_tuning(tuning)
        table = kc.initial_table(rows, 1, 1)
        ctx.kv_table_load(table)
        for e in range(3):
            k, m, t = L.kv_generate(seed=e, rows=rows, fields=1, n_txns=B, n_slots=S, theta=0.5)
            ctx.kv_submit(k, m, t, S)
            ctx.epoch_run()
            ora = oracle.kv_epoch(table, rows, 1, 1, k, m, t, S, inplace=True, want_reads=False)
            for _ in range(2):
                ctx.epoch_run(L.PHASE_CHECK)
                np.testing.assert_array_equal(ctx.commit_bitmap(), ora.bitmap)
                assert ctx.commit_count() == ora.commit_count
        np.testing.assert_array_equal(ctx.kv_table_read(), table)
