"""Contexts whose read values fit the card packed, but not at the fields'
stride in device memory (17-word fields are 32 words apart there)."""
import numpy as np
import pytest

import ltpg_amd as L
from oracle import oracle
from tests import kvcases as kc

pytestmark = pytest.mark.gpu


def check(ctx, table, rows, fields, fw, B, S, scan, seed, counts=False):
    keys, meta, t = L.kv_generate(seed=seed, rows=rows, fields=fields, n_txns=B, n_slots=S, min_ops=1, max_ops=S,
                                  theta=0.3, read_pct=80, distinct_keys=False)
    pick = (meta & 3) == L.KV_READ
    length = np.random.default_rng(seed).integers(1, scan + 1, keys.size).astype(np.uint32)
    meta[pick] = (meta[pick] & ~np.uint32(3)) | L.KV_SCAN | (length[pick] - 1) << 24
    for request_major in (False, True):
        k, m = keys, meta
        if request_major:
            k, m = (np.ascontiguousarray(a.reshape(S, B).T).reshape(-1) for a in (keys, meta))
        ctx.kv_submit(k, m, t, S, request_major=request_major)
        ctx.epoch_run()
        ora = oracle.kv_epoch(table, rows, fields, fw, keys, meta, t, S, inplace=True, max_scan=scan)
        np.testing.assert_array_equal(ctx.commit_bitmap(), ora.bitmap)
        com = np.unpackbits(ora.bitmap.view(np.uint8), bitorder="little")[:B].astype(bool)
        n = np.where((meta & 3) == L.KV_SCAN, (meta >> 24).astype(np.int64) + 1, 0)
        n = np.where(np.tile(com, S), np.minimum(n, rows - keys.astype(np.int64)), 0)
        read = np.arange(scan)[None, :] < n[:, None]
        got, want = (v.reshape(B * S, scan, fw)[read] for v in (ctx.kv_read_values(), ora.read_values))
        np.testing.assert_array_equal(got, want)
    np.testing.assert_array_equal(ctx.kv_table_read().reshape(-1), table.reshape(-1))


# 64 x 12.8M op slots of up to 3 rows of 68 bytes: 167 GB packed, 315 GB apart
@pytest.mark.parametrize("flags", [0, L.FLAG_CONFLICT_COUNTS], ids=["fast", "counts"])
def test_read_values_that_fit_packed_only_match_oracle(gpu, flags):
    rows, fields, fw, scan = 20_000, 2, 17, 3
    with L.Context(workload=L.WORKLOAD_KV, kv_rows=rows, kv_fields=fields, kv_field_bytes=4 * fw,
                   max_txns=12_800_000, kv_max_slots=64, kv_max_scan=scan, flags=flags) as ctx:
        table = kc.initial_table(rows, fields, fw)
        ctx.kv_table_load(table)
        for seed, (B, S) in enumerate([(20, 5), (4001, 7), (32_771, 32)]):  # one workgroup, several, the commit list
            check(ctx, table, rows, fields, fw, B, S, scan, seed)
        if not flags:
            ctx.kv_set_tuning(L.TUNE_LANE_COPY)
            check(ctx, table, rows, fields, fw, 2003, 6, scan, 9)
