"""The key-value launch shape a context picks by size, against the oracle at
the sizes where the pick or its tiles change: the binned EXECUTE (tiles of
4096 and 16384 op slots) just above its lower bound, with whole and partial
last tiles, batches narrower and wider than a tile, TIDs in and out of order
and equal, a hot row, both batch layouts, invalid ops; and the per-op register
path below it."""
import numpy as np
import pytest

import ltpg_amd as L
from oracle import oracle
from tests import kvcases as kc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,B,S", [
    (40_000, 4096, 63),          # below the binned path's 2^18 ops: per-op registers
    (40_000, 4096, 64),          # exactly 2^18 ops, whole tiles
    (32_769, 20_003, 14),        # fewest rows, odd batch, partial last tile
    (70_000, 1_000_001 // 3, 1), # one slot
    (300_000, 65_539, 64),       # 2^22 ops and more: tiles of 16384
    (9_000_000, 66_000, 64),     # 1024 buckets of 16384 rows
    (9_000_000, 66_000, 16),     # 256 hashed buckets of 65536 rows
    (9_000_000, 99_991, 20),     # 512 hashed buckets, tiles of 16384
], ids=lambda v: str(v))
@pytest.mark.parametrize("tids", ["ordered", "shuffled", "equal"])
def test_default_shape_matches_oracle(gpu, rows, B, S, tids):
    fields, fw = 2, 1
    rng = np.random.default_rng(B + S)
    hot = 0 if tids == "equal" else L.NO_HOT_ROW
    keys, meta, t = L.kv_generate(seed=B, rows=rows, fields=fields, n_txns=B, n_slots=S, min_ops=1, max_ops=S,
                                  theta=0.9, read_pct=40, distinct_keys=False)
    if tids == "shuffled":
        t = rng.permutation(t).astype(np.uint32)
    elif tids == "equal":
        t = (t // 5).astype(np.uint32)
    bad = rng.choice(keys.size, 7, replace=False)
    keys[bad[:4]] = rows + bad[:4].astype(np.uint64) * (1 << 31)
    meta[bad[4:]] = L.kv_meta(L.KV_WRITE, fields)
    table = kc.initial_table(rows, fields, fw)
    with L.Context(workload=L.WORKLOAD_KV, kv_rows=rows, kv_fields=fields, kv_field_bytes=4 * fw, max_txns=B,
                   kv_max_slots=S, kv_hot_row=hot) as ctx:
        ctx.kv_table_load(table)
        # the first epoch slot-major, the second request-major
        for request_major in (False, True):
            k, m = keys, meta
            if request_major:
                k, m = (np.ascontiguousarray(a.reshape(S, B).T).reshape(-1) for a in (keys, meta))
            ctx.kv_submit(k, m, t, S, request_major=request_major)
            ctx.epoch_run()
            with pytest.raises(L.LtpgError) as e:
                ctx.sync()
            assert e.value.code == L.ERR_RANGE
            ora = oracle.kv_epoch(table, rows, fields, fw, keys, meta, t, S, inplace=True, hot_row=hot)
            np.testing.assert_array_equal(ctx.commit_bitmap(), ora.bitmap)
            com = np.unpackbits(ora.bitmap.view(np.uint8), bitorder="little")[:B].astype(bool)
            ok = (keys < rows) & (((meta >> 8) & 0xffff) < fields) & ((meta & 3) == L.KV_READ)
            read = (ok.reshape(S, B) & com).reshape(-1)
            np.testing.assert_array_equal(ctx.kv_read_values()[read], ora.read_values[read])
        np.testing.assert_array_equal(ctx.kv_table_read(), table)


@pytest.mark.parametrize("crowd", [4000, 8191, 8192, 40_000])
@pytest.mark.parametrize("tids", ["ordered", "shuffled"])
def test_crowded_hash_bucket_matches_oracle(gpu, crowd, tids):
    """Binned EXECUTE with hashed buckets, 90 % of the operations in one
    bucket: as many distinct rows there as its hash table nearly or exactly
    holds, and more (that bucket then goes through its row arrays part by
    part)."""
    rows, B, S = 6_000_000, 20_000, 14  # 2^23 hashed rows, 64 buckets
    rng = np.random.default_rng(crowd)
    keys, meta, t = L.kv_generate(seed=crowd, rows=rows, fields=1, n_txns=B, n_slots=S, theta=0.0, read_pct=30)
    inverse = pow(0x9E3779B1, -1, 1 << 23)
    bucket = (np.arange(1 << 17, dtype=np.uint64) + np.uint64(5 << 17)) * np.uint64(inverse) % np.uint64(1 << 23)
    bucket = bucket[bucket < rows][:crowd]
    assert bucket.size == crowd
    pick = rng.random(keys.size) < 0.9
    keys[pick] = bucket[rng.integers(0, crowd, int(pick.sum()))]
    if tids == "shuffled":
        t = rng.permutation(t).astype(np.uint32)
    table = kc.initial_table(rows, 1, 1)
    with L.Context(workload=L.WORKLOAD_KV, kv_rows=rows, kv_fields=1, kv_field_bytes=4, max_txns=B,
                   kv_max_slots=S) as ctx:
        ctx.kv_table_load(table)
        ctx.kv_submit(keys, meta, t, S)
        ctx.epoch_run()
        ctx.sync()
        ora = oracle.kv_epoch(table, rows, 1, 1, keys, meta, t, S, inplace=True)
        np.testing.assert_array_equal(ctx.commit_bitmap(), ora.bitmap)
        np.testing.assert_array_equal(ctx.kv_table_read(), table)


@pytest.mark.parametrize("B", [32_767, 32_768, 36_865])
@pytest.mark.parametrize("fw,scan", [(3, 0), (4, 0), (5, 3), (17, 0), (25, 0), (33, 0)])
def test_commit_list_matches_oracle(gpu, B, fw, scan):
    """CHECK's list of committed transactions (2^20 op slots and more) and
    the field copies from it: list blocks of 4096 with a remainder of one,
    fields of one lane, whole and overlapping 16-byte pieces, padded and
    unpadded rows, scans; the phases in one call and one by one; read values
    read back in whole and cut inside a field."""
    rows, fields, S = 500_000, 2, 32
    keys, meta, t = L.kv_generate(seed=B + fw, rows=rows, fields=fields, n_txns=B, n_slots=S, min_ops=1, max_ops=S,
                                  theta=0.3, read_pct=60, scan_len=scan, distinct_keys=False)
    if scan:
        keys[::97] = rows - 2  # clipped at the end of the table
    table = kc.initial_table(rows, fields, fw)
    with L.Context(workload=L.WORKLOAD_KV, kv_rows=rows, kv_fields=fields, kv_field_bytes=4 * fw, max_txns=B,
                   kv_max_slots=S, kv_max_scan=scan) as ctx:
        ctx.kv_table_load(table)
        for ep, steps in enumerate([[L.PHASE_ALL], [L.PHASE_EXECUTE, L.PHASE_CHECK, L.PHASE_WRITEBACK],
                                    [L.PHASE_EXECUTE | L.PHASE_CHECK, L.PHASE_WRITEBACK]]):
            k, m = keys, meta
            if ep == 1:
                k, m = (np.ascontiguousarray(a.reshape(S, B).T).reshape(-1) for a in (keys, meta))
            ctx.kv_submit(k, m, t, S, request_major=ep == 1)
            for phases in steps:
                ctx.epoch_run(phases)
            ctx.sync()
            ora = oracle.kv_epoch(table, rows, fields, fw, keys, meta, t, S, inplace=True, max_scan=scan)
            np.testing.assert_array_equal(ctx.commit_bitmap(), ora.bitmap)
            assert ctx.commit_count() == ora.commit_count
            com = np.unpackbits(ora.bitmap.view(np.uint8), bitorder="little")[:B].astype(bool)
            n = max(1, scan)
            kinds = (meta & 3).astype(np.int64)
            lens = np.where(kinds == 3, (meta >> 24).astype(np.int64) + 1, (kinds == 1).astype(np.int64))
            row = np.arange(n)[None, :]
            read = (row < lens[:, None]) & ((keys.astype(np.int64)[:, None] + row) < rows)
            read &= np.tile(com, S)[:, None]
            got = ctx.kv_read_values()
            np.testing.assert_array_equal(got.reshape(-1, fw)[read.reshape(-1)],
                                          ora.read_values.reshape(-1, fw)[read.reshape(-1)])
            part = np.zeros(7 * fw + 1, np.uint32)
            assert L.lib.ltpg_kv_read_values(ctx.handle, part.ctypes.data_as(L._lib.c_u32p), part.size) == L.OK
            np.testing.assert_array_equal(part, got[:part.size])
        np.testing.assert_array_equal(ctx.kv_table_read(), table)
