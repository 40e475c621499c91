"""WRITEBACK with 64 listed transactions per wave against the oracle, every case
with as many commits as that takes (131,072, and 2^20 op slots among them): a
hot row, copy-back, 2- to 5-word fields, duplicate writes of one transaction and
invalid ops, on 8 slots (the fewest that are listed from 2^20 op slots on) and
9."""
import numpy as np
import pytest

import ltpg_amd as L
from oracle import oracle
from tests import kvcases as kc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,fields,fw,B,S,read_pct,hot,copyback", [
    (4_000_000, 2, 2, 270_000, 9, 90, 3, False),
    (4_000_000, 1, 4, 270_000, 9, 80, 0, False),
    (4_000_000, 2, 5, 200_000, 9, 95, None, True),
    (4_000_000, 2, 3, 270_000, 8, 90, 7, True),
    (4_000_000, 3, 4, 300_007, 8, 85, None, False),
    (4_000_000, 1, 17, 262_144, 8, 85, 1, False),
], ids=lambda v: str(v))
def test_lists_in_slots_match_oracle(gpu, rows, fields, fw, B, S, read_pct, hot, copyback):
    hot_row = L.NO_HOT_ROW if hot is None else hot
    values = L.VALUES_COPYBACK if copyback else L.VALUES_RMW
    keys, meta, t = L.kv_generate(seed=B + S, rows=rows, fields=fields, n_txns=B, n_slots=S, min_ops=1, max_ops=S,
                                  theta=0.0, read_pct=read_pct, distinct_keys=False)
    rng = np.random.default_rng(S)
    k2, m2 = keys.reshape(S, B), meta.reshape(S, B)
    for b in rng.choice(B, 2000, replace=False):  # one field written several times
        to = rng.integers(0, S, 3)
        k2[to, b], m2[to, b] = k2[to[0], b], L.kv_meta(L.KV_WRITE, fields - 1)
    if hot is not None:
        keys[rng.choice(keys.size, B, replace=False)] = hot
    keys[rng.choice(keys.size, 5, replace=False)] = rows + 7
    table = kc.initial_table(rows, fields, fw)
    with L.Context(workload=L.WORKLOAD_KV, kv_rows=rows, kv_fields=fields, kv_field_bytes=4 * fw, max_txns=B,
                   kv_max_slots=S, kv_hot_row=hot_row, values=values) as ctx:
        ctx.kv_table_load(table)
        ctx.kv_submit(keys, meta, t, S)
        ctx.epoch_run()
        ora = oracle.kv_epoch(table, rows, fields, fw, keys, meta, t, S, inplace=True, hot_row=hot_row,
                              want_reads=False, values=values)
        assert ora.commit_count >= 1 << 17 and ora.commit_count * S >= 1 << 20, "too few commits for this form"
        np.testing.assert_array_equal(ctx.commit_bitmap(), ora.bitmap)
        with pytest.raises(L.LtpgError) as e:
            ctx.sync()
        assert e.value.code == L.ERR_RANGE
        np.testing.assert_array_equal(ctx.kv_table_read().reshape(-1), table.reshape(-1))
