"""WRITEBACK of a list of committed transactions against the oracle, where the
list gets long enough for 64 transactions per wave (131,072 commits with 2^20
op slots) and just below: duplicate writes of one transaction, fields of 1 to
25 words, a hot row, copy-back, both batch layouts, invalid ops."""
import numpy as np
import pytest

import ltpg_amd as L
from oracle import oracle
from tests import kvcases as kc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,fields,fw,B,S,read_pct,more", [
    (4_000_000, 2, 1, 140_000, 16, 90, {}),                      # most commit: 64 per wave
    (4_000_000, 2, 3, 150_001, 16, 97, {}),                      # a ragged last wave
    (1_000_000, 3, 4, 300_007, 4, 50, {}),
    (1_000_000, 2, 25, 200_000, 8, 95, {}),
    (3_000_000, 1, 1, 1 << 20, 1, 0, {}),                        # one write each: no list
    (3_000_000, 1, 1, 1 << 20, 2, 30, {}),                       # the fewest ops of few slots that are listed
    (3_000_000, 1, 1, (1 << 20) - 1, 2, 30, {}),                 # not listed
    (2_000_000, 2, 2, 270_000, 5, 60, dict(hot=3)),
    (2_000_000, 2, 5, 200_000, 7, 80, dict(copyback=True)),
    (4_000_000, 2, 1, 140_000, 16, 90, dict(request_major=True)),
    (4_000_000, 2, 1, 140_000, 17, 95, {}),                      # too many slots for it
    (2_000_000, 2, 6, 131_000, 10, 97, {}),                      # too few commits
], ids=lambda v: str(v))
def test_long_lists_match_oracle(gpu, rows, fields, fw, B, S, read_pct, more):
    hot = more.get("hot", L.NO_HOT_ROW)
    values = L.VALUES_COPYBACK if more.get("copyback") else L.VALUES_RMW
    rm = more.get("request_major", False)
    keys, meta, t = L.kv_generate(seed=B + S, rows=rows, fields=fields, n_txns=B, n_slots=S, min_ops=1, max_ops=S,
                                  theta=0.0, read_pct=read_pct, distinct_keys=False)
    rng = np.random.default_rng(S)
    if S > 1:  # some transactions write one field several times
        k2, m2 = keys.reshape(S, B), meta.reshape(S, B)
        for b in rng.choice(B, 2000, replace=False):
            to = rng.integers(0, S, 3)
            k2[to, b], m2[to, b] = k2[to[0], b], L.kv_meta(L.KV_WRITE, fields - 1)
    if hot != L.NO_HOT_ROW:
        keys[rng.choice(keys.size, B, replace=False)] = hot
    keys[rng.choice(keys.size, 5, replace=False)] = rows + 7
    table = kc.initial_table(rows, fields, fw)
    with L.Context(workload=L.WORKLOAD_KV, kv_rows=rows, kv_fields=fields, kv_field_bytes=4 * fw, max_txns=B,
                   kv_max_slots=S, kv_hot_row=hot, values=values) as ctx:
        ctx.kv_table_load(table)
        k, m = keys, meta
        if rm:
            k, m = (np.ascontiguousarray(a.reshape(S, B).T).reshape(-1) for a in (keys, meta))
        ctx.kv_submit(k, m, t, S, request_major=rm)
        ctx.epoch_run()
        ora = oracle.kv_epoch(table, rows, fields, fw, keys, meta, t, S, inplace=True, hot_row=hot,
                              want_reads=False, values=values)
        np.testing.assert_array_equal(ctx.commit_bitmap(), ora.bitmap)
        with pytest.raises(L.LtpgError) as e:
            ctx.sync()
        assert e.value.code == L.ERR_RANGE
        got = ctx.kv_table_read().reshape(-1)
        np.testing.assert_array_equal(got, table.reshape(-1))
