"""Calls that follow a single-workgroup epoch answer as they do after an epoch
of several kernels: the same sequence on both sides of the size where a context
changes from one to the other."""
import numpy as np
import pytest

import ltpg_amd as L
from tests import kvcases as kc

pytestmark = pytest.mark.gpu

# one workgroup; one op past it; one workgroup, chosen; several kernels, chosen
SHAPES = [(256, None), (257, None), (512, L.TUNE_SMALL_EPOCH), (257, 0)]


def context(rows, B, tuning):
    ctx = L.Context(workload=L.WORKLOAD_KV, kv_rows=rows, kv_fields=1, kv_field_bytes=4, max_txns=B, kv_max_slots=4)
    if tuning is not None:
        ctx.kv_set_tuning(tuning)
    ctx.kv_table_load(kc.initial_table(rows, 1, 1))
    return ctx


@pytest.mark.parametrize("B,tuning", SHAPES)
def test_check_after_a_reset_finds_no_conflict(gpu, B, tuning):
    rows = 50
    with context(rows, B, tuning) as ctx:
        for e in range(2):
            k, m, t = L.kv_generate(seed=e, rows=rows, fields=1, n_txns=B, n_slots=4, theta=0.5)
            ctx.kv_submit(k, m, t, 4)
            ctx.epoch_run()
            assert 0 < ctx.commit_count() < B // 2
            ctx.epoch_reset()
            ctx.epoch_run(L.PHASE_CHECK)
            assert ctx.commit_count() == B
            assert np.unpackbits(ctx.commit_bitmap().view(np.uint8), bitorder="little")[:B].all()


@pytest.mark.parametrize("B,tuning", SHAPES)
def test_check_again_counts_no_range_error_twice(gpu, B, tuning):
    rows, bad = 300, 9
    with context(rows, B, tuning) as ctx:
        for e in range(2):
            k, m, t = L.kv_generate(seed=e, rows=rows, fields=1, n_txns=B, n_slots=4, theta=0.5)
            k[:bad] = rows + np.arange(bad)
            ctx.kv_submit(k, m, t, 4)
            ctx.epoch_run()
            bits = ctx.commit_bitmap()
            ctx.epoch_run(L.PHASE_CHECK)
            with pytest.raises(L.LtpgError) as err:
                ctx.sync()
            assert err.value.code == L.ERR_RANGE and f" {bad} op(s)" in str(err.value)
            ctx.epoch_run(L.PHASE_CHECK)
            ctx.sync()
            np.testing.assert_array_equal(ctx.commit_bitmap(), bits)
            ctx.epoch_run(L.PHASE_EXECUTE)  # which counts them, as any EXECUTE does
            with pytest.raises(L.LtpgError):
                ctx.sync()
