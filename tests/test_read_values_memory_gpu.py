"""Reading the read values back takes no device memory."""
import ctypes

import pytest

import ltpg_amd as L
from tests import kvcases as kc

pytestmark = pytest.mark.gpu


def free_memory():
    hip = ctypes.CDLL("libamdhip64.so")
    left, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipMemGetInfo(ctypes.byref(left), ctypes.byref(total)) == 0
    return left.value


def taken_by_reading_back(fw):
    rows, B, S = 20_000, 40_000, 9
    keys, meta, t = L.kv_generate(seed=fw, rows=rows, fields=1, n_txns=B, n_slots=S, theta=0.0, read_pct=90)
    with L.Context(workload=L.WORKLOAD_KV, kv_rows=rows, kv_fields=1, kv_field_bytes=4 * fw, max_txns=B,
                   kv_max_slots=S) as ctx:
        ctx.kv_table_load(kc.initial_table(rows, 1, fw))
        ctx.kv_submit(keys, meta, t, S)
        ctx.epoch_run()
        ctx.sync()
        before = free_memory()
        assert ctx.kv_read_values().size == B * S * fw
        return before - free_memory()


@pytest.mark.parametrize("fw", [17, 25])
def test_reading_back_allocates_nothing(gpu, fw):
    taken_by_reading_back(16)  # the runtime's own buffer for its first large copy to the host
    assert taken_by_reading_back(16) == 0  # fields that are not padded
    assert taken_by_reading_back(fw) == 0
