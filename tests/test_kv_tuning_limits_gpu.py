"""LTPG_TUNE_PARTITIONED is refused above 8192 * 16384 rows, whether or not the
context has bins for its default shape."""
import pytest

import ltpg_amd as L

pytestmark = pytest.mark.gpu

LIMIT = 8192 * 16384


@pytest.mark.parametrize("B", [1000, 1 << 18], ids=["without bins", "with bins"])
@pytest.mark.parametrize("rows", [LIMIT, LIMIT + 1])
def test_rows_limit_of_the_partitioned_shape(gpu, rows, B):
    with L.Context(workload=L.WORKLOAD_KV, kv_rows=rows, kv_fields=1, kv_field_bytes=4, max_txns=B,
                   kv_max_slots=16) as ctx:
        if rows <= LIMIT:
            ctx.kv_set_tuning(L.TUNE_PARTITIONED)
        else:
            with pytest.raises(L.LtpgError) as err:
                ctx.kv_set_tuning(L.TUNE_PARTITIONED)
            assert err.value.code == L.ERR_UNSUPPORTED
