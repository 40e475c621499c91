"""Order-entry epochs where the number of launches changes: the CID phase with
EXECUTE in one call and by itself, the queries' C_IDs where none runs, and the
YTD sums in the WRITEBACK kernel and in one of their own."""
import numpy as np
import pytest

import ltpg_amd as L

pytestmark = pytest.mark.gpu

TYPES = (L.TYPE_NEWORDER, L.TYPE_PAYMENT)
PHASES = (L.PHASE_CID, L.PHASE_EXECUTE, L.PHASE_CHECK, L.PHASE_WRITEBACK)


@pytest.mark.parametrize("txns", [1, 300, 20_000, 49_152])
@pytest.mark.parametrize("cid", [True, False], ids=["cid", "no-cid"])
def test_phases_in_one_call_match_single_phases(gpu, txns, cid):
    W, got = 2, []
    for single in (False, True):
        with L.Context(workload=L.WORKLOAD_TPCC, tpcc_warehouses=W, max_txns=txns) as ctx:
            ctx.tpcc_populate(3)
            gen = L.TpccGenerator(warehouses=W, seed=4)
            for e in range(3):
                b = gen.next(txns, tid_base=e * txns)
                ctx.tpcc_submit(b)
                if b.n_pay:
                    np.testing.assert_array_equal(ctx.tpcc_payment_cid(), b.pf("C_ID"))
                if single:
                    for p in PHASES[0 if cid else 1:]:
                        ctx.epoch_run(p)
                else:
                    ctx.epoch_run(L.PHASE_ALL if cid else L.PHASE_ALL & ~L.PHASE_CID)
                if b.n_pay and not cid:
                    np.testing.assert_array_equal(ctx.tpcc_payment_cid(), b.pf("C_ID"))
                got += [ctx.tpcc_bitmap(t) for t in TYPES] + [ctx.tpcc_payment_cid()]
            got += [ctx.tpcc_table_read(t) for t in (L.TPCC_CUSTOMER, L.TPCC_HISTORY, L.TPCC_DISTRICT)]
    half = len(got) // 2
    for a, b in zip(got[:half], got[half:]):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("small", [0, L.TUNE_TPCC_SMALL_BLOCKS], ids=["256", "64"])
@pytest.mark.parametrize("W,txns", [(1, 5), (3, 9000), (64, 100_000), (372, 3000), (373, 3000)])
def test_ytd_sums_of_committed_payments(gpu, W, txns, small):
    # 372 warehouses are the most whose sums fit beside the WRITEBACK kernel
    with L.Context(workload=L.WORKLOAD_TPCC, tpcc_warehouses=W, max_txns=txns) as ctx:
        ctx.tpcc_populate(1)
        ctx.tpcc_set_tuning(small)
        tables = [(L.TPCC_WAREHOUSE, 2, W), (L.TPCC_DISTRICT, 3, 10 * W)]
        want = [ctx.tpcc_table_read(t).reshape(-1, rows)[col].copy() for t, col, rows in tables]
        gen = L.TpccGenerator(warehouses=W, seed=7)
        for e in range(2):
            b = gen.next(txns, tid_base=e * txns)
            ctx.tpcc_submit(b)
            ctx.epoch_run()
            com = np.unpackbits(ctx.tpcc_bitmap(L.TYPE_PAYMENT).view(np.uint8), count=b.n_pay,
                                bitorder="little").astype(bool)
            w, d, amount = (b.pf(f)[com].astype(np.int64) for f in ("W_ID", "D_ID", "H_AMOUNT"))
            np.add.at(want[0], w, amount.astype(np.uint32))
            np.add.at(want[1], w * 10 + d, amount.astype(np.uint32))
        for (t, col, rows), v in zip(tables, want):
            np.testing.assert_array_equal(ctx.tpcc_table_read(t).reshape(-1, rows)[col], v)


def test_freed_batch_keeps_its_customers(gpu):
    # a device batch freed through its context right after the submit
    with L.Context(workload=L.WORKLOAD_TPCC, tpcc_warehouses=1, max_txns=500) as ctx:
        ctx.tpcc_populate(1)
        b = L.TpccGenerator(warehouses=1, seed=2).next(500)
        dev, bufs = L.upload_tpcc_batch(ctx, b)
        ctx.tpcc_submit(dev, L.MEM_DEVICE)
        for x in bufs:
            x.free()
        np.testing.assert_array_equal(ctx.tpcc_payment_cid(), b.pf("C_ID"))
