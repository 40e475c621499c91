"""Order-entry EXECUTE of large epochs (claimed rows, settled, STOCK binned)
against the oracle, on batches whose orders, order lines, histories and
customers collide: one transaction below its lower bound, at it, and above
with last blocks part full; TIDs in and out of order; NewOrders or Payments
only; rows outside their tables; with Order-Status and Deliveries (which read
the registers it leaves) and with Stock-Level (which keeps the one-kernel
form); both workgroup sizes; epochs one after the other."""
import numpy as np
import pytest

import ltpg_amd as L
from oracle import oracle

pytestmark = pytest.mark.gpu

SEED = 0x4C545047
SPLIT = 3 << 14


def _batch(W, n, pct, seed, shuffled, bad):
    """A generator batch with a third of its orders' ids drawn from few, so
    that rows are written by several transactions."""
    rng = np.random.default_rng(seed)
    b = L.TpccGenerator(warehouses=W, seed=seed, neworder_pct=pct).next(n)
    for name, hi in (("O_ID", 30000), ("N_O_ID", 30000), ("O_OL_ID", 449_985)):
        f = b.nf(name)
        pick = rng.random(f.size) < 0.3
        f[pick] = rng.integers(0, hi, int(pick.sum()))
    f = b.pf("H_ID")
    pick = rng.random(f.size) < 0.3
    f[pick] = rng.integers(0, 30000, int(pick.sum()))
    if shuffled:
        for f in (b.nf("TID"), b.pf("TID")):
            f[:] = rng.permutation(f)
    if bad and b.n_no:
        b.nf("O_ID")[3::997] = 4_000_000
        b.nf("O_OL_ID")[5::991] = W * 450_000 - 3  # some lines past the table
        b.nf("OL_SUPPLY_W_ID", 2)[7::983] = W
    if bad and b.n_pay:
        b.pf("H_ID")[1::977] = 4_000_000
    return b


@pytest.mark.parametrize("n,pct,shuffled,bad,small", [
    (SPLIT - 1, 50, False, False, False),
    (SPLIT, 50, False, True, False),
    (SPLIT, 50, True, False, True),
    (SPLIT + 4097, 90, False, False, True),
    (SPLIT + 1, 100, True, True, False),
    (SPLIT + 1, 0, False, True, False),
])
@pytest.mark.parametrize("rules", [L.RULES_REFERENCE, L.RULES_INTENDED], ids=["reference", "intended"])
@pytest.mark.parametrize("extra", ["none", "order-status+delivery", "stock-level"])
def test_split_execute_matches_oracle(gpu, n, pct, shuffled, bad, small, rules, extra):
    W = 2
    with L.Context(workload=L.WORKLOAD_TPCC, tpcc_warehouses=W, max_txns=n + 4000, rules=rules) as ctx:
        ctx.tpcc_populate(SEED)
        tables, ora = oracle.tpcc_populate(W, SEED), oracle.TpccOracle(W)
        ctx.tpcc_set_tuning(L.TUNE_TPCC_SMALL_BLOCKS if small else 0)
        for ep in range(2):
            b = _batch(W, n, pct, 10 * ep + pct, shuffled, bad)
            ro = dl = None
            ctx.tpcc_submit(b)
            if extra != "none":
                n_os, n_sl = (1500, 0) if extra == "order-status+delivery" else (0, 1500)
                ro = L.readonly_batch(b, W, n_os, n_sl, seed=ep, tid_lo=0, tid_hi=n)
                ctx.tpcc_submit_readonly(ro)
                if n_os:
                    dl = L.delivery_batch(b, W, 1200, seed=ep, tid_lo=0, tid_hi=n)
                    ctx.tpcc_submit_delivery(dl)
            ctx.epoch_run()
            o = ora.epoch(tables, b, rules, L.VALUES_RMW, ro=ro, dl=dl)
            if o.range_errors:
                with pytest.raises(L.LtpgError) as e:
                    ctx.sync()
                assert e.value.code == L.ERR_RANGE and f"{o.range_errors} op" in str(e.value)
            else:
                ctx.sync()
            np.testing.assert_array_equal(ctx.tpcc_bitmap(L.TYPE_NEWORDER), o.no_bitmap[:(b.n_no + 63) // 64])
            np.testing.assert_array_equal(ctx.tpcc_bitmap(L.TYPE_PAYMENT), o.pay_bitmap[:(b.n_pay + 63) // 64])
            if dl:
                np.testing.assert_array_equal(ctx.tpcc_bitmap(L.TYPE_DELIVERY), o.dl["bitmap"])
        for t in range(9):
            np.testing.assert_array_equal(ctx.tpcc_table_read(t), tables[t])
