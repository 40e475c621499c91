"""A context takes memory for binned STOCK writes only where its epochs use
them: up to 2^27 STOCK rows, 1,342 warehouses."""
import ctypes

import pytest

import ltpg_amd as L

pytestmark = pytest.mark.gpu


def free_memory():
    hip = ctypes.CDLL("libamdhip64.so")
    left, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipMemGetInfo(ctypes.byref(left), ctypes.byref(total)) == 0
    return left.value


def taken(warehouses, txns):
    before = free_memory()
    with L.Context(workload=L.WORKLOAD_TPCC, tpcc_warehouses=warehouses, max_txns=txns):
        return before - free_memory()


def test_no_bins_for_tables_beyond_them(gpu):
    txns = 1 << 22
    taken(1, 100)  # what the runtime keeps
    bins = 15 * txns * 4
    # one warehouse more brings tables of some 40 MB, but no bins of 252 MB
    assert taken(1342, txns) - taken(1343, txns) > bins // 2
