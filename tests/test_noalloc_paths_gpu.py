"""ltpg_kv_epoch_noalloc against the oracle where its path changes: the
single-workgroup epoch (at most 2048 op slots), the per-row registers (at most
32,768 rows, or more op slots than the binned path holds) and the binned
EXECUTE, one call after another on the same scratch, TIDs in and out of order;
and replays of a captured call."""
import ctypes

import numpy as np
import pytest
import torch

import ltpg_amd as L
from oracle import oracle
from tests import kvcases as kc

pytestmark = pytest.mark.gpu


class Call:
    def __init__(self, rows, fields, fw, B, S, seed, theta=0.8, shuffled=False, bad=0):
        self.rows, self.fields, self.fw, self.B, self.S = rows, fields, fw, B, S
        keys, meta, tids = L.kv_generate(seed=seed, rows=rows, fields=fields, n_txns=B, n_slots=S, min_ops=1,
                                         max_ops=S, theta=theta, distinct_keys=False)
        if shuffled:
            tids = np.random.default_rng(seed).permutation(tids).astype(np.uint32)
        keys[:bad] = rows
        meta[:bad] = L.kv_meta(L.KV_READ, 0)
        self.bad, self.batch = bad, (keys, meta, tids)
        self.table0 = kc.initial_table(rows, fields, fw)
        dev = [torch.from_numpy(a.view(np.int64 if a.dtype.itemsize == 8 else np.int32)).cuda() for a in self.batch]
        self.dev = dev
        self.table = torch.from_numpy(self.table0.view(np.int32)).cuda()
        self.bitmap = torch.full(((B + 63) // 64,), -1, dtype=torch.int64, device="cuda")
        self.reads = torch.zeros(B * S * fw, dtype=torch.int32, device="cuda")
        self.result = torch.full((2,), -1, dtype=torch.int32, device="cuda")
        self.struct = L.KvBatch(B, S, *(d.data_ptr() for d in dev))

    def run(self, result=True):
        rc = L.lib.ltpg_kv_epoch_noalloc(self.table.data_ptr(), self.rows, self.fields, 4 * self.fw,
                                         ctypes.byref(self.struct), L.VALUES_RMW, self.bitmap.data_ptr(),
                                         self.reads.data_ptr(), self.result.data_ptr() if result else None,
                                         torch.cuda.current_stream().cuda_stream)
        assert rc == L.OK, L.lib.ltpg_last_error()

    def check(self, epochs=1, result=True):
        torch.cuda.synchronize()
        table = self.table0.copy()
        for _ in range(epochs):
            ora = oracle.kv_epoch(table, self.rows, self.fields, self.fw, *self.batch, self.S, inplace=True)
        np.testing.assert_array_equal(self.bitmap.cpu().numpy().view(np.uint64), ora.bitmap)
        np.testing.assert_array_equal(self.table.cpu().numpy().view(np.uint32), table)
        com = np.unpackbits(ora.bitmap.view(np.uint8), bitorder="little")[:self.B].astype(bool)
        keys, meta, _ = self.batch
        read = ((meta & 3) == L.KV_READ) & (keys < self.rows) & np.tile(com, self.S)
        got = self.reads.cpu().numpy().view(np.uint32).reshape(-1, self.fw)
        np.testing.assert_array_equal(got[read], ora.read_values.reshape(-1, self.fw)[read])
        assert not got[~read].any(), "only committed reads are written"
        if result:
            assert self.result.cpu().tolist() == [ora.commit_count, self.bad]


@pytest.mark.parametrize("rows,fw,B,S", [
    (3000, 25, 512, 4),              # 2048 op slots: one workgroup
    (3000, 25, 683, 3),              # 2049: registers
    (32_768, 1, 5000, 10),           # the most rows on the registers
    (32_769, 1, 5000, 10),           # binned, 8 bits of row per bucket
    (1 << 20, 2, 1000, 7),           # binned, one short tile
    (1_000_003, 5, 40_000, 9),       # commit list
    (200_000, 1, 1 << 20, 17),       # more op slots than the binned path holds
], ids=lambda v: str(v))
def test_noalloc_paths_match_oracle(gpu, rows, fw, B, S):
    for seed, shuffled in ((1, False), (2, True), (3, False)):
        if B * S > 1 << 24 and seed > 1:
            break
        c = Call(rows, 2, fw, B, S, seed, shuffled=shuffled, bad=3 if seed == 1 else 0)
        c.run(result=seed != 2)
        c.check(result=seed != 2)


@pytest.mark.parametrize("rows,B,S", [(2000, 100, 5), (20_000, 3000, 6), (100_000, 40_000, 6)])
def test_noalloc_captured_replays_match_oracle(gpu, rows, B, S):
    c = Call(rows, 2, 3, B, S, 5)
    other = Call(rows, 2, 3, B, S, 6, shuffled=True)
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        c.run()
        s.synchronize()
        c.table.copy_(torch.from_numpy(c.table0.view(np.int32)))
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            c.run()
        for k in range(1, 4):  # an eager call of another batch on the same scratch between replays
            g.replay()
            s.synchronize()
            c.check(epochs=k)
            other.run()
            s.synchronize()
            other.check(epochs=k)
