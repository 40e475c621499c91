"""ltpg_kv_epoch_noalloc against the oracle where its path changes: the
single-workgroup epoch (at most 2048 op slots), the per-row registers (at most
32,768 rows, or more op slots than the binned path holds) and the binned
EXECUTE, one call after another on the same scratch, TIDs in and out of order;
and replays of a captured call."""
import ctypes

import numpy as np
import pytest

import ltpg_amd as L
from oracle import oracle
from tests import kvcases as kc

pytestmark = pytest.mark.gpu


class Hip:
    """The runtime's stream and graph calls that the captured replays need."""

    def __init__(self):
        self.lib = ctypes.CDLL("libamdhip64.so")

    def __call__(self, name, *args):
        rc = getattr(self.lib, name)(*args)
        assert rc == 0, (name, rc)

    def new(self, name, *args):
        out = ctypes.c_void_p()
        self(name, ctypes.byref(out), *args)
        return out


class Call:
    def __init__(self, ctx, rows, fields, fw, B, S, seed, theta=0.8, shuffled=False, bad=0):
        self.rows, self.fields, self.fw, self.B, self.S = rows, fields, fw, B, S
        keys, meta, tids = L.kv_generate(seed=seed, rows=rows, fields=fields, n_txns=B, n_slots=S, min_ops=1,
                                         max_ops=S, theta=theta, distinct_keys=False)
        if shuffled:
            tids = np.random.default_rng(seed).permutation(tids).astype(np.uint32)
        keys[:bad] = rows
        meta[:bad] = L.kv_meta(L.KV_READ, 0)
        self.bad, self.batch = bad, (keys, meta, tids)
        self.table0 = kc.initial_table(rows, fields, fw)
        self.dev = L.DeviceKvBatch(ctx, keys, meta, tids, S)
        self.out = [np.full(self.table0.shape, 0, np.uint32), np.full((B + 63) // 64, -1, np.int64).view(np.uint64),
                    np.zeros(B * S * fw, np.uint32), np.full(2, -1, np.int32).view(np.uint32)]
        self.bufs = [L.DeviceBuffer(ctx, a.nbytes) for a in self.out]
        self.reset()
        for k in (1, 2, 3):
            self.bufs[k].upload(self.out[k])
        self.struct = self.dev.struct()

    def reset(self):
        self.bufs[0].upload(self.table0)

    def run(self, result=True, stream=None):
        table, bitmap, reads, res = (ctypes.c_void_p(b.ptr) for b in self.bufs)
        rc = L.lib.ltpg_kv_epoch_noalloc(table, self.rows, self.fields, 4 * self.fw, ctypes.byref(self.struct),
                                         L.VALUES_RMW, bitmap, reads, res if result else None, stream)
        assert rc == L.OK, L.lib.ltpg_last_error()

    def free(self):
        self.dev.free()
        for b in self.bufs:
            b.free()

    def check(self, epochs=1, result=True):
        for buf, a in zip(self.bufs, self.out):
            buf.download(a)
        table_out, bitmap, reads, res = self.out
        table = self.table0.copy()
        for _ in range(epochs):
            ora = oracle.kv_epoch(table, self.rows, self.fields, self.fw, *self.batch, self.S, inplace=True)
        np.testing.assert_array_equal(bitmap, ora.bitmap)
        np.testing.assert_array_equal(table_out, table)
        com = np.unpackbits(ora.bitmap.view(np.uint8), bitorder="little")[:self.B].astype(bool)
        keys, meta, _ = self.batch
        read = ((meta & 3) == L.KV_READ) & (keys < self.rows) & np.tile(com, self.S)
        got = reads.reshape(-1, self.fw)
        np.testing.assert_array_equal(got[read], ora.read_values.reshape(-1, self.fw)[read])
        assert not got[~read].any(), "only committed reads are written"
        if result:
            assert res.tolist() == [ora.commit_count, self.bad]


@pytest.mark.parametrize("rows,fw,B,S", [
    (3000, 24, 512, 4),              # 2048 op slots, 49,152 words: one workgroup
    (3000, 25, 512, 4),              # more words
    (3000, 256, 192, 1),             # 49,152 words in few fields
    (3000, 25, 683, 3),              # 2049: registers
    (32_768, 1, 5000, 10),           # the most rows on the registers
    (32_769, 1, 5000, 10),           # binned, 8 bits of row per bucket
    (1 << 20, 2, 1000, 7),           # binned, one short tile
    (1_000_003, 5, 40_000, 9),       # chunks of transactions
    (1_000_003, 5, 120_001, 9),      # commit list
    (200_000, 1, 1 << 20, 17),       # more op slots than the binned path holds
], ids=lambda v: str(v))
def test_noalloc_paths_match_oracle(gpu, rows, fw, B, S):
    hip = Hip()
    with L.Context(workload=L.WORKLOAD_KV, kv_rows=64, kv_fields=1, max_txns=64, kv_max_slots=1) as ctx:
        for seed, shuffled in ((1, False), (2, True), (3, False)):
            if B * S > 1 << 24 and seed > 1:
                break
            c = Call(ctx, rows, 2, fw, B, S, seed, shuffled=shuffled, bad=3 if seed == 1 else 0)
            c.run(result=seed != 2)
            hip("hipDeviceSynchronize")
            c.check(result=seed != 2)
            c.free()


@pytest.mark.parametrize("rows,B,S", [(2000, 100, 5), (20_000, 3000, 6), (100_000, 40_000, 6)])
def test_noalloc_captured_replays_match_oracle(gpu, rows, B, S):
    hip = Hip()
    with L.Context(workload=L.WORKLOAD_KV, kv_rows=64, kv_fields=1, max_txns=64, kv_max_slots=1) as ctx:
        c = Call(ctx, rows, 2, 3, B, S, 5)
        other = Call(ctx, rows, 2, 3, B, S, 6, shuffled=True)
        s = hip.new("hipStreamCreate")
        c.run(stream=s)
        hip("hipStreamSynchronize", s)
        c.reset()
        hip("hipStreamBeginCapture", s, 0)
        c.run(stream=s)
        graph = ctypes.c_void_p()
        hip("hipStreamEndCapture", s, ctypes.byref(graph))
        run = hip.new("hipGraphInstantiate", graph, None, None, ctypes.c_size_t(0))
        for k in range(1, 4):  # an eager call of another batch on the same scratch between replays
            hip("hipGraphLaunch", run, s)
            hip("hipStreamSynchronize", s)
            c.check(epochs=k)
            other.run(stream=s)
            hip("hipStreamSynchronize", s)
            other.check(epochs=k)
        hip("hipGraphExecDestroy", run)
        hip("hipGraphDestroy", graph)
        hip("hipStreamDestroy", s)
        c.free()
        other.free()


@pytest.mark.parametrize("result", [True, False])
def test_noalloc_empty_epoch(gpu, result):
    hip = Hip()
    with L.Context(workload=L.WORKLOAD_KV, kv_rows=64, kv_fields=1, max_txns=64, kv_max_slots=1) as ctx:
        c = Call(ctx, 100, 2, 1, 8, 2, 1)
        c.struct.n_txns = 0
        c.run(result=result)
        hip("hipDeviceSynchronize")
        c.bufs[3].download(c.out[3])
        assert c.out[3].tolist() == ([0, 0] if result else [0xFFFFFFFF] * 2)
        c.free()
