"""The calls that users of this library make, with their sizes.

listed() holds twelve of them and draw(rng) makes more of the same ranges;
prepare / run / work take one case each.  A case's "kind" names the entry
point:

  noalloc   ltpg_kv_epoch_noalloc on the caller's device arrays (a serving
            loop, or code under graph capture): returns the whole table, the
            commit bitmap, the read values and the result words;
  kv        Context: submit a batch, run the epoch's phases, read the commit
            bitmap back (the plain driver loop); with `values_back` the
            committed read values too;
  tpcc      the same for order-entry batches, all five transaction types;
  batched   Batched.run over a list of mixed batches, then every bitmap;
  serve     a burst of requests through a running Server, until every one has
            committed, and their completion records.

Every output is whole numbers (commit bits, table words, ids), so there is no
64-bit result to be near to: outputs are right or wrong.
"""
import ctypes
import math

import numpy as np
import torch

import ltpg_amd as L


def _kv(kind, name, rows, fields, words, txns, slots, min_ops, read_pct, theta, **more):
    c = dict(kind=kind, rows=rows, fields=fields, words=words, txns=txns, slots=slots, min_ops=min_ops,
             read_pct=read_pct, theta=theta, scan=0, hot=False, copyback=False, request_major=False, host=False,
             values_back=False, counts=False)
    c.update(more)
    return dict(c, name=name) if name else c


def _tpcc(name, warehouses, txns, os=0, sl=0, dl=0, intended=False, host=False, values_back=False):
    c = dict(kind="tpcc", warehouses=warehouses, txns=txns, os=os, sl=sl, dl=dl, intended=intended, host=host,
             values_back=values_back)
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest call: a serving loop's epoch of a few requests
        _kv("noalloc", "noalloc-64x4", 10_000, 10, 1, 64, 4, 1, 50, 0.8),
        # the u32 table of the replay configuration: 65,536 transactions of 10 ops
        _kv("noalloc", "noalloc-65536x10", 1_000_000, 10, 1, 65_536, 10, 10, 50, 0.8),
        # records of 10 x 100 bytes, ragged transactions, odd sizes
        _kv("noalloc", "noalloc-262143x16-wide", 1_000_003, 10, 25, 262_143, 16, 1, 50, 0.6),
        # the large-batch configuration: 2^20 transactions of 16 ops on 10M records of 10 x 100 bytes
        _kv("kv", "kv-1048576x16-zipf0.6", 10_000_000, 10, 25, 1 << 20, 16, 16, 50, 0.6),
        # the same under heavy skew, where almost everything aborts
        _kv("kv", "kv-1048576x16-zipf0.99", 10_000_000, 10, 25, 1 << 20, 16, 16, 50, 0.99),
        # 9 reads and 1 read-modify-write on uniform keys: most transactions commit
        _kv("kv", "kv-1048576x10-read90", 10_000_000, 10, 25, 1 << 20, 10, 10, 90, 0.0),
        # scans of 10 rows on the u32 table
        _kv("kv", "kv-10000x10-scans", 1_000_000, 10, 1, 10_000, 10, 10, 90, 0.0, scan=10),
        # a batch handed over from host memory, one row declared hot, reads read back
        _kv("kv", "kv-16000x8-host-hot", 1_000_000, 10, 2, 16_000, 8, 1, 50, 0.99, hot=True, host=True,
            values_back=True),
        # order entry at its measured configuration: half NewOrder, half Payment
        _tpcc("tpcc-262144", 64, 1 << 18),
        # every order-entry type at an ordinary size, from host memory, values read back
        _tpcc("tpcc-10001-all-types", 16, 10_001, os=600, sl=600, dl=400, intended=True, host=True, values_back=True),
        # uneven batches of both workloads in one submission
        dict(kind="batched", name="batched-24", batches=24, lo=1000, hi=200_000, rows=10_000_000, words=25, slots=32,
             theta=0.9, warehouses=16),
        # requests that arrive at a running server
        dict(kind="serve", name="serve-2000x16", rows=1_000_000, words=25, requests=2000, slots=16, theta=0.99),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["noalloc", "noalloc", "noalloc", "kv", "kv", "kv", "kv", "tpcc", "tpcc", "batched", "serve"])
    theta = rng.choice([0.0, 0.6, 0.8, 0.9, 0.99])
    if kind == "noalloc":
        slots = rng.randint(2, 24)
        txns = _log(rng, 32, min(1 << 20, (1 << 23) // slots))
        words = rng.choice([1, 2, 4, 25]) if txns * slots <= 1 << 22 else rng.choice([1, 2, 4])
        return _kv(kind, "", _log(rng, 4000, 1 << 20), rng.randint(1, 12), words, txns, slots, rng.randint(1, slots),
                   rng.choice([0, 50, 90, 100]), theta, copyback=rng.random() < 0.2)
    if kind == "kv":
        slots = rng.randint(1, 64)
        txns = _log(rng, 200, min(1 << 20, (1 << 24) // slots))
        words = rng.choice([1, 2, 4, 16, 25])
        rows = _log(rng, 20_000, 10_000_000)
        scan = rng.choice([0, 0, 0, 10]) if words <= 2 and txns * slots <= 200_000 else 0
        small = txns * slots * words <= 1 << 22
        return _kv(kind, "", rows, 10, words, txns, slots, rng.choice([1, slots]), rng.choice([20, 50, 90]), theta,
                   scan=scan, hot=rng.random() < 0.2, copyback=rng.random() < 0.2, request_major=rng.random() < 0.25,
                   host=small and rng.random() < 0.3, values_back=small and not scan and rng.random() < 0.5,
                   counts=rng.random() < 0.15)
    if kind == "tpcc":
        txns = _log(rng, 200, 1 << 18)
        small = txns <= 20_000
        extra = small and rng.random() < 0.6
        return _tpcc("", rng.choice([1, 4, 16, 64]), txns, os=txns // 16 if extra else 0, sl=txns // 17 if extra else 0,
                     dl=txns // 25 if extra else 0, intended=rng.random() < 0.5, host=small and rng.random() < 0.5,
                     values_back=small and rng.random() < 0.5)
    if kind == "batched":
        return dict(kind=kind, batches=rng.randint(2, 24), lo=500, hi=_log(rng, 4000, 200_000),
                    rows=_log(rng, 100_000, 10_000_000), words=rng.choice([2, 25]), slots=rng.choice([4, 16, 32]),
                    theta=theta, warehouses=rng.choice([2, 16]))
    return dict(kind=kind, rows=_log(rng, 50_000, 1_000_000), words=rng.choice([2, 25]),
                requests=_log(rng, 200, 2000), slots=rng.randint(2, 32), theta=rng.choice([0.6, 0.9, 0.99]))


class State:
    """What a program holds across calls; contexts close last."""

    def __init__(self, case):
        self.case = case
        self.kv = self.tp = self.runner = self.server = None
        self.device_batches = []

    def __del__(self):
        if self.server:
            self.server.stop()
        if self.runner:
            self.runner.close()
        for b in self.device_batches:
            b.free()
        for ctx in (self.kv, self.tp):
            if ctx:
                ctx.close()


def _kv_batch(c, seed, tid_base=0):
    return L.kv_generate(seed=seed, rows=c["rows"], fields=c["fields"], n_txns=c["txns"], n_slots=c["slots"],
                         min_ops=c["min_ops"], max_ops=c["slots"], read_pct=c["read_pct"], theta=c["theta"],
                         tid_base=tid_base, distinct_keys=c["rows"] > 64 * c["slots"], scan_len=c["scan"])


def _cuda(a):
    return torch.from_numpy(a.view(np.int64 if a.dtype.itemsize == 8 else np.int32)).cuda()


def _prepare_noalloc(st, seed):
    c = st.case
    keys, meta, tids = (_cuda(a) for a in _kv_batch(c, seed))
    n_ops = c["txns"] * c["slots"]
    word = torch.arange(c["fields"], dtype=torch.int32, device="cuda") + seed % 1000
    st.table = word.repeat_interleave(c["words"]).repeat(c["rows"])
    st.bitmap = torch.zeros((c["txns"] + 63) // 64, dtype=torch.int64, device="cuda")
    st.reads = torch.zeros(n_ops * c["words"], dtype=torch.int32, device="cuda")
    st.result = torch.zeros(2, dtype=torch.int32, device="cuda")
    st.inputs = (keys, meta, tids)
    st.batch = L.KvBatch(c["txns"], c["slots"], keys.data_ptr(), meta.data_ptr(), tids.data_ptr())
    st.values = L.VALUES_COPYBACK if c["copyback"] else L.VALUES_RMW


def _run_noalloc(st):
    c = st.case
    rc = L.lib.ltpg_kv_epoch_noalloc(st.table.data_ptr(), c["rows"], c["fields"], 4 * c["words"],
                                     ctypes.byref(st.batch), st.values, st.bitmap.data_ptr(), st.reads.data_ptr(),
                                     st.result.data_ptr(), torch.cuda.current_stream().cuda_stream)
    if rc != L.OK:
        raise L.LtpgError(rc, "ltpg_kv_epoch_noalloc")
    return {"table": st.table, "bitmap": st.bitmap, "reads": st.reads, "result": st.result}


def _prepare_kv(st, seed):
    c = st.case
    st.kv = L.Context(workload=L.WORKLOAD_KV, kv_rows=c["rows"], kv_fields=c["fields"], kv_field_bytes=4 * c["words"],
                      max_txns=c["txns"], kv_max_slots=c["slots"], kv_max_scan=c["scan"],
                      kv_hot_row=0 if c["hot"] else L.NO_HOT_ROW,
                      values=L.VALUES_COPYBACK if c["copyback"] else L.VALUES_RMW,
                      flags=L.FLAG_CONFLICT_COUNTS if c["counts"] else 0)
    st.kv.kv_fill_reference()
    keys, meta, tids = _kv_batch(c, seed)
    st.read_slots = ((meta & 3) == L.KV_READ).reshape(c["slots"], c["txns"])
    if c["request_major"]:
        keys, meta = (np.ascontiguousarray(a.reshape(c["slots"], c["txns"]).T).reshape(-1) for a in (keys, meta))
    if c["host"]:
        st.host = (keys, meta, tids)
    else:
        st.device = L.DeviceKvBatch(st.kv, keys, meta, tids, c["slots"], request_major=c["request_major"])
        st.device_batches.append(st.device)


def _run_kv(st):
    c, ctx = st.case, st.kv
    if c["host"]:
        ctx.kv_submit(*st.host, c["slots"], request_major=c["request_major"])
    else:
        ctx.kv_submit_device(st.device)
    ctx.epoch_run(L.PHASE_ALL)
    bits = ctx.commit_bitmap()
    out = [bits.view(np.int64)]
    if c["counts"]:
        out.append(ctx.conflict_counters().view(np.int32))
    if c["values_back"]:
        # results are the read slots of committed transactions; the other entries are dropped
        values = ctx.kv_read_values().view(np.int32).reshape(c["slots"], c["txns"], c["words"])
        out.append(values * (st.read_slots & _committed(bits, c["txns"]))[:, :, None])
    return out


def _committed(bits, n):
    return np.unpackbits(bits.view(np.uint8), count=n, bitorder="little").view(bool)


class _Buffers:
    """Device buffers freed together, as a device batch is."""

    def __init__(self, bufs):
        self.bufs = bufs

    def free(self):
        for b in self.bufs:
            b.free()


TYPES = (L.TYPE_NEWORDER, L.TYPE_PAYMENT, L.TYPE_ORDERSTATUS, L.TYPE_STOCKLEVEL, L.TYPE_DELIVERY)


def _prepare_tpcc(st, seed):
    c = st.case
    st.tp = L.Context(workload=L.WORKLOAD_TPCC, tpcc_warehouses=c["warehouses"],
                      max_txns=c["txns"] + c["os"] + c["sl"] + c["dl"],
                      rules=L.RULES_INTENDED if c["intended"] else L.RULES_REFERENCE)
    st.tp.tpcc_populate(seed)
    b = L.TpccGenerator(warehouses=c["warehouses"], seed=seed).next(c["txns"])
    st.n_no = b.n_no
    ro = L.readonly_batch(b, c["warehouses"], c["os"], c["sl"], seed) if c["os"] or c["sl"] else None
    dl = L.delivery_batch(b, c["warehouses"], c["dl"], seed) if c["dl"] else None
    if not c["host"]:
        b, bufs = L.upload_tpcc_batch(st.tp, b)
        if ro:
            ro, more = L.upload_readonly_batch(st.tp, ro)
            bufs += more
        if dl:
            dl, more = L.upload_delivery_batch(st.tp, dl)
            bufs += more
        st.device_batches.append(_Buffers(bufs))
    st.batch = (b, ro, dl)


def _run_tpcc(st):
    c, ctx = st.case, st.tp
    b, ro, dl = st.batch
    mem = L.MEM_HOST if c["host"] else L.MEM_DEVICE
    ctx.tpcc_submit(b, mem)
    if ro:
        ctx.tpcc_submit_readonly(ro, mem)
    if dl:
        ctx.tpcc_submit_delivery(dl, mem)
    ctx.epoch_run(L.PHASE_ALL)
    types = [t for t, n in zip(TYPES, (1, 1, c["os"], c["sl"], c["dl"])) if n]
    bits = [ctx.tpcc_bitmap(t) for t in types]
    out = [b.view(np.int64) for b in bits]
    if c["values_back"]:
        counts = dict(zip(TYPES, (st.n_no, c["txns"] - st.n_no, c["os"], c["sl"], c["dl"])))
        for t, b in zip(types, bits):
            n = counts[t]
            out.append(ctx.tpcc_read_values(t).view(np.int32).reshape(-1, n) * _committed(b, n))
    return out


def _prepare_batched(st, seed):
    c = st.case
    rng = np.random.default_rng(c["batches"])  # sizes belong to the case, contents to the seed
    shape = dict(rows=c["rows"], fields=10, slots=c["slots"], min_ops=1, read_pct=50, theta=c["theta"], scan=0)
    sizes = np.exp(rng.uniform(np.log(c["lo"]), np.log(c["hi"]), c["batches"])).astype(int)
    st.kv = L.Context(workload=L.WORKLOAD_KV, kv_rows=c["rows"], kv_fields=10, kv_field_bytes=4 * c["words"],
                      max_txns=c["hi"], kv_max_slots=c["slots"])
    st.kv.kv_fill_reference()
    st.tp = L.Context(workload=L.WORKLOAD_TPCC, tpcc_warehouses=c["warehouses"], max_txns=c["hi"])
    st.tp.tpcc_populate(seed)
    gen = L.TpccGenerator(warehouses=c["warehouses"], seed=seed)
    descs, st.types = [], []
    for i, n in enumerate(int(s) for s in sizes):
        if i % 2 == 0:
            keys, meta, tids = _kv_batch(dict(shape, txns=n), seed + i, tid_base=i * c["hi"])
            dev = L.DeviceKvBatch(st.kv, keys, meta, tids, c["slots"])
            st.device_batches.append(dev)
            descs.append(L.kv_desc(dev))
            st.types.append((L.TYPE_KV,))
        else:
            dev, bufs = L.upload_tpcc_batch(st.tp, gen.next(n, tid_base=i * c["hi"]))
            st.device_batches.append(_Buffers(bufs))
            descs.append(L.tpcc_desc(dev))
            st.types.append((L.TYPE_NEWORDER, L.TYPE_PAYMENT))
    st.runner = L.Batched(st.kv, st.tp, descs)


def _run_batched(st):
    st.runner.run(L.RUN_GRAPH)
    return [np.concatenate([st.runner.bitmap(i, t) for t in types]).view(np.int64) for i, types in enumerate(st.types)]


def _prepare_serve(st, seed):
    c = st.case
    st.kv = L.Context(workload=L.WORKLOAD_KV, kv_rows=c["rows"], kv_fields=10, kv_field_bytes=4 * c["words"],
                      max_txns=4096, kv_max_slots=c["slots"])
    st.kv.kv_fill_reference()
    keys, meta, _ = _kv_batch(dict(rows=c["rows"], fields=10, txns=c["requests"], slots=c["slots"], min_ops=1,
                                   read_pct=50, theta=c["theta"], scan=0), seed)
    st.requests = [np.ascontiguousarray(a.reshape(c["slots"], c["requests"]).T) for a in (keys, meta)]
    st.server = L.Server(kv_ctx=st.kv, kv_ops=c["slots"])


def _run_serve(st):
    first = st.server.submit_kv(*st.requests)
    st.server.drain()
    done = []
    while len(done) < st.case["requests"]:
        done += st.server.poll()
    # which request a record is for, and its type; the epoch it committed in depends on when requests arrived
    keys = np.asarray(st.requests[0][:, 0]).view(np.int64)
    order = np.array(sorted((d["id"] - first, d["type"]) for d in done), dtype=np.int64)
    return {"done": order, "first_key": keys[order[:, 0]]}


_PREPARE = {"noalloc": _prepare_noalloc, "kv": _prepare_kv, "tpcc": _prepare_tpcc, "batched": _prepare_batched,
            "serve": _prepare_serve}
_RUN = {"noalloc": _run_noalloc, "kv": _run_kv, "tpcc": _run_tpcc, "batched": _run_batched, "serve": _run_serve}


def prepare(case, seed):
    st = State(case)
    _PREPARE[case["kind"]](st, seed)
    return st


def run(state):
    return _RUN[state.case["kind"]](state)


def _behind(rate, theta, rows):
    """P(op of priority quantile u is behind another of `rate` ops of a
    Zipf(theta) draw on its row), for 32 values of u: the mean over the draw
    of 1 - exp(-u m), m = the ops expected on the row."""
    edges = np.unique(np.geomspace(1, rows + 1, 400).astype(np.int64))
    mid = np.sqrt(edges[:-1] * (edges[1:] - 1.0))
    p = mid ** -theta
    n = np.diff(edges)
    p /= (p * n).sum()
    u = np.geomspace(1e-6, 1, 32)[:, None]
    return u[:, 0], -(n * p * np.expm1(-u * rate * p)).sum(axis=1)


def _commits(c, reads, writes):
    """Expected share of transactions that commit (reads and writes per
    transaction): no write behind another writer of its row, and not both a
    read behind a writer and a write behind a reader."""
    u, w = _behind(c["txns"] * writes, c["theta"], c["rows"])
    r = _behind(c["txns"] * reads, c["theta"], c["rows"])[1]
    commit = (1 - w) ** writes * (1 - (1 - (1 - w) ** reads) * (1 - (1 - r) ** writes))
    return float((np.diff(u, prepend=0.0) * commit).sum())


def _kv_bytes(c):
    ops = (c["min_ops"] + c["slots"]) / 2
    reads, writes = ops * c["read_pct"] / 100, ops * (100 - c["read_pct"]) / 100
    rows_read = reads * max(1, c["scan"])
    field = 4 * c["words"]
    inputs = c["txns"] * (12 * c["slots"] + 4 + 1 / 8)
    fields = c["txns"] * _commits(c, rows_read, writes) * (rows_read + writes) * 2 * field
    back = c["txns"] * c["slots"] * field if c["values_back"] else 0
    return inputs + fields + back


def _tpcc_bytes(n, both=0.5):
    # query fields of a NewOrder of 10 lines and of a Payment; the reads and writes of the Payments
    return n * both * (32 + 120) + n * both * (40 + 96 + 96 + 84) + n / 8


def work(case):
    c = case
    if c["kind"] in ("noalloc", "kv"):
        b = _kv_bytes(c)
    elif c["kind"] == "tpcc":
        b = _tpcc_bytes(c["txns"]) + 36 * c["os"] + 16 * c["sl"] + 24 * c["dl"]
    elif c["kind"] == "batched":
        mean = (c["hi"] - c["lo"]) / math.log(c["hi"] / c["lo"])
        b = c["batches"] * mean / 2 * (12 * c["slots"] + 4 + 1 / 8) + _tpcc_bytes(c["batches"] * mean / 2)
    else:
        b = c["requests"] * (12 * c["slots"] + 16)
    return {"bytes": float(b), "flops": 0.0}
