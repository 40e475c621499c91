"""Binned EXECUTE where a tile's last buckets are empty and every slot of the
tile registers: the runs of those buckets begin at the tile's end, which for
the last tile of the largest batch is the end of the buffer."""
import os
import subprocess

import numpy as np
import pytest

import ltpg_amd as L
from oracle import oracle
from tests import kvcases as kc

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include "ltpg_internal.h"
#include <cstdio>
using namespace ltpg;
int main()
{
    const uint64_t shapes[][2] = {{10000000, 1 << 24}, {10000000, 10 << 20}, {40000, 4096 * 64}, {1000000, 1 << 20},
                                  {100000000, 1 << 24}, {9000000, 65536 * 16}};
    for (const auto &c : shapes) {
        const BinShape f = bin_shape(c[0], c[1]);
        const uint32_t T = 1u << f.tile_bits;
        const uint64_t entries = (uint64_t)f.tiles << f.tile_bits;
        for (uint32_t tile : {0u, f.tiles / 2, f.tiles - 1})
            for (uint32_t from : {0u, 1u, T / 2, T - 1, T})
                for (uint32_t to : {from, from + 1, T}) {
                    if (to > T || to < from) continue;
                    const uint32_t start = bin_run_start(tile, f.tile_bits, from, to), len = to - from;
                    for (uint32_t l : {0u, 1u, 31u, len ? len - 1 : 0u}) {
                        const uint64_t at = start + (l < len ? l : 0u);  // lane l of the run
                        const bool own = at >= ((uint64_t)tile << f.tile_bits) + from &&
                                         at < ((uint64_t)tile << f.tile_bits) + to;
                        if (at >= entries || (len && !own)) {
                            std::printf("rows %lu ops %lu tile %u run [%u, %u) lane %u: entry %lu of %lu\n",
                                        (unsigned long)c[0], (unsigned long)c[1], tile, from, to, l,
                                        (unsigned long)at, (unsigned long)entries);
                            return 1;
                        }
                    }
                }
    }
    std::puts("in bounds");
    return 0;
}
"""


def test_loads_of_empty_runs_stay_inside_the_buffer(tmp_path):
    src, exe = tmp_path / "runs.cpp", tmp_path / "runs"
    src.write_text(PROGRAM)
    r = subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                        "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(ROOT, "ltpg_amd", "csrc"),
                        str(src), "-o", str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout


@pytest.mark.gpu
@pytest.mark.parametrize("rows,B,S", [(40_000, 4096, 64), (1_000_000, 65_536, 16), (9_000_000, 65_536, 16),
                                      (9_000_000, 65_536, 64)], ids=lambda v: str(v))
@pytest.mark.parametrize("request_major", [False, True])
def test_full_tiles_of_reads_on_few_rows_match_oracle(gpu, rows, B, S, request_major):
    rng = np.random.default_rng(B)
    keys = rng.integers(0, 3, B * S).astype(np.uint64)
    meta = np.full(B * S, L.kv_meta(L.KV_READ, 0), np.uint32)
    tids = np.arange(B, dtype=np.uint32)
    table = kc.initial_table(rows, 1, 1)
    with L.Context(workload=L.WORKLOAD_KV, kv_rows=rows, kv_fields=1, kv_field_bytes=4, max_txns=B,
                   kv_max_slots=S) as ctx:
        ctx.kv_table_load(table)
        k, m = keys, meta
        if request_major:
            k, m = (np.ascontiguousarray(a.reshape(S, B).T).reshape(-1) for a in (keys, meta))
        ctx.kv_submit(k, m, tids, S, request_major=request_major)
        ctx.epoch_run()
        ctx.sync()
        ora = oracle.kv_epoch(table, rows, 1, 1, keys, meta, tids, S, inplace=True)
        assert ctx.commit_count() == ora.commit_count == B
        np.testing.assert_array_equal(ctx.commit_bitmap(), ora.bitmap)
        np.testing.assert_array_equal(ctx.kv_read_values(), ora.read_values)
        np.testing.assert_array_equal(ctx.kv_table_read(), table)
