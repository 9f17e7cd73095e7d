"""The measured work of the transaction path: what a program of this library
has it do, through the public entry points, from the smallest call to the
largest.

Kinds of case (the forms that the library offers):

  static   gcctb_run_plain_static: tables, ops, reads and order in the caller's
           own device buffers, one batch per call, nothing allocated
  plain    gcctb_run_plain: the reference driver's batch after batch launches
  persist  gcctb_run_persistent: the loaded stream in one launch, at the tuned
           launch shape (autotune.lookup), as bench.py runs it
  graph    gcctb_run_graph: the same launches replayed from one hipGraph
  tpcc     TPC-C orders in the plain form

The serving form (gcctb_serve) is not among them: its launch waits for copies
on a second stream, which several contexts in one process, as measured here,
may put behind that launch on one hardware queue.

A pass of the context forms runs the loaded transactions once and brings the
result back to pinned host memory with gcctb_fetch: every read's value or, for
`out` = "table", the whole table.  The table of a scheme whose serialization
order depends on timing (every scheme but gacco and gputx) agrees between two
runs but for the few cells that transactions in flight together both wrote;
its reads do only at low contention, so contended cases of those schemes
return the table.  The table keeps each pass's result, as in a program that
runs on.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

import gpu_cc_tb_amd as g
from gpu_cc_tb_amd import autotune, workloads

ORDERED = ("gacco", "gputx")  # their outcome is fixed by the transaction ids
COLS = 10                     # u64 cells per row (80 B), the bench workload's table
STATIC_SHAPE = (3, 8)         # run_plain_static's default launch shape


def _case(kind, scheme, rows, ntx, theta, read_ratio, *, len_min=16, len_max=16, batch=65536, out="reads"):
    return {"kind": kind, "scheme": scheme, "rows": rows, "ntx": ntx, "theta": theta, "read_ratio": read_ratio,
            "len_min": len_min, "len_max": len_max, "batch": batch, "out": out}


def listed():
    def named(name, c):
        return dict(c, name=name)

    return [
        # a handful of requests on a caller's own buffers: latency and launches
        named("static_silo_tiny", _case("static", "silo", 1000003, 40, 0.1, 0.9)),
        # an ordinary batch: odd sizes, transactions of 4 to 32 ops
        named("static_tpl_nw_mid", _case("static", "tpl_nw", 131071, 6007, 0.1, 0.5, len_min=4, len_max=32)),
        # one full batch of the reference's size (65,536 transactions of 16 ops)
        named("static_mvcc_full", _case("static", "mvcc", 1048576, 65536, 0.1, 0.9)),
        # the bench workload: 1,048,576 transactions on 10,485,760 rows, low contention
        named("persist_silo_1m", _case("persist", "silo", 10485760, 1048576, 0.1, 0.9)),
        # half the ops write, sizes off every power of two
        named("persist_tpl_wd_300k", _case("persist", "tpl_wd", 1048573, 300007, 0.1, 0.5)),
        # a skewed stream: hot keys, aborts and retries
        named("persist_tictoc_hot", _case("persist", "tictoc", 2097152, 131072, 0.9, 0.9, out="table")),
        # the bench workload under the two schemes that order every access first
        named("persist_gacco_1m", _case("persist", "gacco", 10485760, 1048576, 0.1, 0.9)),
        named("persist_gputx_1m", _case("persist", "gputx", 10485760, 1048576, 0.1, 0.9)),
        # long queues on the hot rows, transactions of 4 to 32 ops
        named("persist_gacco_hot", _case("persist", "gacco", 4194304, 262144, 0.99, 0.5, len_min=4, len_max=32)),
        # the driver's own structure: one launch per rank level
        named("plain_gputx_64k", _case("plain", "gputx", 1048576, 65536, 0.1, 0.9)),
        # and the same structure under the other schemes: batches of 65,536
        named("plain_to_262k", _case("plain", "to", 10485760, 262144, 0.1, 0.9)),
        # TPC-C orders, 16 warehouses, batch after batch
        named("tpcc_gacco_new_order", _case("tpcc", "gacco", 16, 131072, 0.0, 0.0, batch=16384)),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _lengths(rng):
    """Ops per transaction: the bench's 16, the stream's 4 to 32, or another fixed count."""
    k = rng.random()
    if k < 0.4:
        return 16, 16
    if k < 0.7:
        return 4, 32
    n = rng.randint(1, 32)
    return n, n


def draw(rng):
    """One more case of the ranges above."""
    kind = rng.choices(["static", "persist", "plain", "tpcc"], [5, 9, 4, 2])[0]
    timed = [s for s in g.SCHEMES if s not in ORDERED]  # outcome depends on timing
    lo, hi = _lengths(rng)
    if kind == "static":
        # Read-only, or a table sized so that either no two transactions meet
        # in a cell or many do: a handful of meetings is a toss that two runs
        # of one program decide differently.
        scheme, ntx = rng.choice(timed), _log_int(rng, 1, min(131072, 1048576 // hi))
        nops = ntx * (lo + hi) // 2
        if nops < 700:
            rows, rr = rng.randint(900000, 1048576), rng.choice([0.5, 0.9])
        elif 100000 < nops < 524288:
            rows, rr = 2 * nops, 0.5
        elif nops >= 524288:
            rows, rr = 1048576, 0.9
        if rng.random() < 0.35 or 700 <= nops <= 100000:
            return _case("static", scheme, _log_int(rng, 64 * hi, 1048576), ntx, rng.choice([0.0, 0.1, 0.6, 0.99]), 1.0,
                         len_min=lo, len_max=hi, batch=ntx)
        return _case("static", scheme, rows, ntx, rng.choice([0.0, 0.1]), rr, len_min=lo, len_max=hi, batch=ntx)
    if kind == "tpcc":
        if rng.random() < 0.6:
            return _case("tpcc", "gacco", rng.randint(4, 16), _log_int(rng, 1000, 131072), 0.0, 0.0,
                         batch=rng.choice([16384, 65536]))
        # the final quantities and counts of the stock do not depend on the order
        return _case("tpcc", rng.choice(["silo", "tpl_nw", "to"]), rng.randint(8, 16), _log_int(rng, 1000, 65536),
                     0.0, 0.0, batch=rng.choice([16384, 65536]), out="table")
    most = 16000000 // hi  # no more ops than the bench workload's
    if kind == "plain":
        if rng.random() < 0.3:
            kind = "graph"
        if rng.random() < 0.5:
            return _case(kind, "gacco", _log_int(rng, 1000000, 10485760), _log_int(rng, 1000, min(most, 500000)),
                         rng.choice([0.0, 0.1, 0.6]), rng.choice([0.5, 0.9, 1.0]), len_min=lo, len_max=hi,
                         batch=rng.choice([16384, 65536, 262144]))
        if rng.random() < 0.3:
            return _case(kind, "gputx", _log_int(rng, 1000000, 10485760), _log_int(rng, 1000, 65536), 0.1,
                         rng.choice([0.9, 1.0]), len_min=lo, len_max=hi)
        return _case(kind, rng.choice(timed), 10485760, _log_int(rng, 200000, 700000), 0.1,
                     rng.choice([0.9, 1.0]), batch=rng.choice([65536, 262144]))
    k = rng.random()
    if k < 0.3:  # the outcome fixed: any size and skew
        return _case("persist", "gacco", _log_int(rng, 100000, 10485760), _log_int(rng, 100, most),
                     rng.choice([0.0, 0.1, 0.6, 0.9, 0.99]), rng.choice([0.5, 0.9, 1.0]), len_min=lo, len_max=hi)
    if k < 0.55:
        return _case("persist", "gputx", _log_int(rng, 1000000, 10485760), _log_int(rng, 100, min(most, 500000)),
                     rng.choice([0.0, 0.1, 0.6]), rng.choice([0.9, 1.0]), len_min=lo, len_max=hi)
    if k < 0.7:  # the other six, read-only at the bench workload's size
        return _case("persist", rng.choice(timed), _log_int(rng, 1000000, 10485760), _log_int(rng, 100, most),
                     rng.choice([0.0, 0.1, 0.6]), 1.0, len_min=lo, len_max=hi)
    if k < 0.85:  # and with writes
        return _case("persist", rng.choice(timed), _log_int(rng, 700000, 1400000), _log_int(rng, 400000, 900000),
                     rng.choice([0.0, 0.1]), rng.choice([0.5, 0.9]))
    return _case("persist", rng.choice(timed), _log_int(rng, 2097152, 4194304), _log_int(rng, 65536, 131072),
                 rng.choice([0.9, 0.99]), 0.9, out="table")


def _ops(c, seed):
    if c["kind"] == "tpcc":
        return g.tpcc_generate(c["rows"], c["ntx"], new_order=True, seed=seed)
    return g.generate(c["rows"], c["ntx"], theta=c["theta"], read_ratio=c["read_ratio"], len_min=c["len_min"],
                      len_max=c["len_max"], seed=seed)


def _device(a):
    return torch.from_numpy(a.view(np.int64)).cuda()


def prepare(case, seed):
    c, seed = case, g.SEED ^ (int(seed) * 2654435761)
    if c["kind"] == "tpcc":
        return _prepare_tpcc(c, seed)
    w = _ops(c, seed)
    if c["kind"] == "static":
        r = np.random.default_rng(seed & 0xFFFFFFFF)
        cells = torch.randint(-(1 << 62), 1 << 62, (c["rows"] * COLS,), dtype=torch.int64, device="cuda",
                              generator=torch.Generator("cuda").manual_seed(int(r.integers(1 << 40))))
        return {"kind": "static", "scheme": c["scheme"], "rows": c["rows"], "ntx": w.ntx, "nops": w.nops,
                "batch": c["batch"], "seed": seed, "cells": cells, "ops": _device(w.ops), "off": _device(w.tx_off),
                "reads": torch.zeros(w.ntx * c["len_max"], dtype=torch.int64, device="cuda"),
                "order": torch.zeros(max(1, 2 * w.ntx), dtype=torch.int64, device="cuda")}
    persist = c["kind"] == "persist"
    table = autotune.load_table()
    if persist:
        shape = autotune.lookup(c["scheme"], c["theta"], c["read_ratio"], table)
    else:
        shape = autotune.lookup_plain(c["scheme"], c["theta"], c["read_ratio"], table)
    ctx = g.Context(c["scheme"], rows=c["rows"], cols=COLS, warp_density=shape["warp_density"],
                    block_size=shape["block_size"], batch_size=c["batch"], seed=seed,
                    persist_window=shape["window"] if persist else 0)
    ctx.seed_table()
    ctx.load_ops(w)
    return _context_state(c, ctx, COLS)


def _prepare_tpcc(c, seed):
    w = _ops(c, seed)
    cells, _ = g.tpcc_seed_tables(c["rows"], seed)
    # a new_order holds 6 to 16 ops: 16 lanes per transaction, 512-thread workgroups
    ctx = g.Context(c["scheme"], rows=g.tpcc_rows(c["rows"]), cols=g.TPCC_COLS, warp_density=4, block_size=16,
                    batch_size=c["batch"], seed=seed, tpcc=True)
    ctx.load_table(cells)
    ctx.load_ops(w)
    ctx.load_params(w.params)
    return _context_state(c, ctx, g.TPCC_COLS)


def _context_state(c, ctx, cols):
    # reads: room for the longest transactions, so that every seed's result has one shape
    n = ctx.rows * cols if c["out"] == "table" else c["ntx"] * c["len_max"]
    return {"kind": c["kind"], "ctx": ctx, "out": c["out"],
            "host": torch.zeros(n, dtype=torch.int64, pin_memory=True)}


def run(state):
    s = state
    if s["kind"] == "static":
        st = g.run_plain_static(s["scheme"], cells=s["cells"].data_ptr(), rows=s["rows"], cols=COLS,
                                ops=s["ops"].data_ptr(), tx_off=s["off"].data_ptr(), ntx=s["ntx"], nops=s["nops"],
                                reads=s["reads"].data_ptr(), order=s["order"].data_ptr(),
                                warp_density=STATIC_SHAPE[0], block_size=STATIC_SHAPE[1], batch_size=s["batch"],
                                seed=s["seed"] & 0xFFFFFFFFFFFFFFFF)
        return {"committed": st["committed"], "cells": s["cells"], "reads": s["reads"]}
    ctx = s["ctx"]
    st = ctx.run({"persist": "persistent", "graph": "graph"}.get(s["kind"], "plain"))
    to = C.c_void_p(s["host"].data_ptr())
    rc = g.load_library().gcctb_fetch(ctx._h, to if s["out"] == "table" else None,
                                      None if s["out"] == "table" else to, None, None)
    if rc != 0:
        raise RuntimeError("gcctb_fetch failed: %d" % rc)
    return {"committed": st["committed"], s["out"]: s["host"]}


def work(case):
    """Each op is read (8 B) with its share of an offset, its cell is read or
    written (8 B; in TPC-C the whole row is read and written), a read's value
    is written (8 B) and the result is read once more and written to the host."""
    c = case
    if c["kind"] == "tpcc":
        nops, reads, row = 11 * c["ntx"], 11 * c["ntx"], 2 * 8 * g.TPCC_COLS
        table = 8 * g.TPCC_COLS * 130011 * c["rows"]
    else:
        nops = c["ntx"] * (c["len_min"] + c["len_max"]) / 2
        reads, row = nops * c["read_ratio"], 8
        table = 8 * COLS * c["rows"]
    bytes_ = 8 * c["ntx"] + (8 + row) * nops + 8 * reads
    if c["kind"] != "static":
        bytes_ += 2 * (table if c["out"] == "table" else 8 * nops)
    return {"bytes": bytes_, "flops": 0}


def exact(case, seed):
    """Whole numbers and table bytes only: nothing is rounded."""
    return None
