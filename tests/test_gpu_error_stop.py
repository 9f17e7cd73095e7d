"""What a run does after a launch that reports an error.  The error is the
kernels' own bounded wait (GCCTB_WATCHDOG_S, set from the host): every kernel
ends by itself."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

import gpu_cc_tb_amd as g
import oracle_lib as orc
from test_zz_no_alloc import COLS, SCHEMES6, run_static

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["plain", "graph"])
def test_failing_launch_runs_whole(form, monkeypatch):
    """An error stops the launches behind its own, never its own: with a wait
    of 10 ns, 64 transactions that queue on one row end after the first of
    them, and the 65,536 free ones of the same launch, most of which start
    after the error, all commit."""
    monkeypatch.setenv("GCCTB_WATCHDOG_S", "0.00000001")
    first, chain, free = 100, 64, 65536
    ntx = first + chain + free
    keys = np.arange(ntx, dtype=np.uint64)
    keys[first:first + chain] = first
    w = g.Ops(g.make_ops(keys, np.zeros(ntx), np.ones(ntx, dtype=bool)), np.arange(ntx + 1, dtype=np.uint64))
    print(f"[error-stop] own launch form={form}", flush=True)
    with g.Context("gacco", rows=ntx, warp_density=5, block_size=4) as ctx:
        ctx.seed_table()
        ctx.load_ops(w)
        ctx.set_batches([first, chain + free])
        st = ctx.run(form, check=False)
        table = ctx.fetch()["table"].reshape(ntx, 10)
    assert st["rc"] == -6 and st["error_flags"] == 16
    assert st["committed"] == first + 1 + free
    changed = np.any(table != orc.seed_table(g.SEED, ntx, 10).reshape(ntx, 10), axis=1)
    assert np.all(changed[:first + 1]) and not np.any(changed[first + 1:first + chain])
    assert np.all(changed[first + chain:])


@pytest.fixture(scope="module")
def combine(tmp_path_factory):
    """launch::tpcc_combine of the built library (combine_shim.cpp)."""
    g.load_library()
    so = str(tmp_path_factory.mktemp("shim") / "combine_shim.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    os.path.join(ROOT, "tests/combine_shim.cpp"), "-o", so, f"-L{ROOT}/gpu_cc_tb_amd", "-lgcctb",
                    f"-Wl,-rpath,{ROOT}/gpu_cc_tb_amd", "-L/opt/rocm/lib", "-lamdhip64"], check=True)
    return C.CDLL(so).combine_queues


@pytest.mark.gpu
@pytest.mark.parametrize("error", [0, 16, (3 << 32) | 16])
def test_tpcc_combiner_after_an_error(combine, error):
    """TPC-C under GaccO applies a batch's queues before its launch: not once an
    earlier launch has reported an error."""
    lens = np.array([70, 1, 3])
    nops, rows = int(lens.sum()), 4
    rng = np.random.default_rng(5)
    w = g.tpcc_generate(1, nops, new_order=False, seed=3)
    first = w.tx_off[:-1].astype(np.int64)  # each payment's warehouse update
    ops, params = np.ascontiguousarray(w.ops[first]), np.ascontiguousarray(w.params[first])
    srow = np.repeat(np.array([0, 1, 3], dtype=np.uint32), lens)
    sop = np.arange(nops, dtype=np.uint32) | np.uint32(1 << 31)
    cells = rng.integers(0, 1 << 30, rows * 5).astype(np.uint64)
    reads, need = np.full(nops, 7, dtype=np.uint64), np.full(nops, 1 << 31, dtype=np.uint32)
    out_c, out_r, out_n, listed = cells.copy(), reads.copy(), need.copy(), C.c_uint32(9)
    ptr = lambda a: a.ctypes.data_as(C.c_void_p)  # noqa: E731
    print(f"[error-stop] combiner error={error}", flush=True)
    rc = combine(ptr(srow), ptr(sop), C.c_uint32(nops), ptr(ops), ptr(params), C.c_uint64(rows), ptr(out_c), ptr(out_r),
                 ptr(out_n), C.c_uint64(error), C.byref(listed))
    assert rc == 0 and listed.value == (0 if error else 2)
    for i in np.flatnonzero(srow != 1):
        if error:  # the queues keep their turns
            at = i if srow[i] == 0 else i - 71
            need[i] = at | (1 << 31 if at == lens[srow[i] if srow[i] == 0 else 2] - 1 else 0)
        else:
            row = cells[5 * int(srow[i]):5 * int(srow[i]) + 5]
            reads[i] = orc.lib().orc_tpcc_apply(int(g.op_col(ops[i:i + 1])[0]), int(params[i]), row)
            need[i] = 0xFFFFFFFF
    assert np.array_equal(out_c, cells) and np.array_equal(out_r, reads) and np.array_equal(out_n, need)


def _hot_first_batch(rows, n, later):
    """One write each: n transactions on row 0, then 3 x later, each on a row of its own."""
    keys = np.concatenate([np.zeros(n, dtype=np.uint64), 1 + np.arange(3 * later, dtype=np.uint64)])
    return g.Ops(g.make_ops(keys, np.full(keys.size, 2), np.ones(keys.size, dtype=bool)),
                 np.arange(keys.size + 1, dtype=np.uint64))


HOT, LATER = 4096, 512  # 4,096 commits on one row, at least a memory latency each, outlast a wait of 50 us


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["plain", "graph"])
@pytest.mark.parametrize("scheme", ["tpl_nw", "tpl_wd", "to", "mvcc", "silo", "tictoc", "gacco"])
def test_batches_behind_an_error(scheme, form, monkeypatch):
    """The first of four batches runs into its bounded wait: the three behind
    it write nothing, commit nothing and are not counted, and once the wait is
    long enough the next context commits them all."""
    rows = 1 + 3 * LATER
    w = _hot_first_batch(rows, HOT, LATER)
    init = orc.seed_table(g.SEED, rows, 10).reshape(rows, 10)
    for wait in ("0.00005", None):
        if wait:
            monkeypatch.setenv("GCCTB_WATCHDOG_S", wait)
        else:
            monkeypatch.delenv("GCCTB_WATCHDOG_S")
        print(f"[error-stop] scheme={scheme} form={form} wait={wait}", flush=True)
        with g.Context(scheme, rows=rows, warp_density=3, block_size=8) as ctx:
            ctx.seed_table()
            ctx.load_ops(w)
            ctx.set_batches([HOT, LATER, LATER, LATER])
            st = ctx.run(form, check=False)
            table = ctx.fetch()["table"].reshape(rows, 10)
            changed = np.any(table != init, axis=1)[1:]
            if wait:
                assert st["rc"] == -6 and st["error_flags"] & 16
                assert st["batches"] == 1 and st["committed"] < HOT
                assert not np.any(changed), "a batch behind the error ran"
                assert not np.any(ctx.fetch_cc())
            else:
                assert st["rc"] == 0 and st["batches"] == 4 and st["committed"] == w.ntx and np.all(changed)


@pytest.mark.gpu
@pytest.mark.parametrize("scheme", SCHEMES6)
def test_static_batches_behind_an_error(scheme, monkeypatch):
    """The same through gcctb_run_plain_static, whose calls share their words:
    the batches behind the error leave the table alone, and the call
    after it runs whole."""
    rows = 1 + 3 * LATER
    w = _hot_first_batch(rows, HOT, LATER)
    init = orc.seed_table(g.SEED, rows, COLS).reshape(rows, COLS)
    call = g.run_plain_static
    monkeypatch.setattr(g, "run_plain_static", lambda *a, **k: call(*a, **k, check=False))
    for wait in ("0.00005", None):
        if wait:
            monkeypatch.setenv("GCCTB_WATCHDOG_S", wait)
        else:
            monkeypatch.delenv("GCCTB_WATCHDOG_S")
        print(f"[error-stop] static scheme={scheme} wait={wait}", flush=True)
        st, res = run_static(scheme, rows, w, HOT, 3, 8)
        changed = np.any(res["table"].reshape(rows, COLS) != init, axis=1)[1:]
        if wait:
            assert st["rc"] == -6 and st["error_flags"] & 16 and st["batches"] == 1 and st["committed"] < HOT
            assert not np.any(changed)
        else:
            assert st["rc"] == 0 and st["batches"] == 2 and st["committed"] == w.ntx and np.all(changed)
