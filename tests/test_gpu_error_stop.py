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
@pytest.mark.parametrize("launch_no,failed", [(1, 0), (2, 0), (2, 1), (7, 3)])
def test_tpcc_combiner_after_an_error(combine, launch_no, failed):
    """TPC-C under GaccO applies a batch's queues before its launch: not once an
    earlier launch has reported an error."""
    lens = np.array([70, 3], dtype=np.uint32)
    nops, rows = int(lens.sum()), 4
    rng = np.random.default_rng(launch_no * 10 + failed)
    w = g.tpcc_generate(1, nops, new_order=False, seed=3)
    first = w.tx_off[:-1].astype(np.int64)  # each payment's warehouse update
    ops, params = np.ascontiguousarray(w.ops[first]), np.ascontiguousarray(w.params[first])
    srow = np.repeat(np.array([1, 3], dtype=np.uint32), lens)
    sop = np.arange(nops, dtype=np.uint32) | np.uint32(1 << 31)
    cells = rng.integers(0, 1 << 30, rows * 5).astype(np.uint64)
    reads, need = np.full(nops, 7, dtype=np.uint64), np.full(nops, 5, dtype=np.uint32)
    out_c, out_r, out_n = cells.copy(), reads.copy(), need.copy()
    ptr = lambda a: a.ctypes.data_as(C.c_void_p)  # noqa: E731
    print(f"[error-stop] combiner launch={launch_no} failed={failed}", flush=True)
    rc = combine(C.c_uint32(2), ptr(lens), ptr(srow), ptr(sop), C.c_uint32(nops), ptr(ops), ptr(params), C.c_uint64(rows),
                 ptr(out_c), ptr(out_r), ptr(out_n), C.c_uint32(launch_no), C.c_uint64(failed))
    assert rc == 0
    if not failed:
        for i in range(nops):
            row = cells[5 * int(srow[i]):5 * int(srow[i]) + 5]
            reads[i] = orc.lib().orc_tpcc_apply(int(g.op_col(ops[i:i + 1])[0]), int(params[i]), row)
        need[:] = 0xFFFFFFFF
    assert np.array_equal(out_c, cells) and np.array_equal(out_r, reads) and np.array_equal(out_n, need)
