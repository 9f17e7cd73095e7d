"""gcctb_run_plain_static on either side of the line that decides what a call
clears first: the words of the rows that its ops name (8 times fewer ops than
rows), or every word.  Calls of different table sizes follow one another on
the same static array, in one batch and in several."""
import numpy as np
import pytest

import gpu_cc_tb_amd as g
from test_zz_no_alloc import SCHEMES6, check_replay, run_static

# (rows, ntx, ops per transaction, batch)
CALLS = [(50021, 40, 16, 1 << 30), (4096, 512, 1, 100), (4096, 511, 1, 100), (20000, 300, 8, 128), (3001, 900, 6, 1 << 30),
         (50021, 1, 1, 1)]


@pytest.mark.gpu
@pytest.mark.parametrize("scheme", SCHEMES6)
def test_static_call_sequence(scheme):
    for i, (rows, ntx, length, batch) in enumerate(CALLS):
        print(f"[static-calls] scheme={scheme} call={i} rows={rows} ntx={ntx}x{length} batch={batch}", flush=True)
        w = g.generate(rows, ntx, theta=0.6, read_ratio=0.5, len_min=length, seed=g.SEED + i)
        st, res = run_static(scheme, rows, w, batch, 3, 8)
        assert st["committed"] == ntx and st["error_flags"] == 0
        assert st["batches"] == (ntx + batch - 1) // batch
        check_replay(rows, w, res, f"call {i}")


@pytest.mark.gpu
def test_static_error_then_clean(monkeypatch):
    """A watchdog of 20 us (the kernels' own bounded wait) may stop the first
    batch: nothing after it runs, and the next call finds clean words."""
    w = g.generate(64, 2048, theta=0.99, read_ratio=0.5, len_min=8)
    monkeypatch.setenv("GCCTB_WATCHDOG_S", "0.00002")
    print("[static-calls] watchdog", flush=True)
    with pytest.raises(g.GcctbError) as e:
        for _ in range(5):
            run_static("tpl_nw", 64, w, 256, 3, 8)
    assert e.value.code == -6
    monkeypatch.delenv("GCCTB_WATCHDOG_S")
    st, res = run_static("tpl_nw", 64, w, 256, 3, 8)
    assert st["committed"] == 2048
    check_replay(64, w, res, "after a stopped call")
