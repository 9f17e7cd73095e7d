"""What a run does after a launch that reports an error.  The error is the
kernels' own bounded wait (GCCTB_WATCHDOG_S, set from the host): every kernel
ends by itself."""
import numpy as np
import pytest

import gpu_cc_tb_amd as g
import oracle_lib as orc


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
