"""The end of a contended launch, where resting waves look up how many groups
are left: the smallest launches (one group, one half wave), groups that do not
fill a wave or a block, several batches and several runs of one context."""
import numpy as np
import pytest

import gpu_cc_tb_amd as g
import oracle_lib as orc

SHAPES = [(0, 1), (1, 3), (3, 8), (5, 1), (5, 2)]  # (warp_density, block_size)


@pytest.mark.gpu
@pytest.mark.parametrize("scheme", ["tpl_nw", "tpl_wd", "to", "mvcc", "silo", "tictoc"])
@pytest.mark.parametrize("form", ["plain", "persistent", "graph"])
def test_contended_launch_ends(scheme, form):
    rows = 300
    init = orc.seed_table(g.SEED, rows, 10)
    for ntx, batch in [(1, 1 << 20), (33, 1 << 20), (1501, 700)]:
        w = g.generate(rows, ntx, theta=0.9, read_ratio=0.5, len_min=8, seed=g.SEED + ntx)
        isr = ~g.op_is_write(w.ops)
        for wd, bs in SHAPES:
            print(f"[launch-end] scheme={scheme} form={form} ntx={ntx} shape={wd},{bs}", flush=True)
            with g.Context(scheme, rows=rows, warp_density=wd, block_size=bs, batch_size=batch,
                           persist_window=256 if form == "persistent" else 0) as ctx:
                ctx.load_ops(w)
                for _ in range(2):
                    ctx.seed_table()
                    st = ctx.run(form)
                    res = ctx.fetch()
                    assert st["committed"] == ntx and st["error_flags"] == 0
                    table, reads, ties = orc.replay(rows, 10, g.SEED, init, w.ops, w.tx_off, res["order"])
                    assert ties == 0 and np.array_equal(res["table"], table)
                    assert np.array_equal(res["reads"][isr], reads[isr])
