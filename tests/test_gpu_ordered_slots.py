"""GaccO and GPUTx at every number of op slots per lane (32 to 1), on few rows,
so that the slots of one lane, of several accesses at a time, wait for
different turns."""
import numpy as np
import pytest

import gpu_cc_tb_amd as g
import oracle_lib as orc

ROWS, NTX = 97, 700


def _stream(wd):
    return g.generate(ROWS, NTX, theta=0.7, read_ratio=0.5, len_min=1, len_max=32, seed=g.SEED + wd)


@pytest.mark.gpu
@pytest.mark.parametrize("wd", range(6))
@pytest.mark.parametrize("scheme,form", [("gacco", "plain"), ("gacco", "persistent"), ("gputx", "plain"), ("gputx", "persistent")])
def test_ordered_slots(scheme, form, wd, monkeypatch):
    monkeypatch.setenv("GCCTB_COMBINE_MIN", "0")  # every access takes its turn
    w = _stream(wd)
    print(f"[ordered-slots] scheme={scheme} form={form} wd={wd}", flush=True)
    with g.Context(scheme, rows=ROWS, warp_density=wd, block_size=4, batch_size=300, persist_window=256) as ctx:
        ctx.seed_table()
        ctx.load_ops(w)
        st = ctx.run(form)
        res = ctx.fetch()
    assert st["committed"] == NTX and st["error_flags"] == 0
    init = orc.seed_table(g.SEED, ROWS, 10)
    exp_t, exp_r, ties = orc.replay(ROWS, 10, g.SEED, init, w.ops, w.tx_off, res["order"])
    isr = ~g.op_is_write(w.ops)
    assert ties == 0 and np.array_equal(res["table"], exp_t) and np.array_equal(res["reads"][isr], exp_r[isr])
    if scheme == "gacco":
        t2, r2 = orc.replay_txid(ROWS, 10, g.SEED, init, w.ops, w.tx_off)
        assert np.array_equal(res["table"], t2) and np.array_equal(res["reads"][isr], r2[isr])


@pytest.mark.gpu
@pytest.mark.parametrize("wd", range(6))
def test_ordered_event_stamps(wd):
    """An access is stamped before its turn passes on: every row's stamps of
    accesses that conflict follow the transactions' order."""
    w = _stream(wd)
    print(f"[ordered-events] wd={wd}", flush=True)
    with g.Context("gacco", rows=ROWS, warp_density=wd, block_size=4, debug_events=True) as ctx:
        ctx.seed_table()
        ctx.load_ops(w)
        ctx.run("plain")
        ev = ctx.fetch_events()
    chk = g.conflict_check(ev, NTX)
    assert chk["uncommitted"] == 0 and chk["cycle"] == []
    acc = ev[ev["type"] != 2]
    assert len(acc) == w.nops
    for row in range(ROWS):
        e = np.sort(acc[acc["oid"] == row], order="id")
        for i in np.flatnonzero(e["type"] == 1):  # a write comes after every lower transaction and before every higher
            assert np.all(e["tid"][:i] < e["tid"][i]) and np.all(e["tid"][i + 1:] > e["tid"][i])
