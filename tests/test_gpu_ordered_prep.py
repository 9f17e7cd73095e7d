"""The preparation kernels of GaccO and GPUTx at the sizes where they change
course: tile edges, the switch between tile sizes, rows that span tiles."""
import numpy as np
import pytest

import gpu_cc_tb_amd as g
import oracle_lib as orc

SHORT_MAX = 1 << 20  # pairs up to which the sort uses its short tile (1,024)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1023, 1025, SHORT_MAX, SHORT_MAX + 1])
@pytest.mark.parametrize("dtype,bits", [(np.uint32, 17), (np.uint64, 33)])
def test_sort_tile_sizes(n, dtype, bits):
    """Either tile size, with key bits that split unevenly over the passes."""
    rng = np.random.default_rng(n + bits)
    keys = rng.integers(0, np.iinfo(dtype).max, n, dtype=dtype, endpoint=True)
    vals = np.arange(n, dtype=np.uint32)
    print(f"[sort-tiles] n={n} bits={bits}", flush=True)
    k, v, _ = g.sort_pairs(keys, vals, key_bits=bits)
    order = np.argsort(keys & dtype((1 << bits) - 1), kind="stable")
    assert np.array_equal(v, order.astype(np.uint32)) and np.array_equal(k, keys[order])


OWN_SCAN_COUNTS = 24 * 4 * 256  # counts (tiles x digits) that a scatter block adds up itself


@pytest.mark.gpu
@pytest.mark.parametrize("n", [2, 1024, 5121] + [OWN_SCAN_COUNTS // d * 1024 + e for d in (256, 128, 32) for e in (0, 1)])
@pytest.mark.parametrize("dtype,bits", [(np.uint32, 4), (np.uint32, 5), (np.uint32, 21), (np.uint32, 32), (np.uint64, 41)])
def test_sort_without_scan_launch(n, dtype, bits):
    """One tile, a few, and as many as digits of 8, 7 and 5 bits allow and one
    more; digits of 4 to 8 bits: the stable sort."""
    rng = np.random.default_rng(n * 64 + bits)
    keys = rng.integers(0, np.iinfo(dtype).max, n, dtype=dtype, endpoint=True)
    keys[: n // 3] = keys[0]  # one digit with a long run
    vals = np.arange(n, dtype=np.uint32)
    print(f"[sort-own-scan] n={n} bits={bits}", flush=True)
    k, v, _ = g.sort_pairs(keys, vals, key_bits=bits)
    order = np.argsort(keys & dtype((1 << bits) - 1), kind="stable")
    assert np.array_equal(v, order.astype(np.uint32)) and np.array_equal(k, keys[order])


def _one_row_stream(ntx, writes, rows, seed):
    """ntx transactions of 2 ops: row 0, read or (at the given transactions)
    written, and a row of their own, so one queue runs through the sorted
    accesses and every other row is met once."""
    rng = np.random.default_rng(seed)
    keys = np.zeros((ntx, 2), dtype=np.uint64)
    keys[:, 1] = 1 + rng.permutation(rows - 1)[:ntx]
    wr = np.zeros((ntx, 2), dtype=np.uint64)
    wr[writes, 0] = 1
    wr[:, 1] = rng.integers(0, 2, ntx)
    ops = g.make_ops(keys.reshape(-1), rng.integers(0, 10, 2 * ntx), wr.reshape(-1))
    return g.Ops(ops, np.arange(ntx + 1, dtype=np.uint64) * np.uint64(2))


TURN_TILE = 2048  # accesses per tile of the turn kernels; carries look back 64 tiles a step
TURN_SHORT = 512  # up to SHORT_MAX accesses
TURN_CASES = {
    # name: (ntx, transactions that write row 0)
    "no_writes": (TURN_TILE, []),
    "tile_edges": (2 * TURN_TILE + 1, [TURN_TILE - 1, TURN_TILE, 2 * TURN_TILE]),
    "first_and_last": (TURN_TILE + 7, [0, TURN_TILE + 6]),
    "past_64_tiles": (66 * TURN_TILE + 5, [0, 3, 66 * TURN_TILE + 1]),
    "short_tile_edges": (2 * TURN_SHORT + 1, [TURN_SHORT - 1, TURN_SHORT, 2 * TURN_SHORT]),
    "longest_short": (SHORT_MAX // 2, [0, 3, SHORT_MAX // 2 - 1]),
    "shortest_long": (SHORT_MAX // 2 + 1, [0, 3, TURN_TILE, SHORT_MAX // 2]),
}


@pytest.mark.gpu
@pytest.mark.parametrize("case", list(TURN_CASES))
@pytest.mark.parametrize("scheme", ["gacco", "gputx"])
@pytest.mark.parametrize("form", ["plain", "persistent"])
def test_turns_of_a_long_queue(scheme, case, form, monkeypatch):
    """One row's queue across tile edges and beyond one look-back step, turn
    by turn (no combiner): the serial replay in the reported order."""
    monkeypatch.setenv("GCCTB_COMBINE_MIN", "0")
    ntx, writes = TURN_CASES[case]
    rows = ntx + 1
    w = _one_row_stream(ntx, writes, rows, ntx)
    print(f"[turns] scheme={scheme} case={case} form={form}", flush=True)
    with g.Context(scheme, rows=rows, warp_density=1, block_size=8, batch_size=1 << 20) as ctx:
        ctx.seed_table()
        ctx.load_ops(w)
        st = ctx.run(form)
        res = ctx.fetch()
        rank = ctx.fetch_ranks()[0] if scheme == "gputx" else None
    assert st["committed"] == ntx and st["error_flags"] == 0
    init = orc.seed_table(g.SEED, rows, 10)
    exp_t, exp_r, ties = orc.replay(rows, 10, g.SEED, init, w.ops, w.tx_off, res["order"])
    isr = ~g.op_is_write(w.ops)
    assert ties == 0 and np.array_equal(res["table"], exp_t) and np.array_equal(res["reads"][isr], exp_r[isr])
    if scheme == "gacco":
        t2, r2 = orc.replay_txid(rows, 10, g.SEED, init, w.ops, w.tx_off)
        assert np.array_equal(res["table"], t2) and np.array_equal(res["reads"][isr], r2[isr])
    else:
        # group starts of row 0's queue up to each transaction
        wr = np.zeros(ntx, dtype=bool)
        wr[writes] = True
        start = np.zeros(ntx, dtype=np.int64)
        start[1:] = wr[1:] | wr[:-1]
        assert np.array_equal(rank, np.cumsum(start).astype(np.uint32))


# (warp_density, block_size, window, ntx): blocks of 64, 64, 1 and 16 groups;
# streams of one slot past a block, many chunks, and none to stash
STASH_CASES = [(2, 8, 64, 65), (2, 8, 128, 2001), (5, 1, 4, 33), (4, 8, 32, 32), (4, 8, 32, 515)]


@pytest.mark.gpu
@pytest.mark.parametrize("wd,bs,window,ntx", STASH_CASES)
@pytest.mark.parametrize("scheme", ["gacco", "gputx"])
def test_slot_stash(scheme, wd, bs, window, ntx):
    """Blocks that draw their slots in chunks run every transaction once, in
    an order that the waits on lower slots allow, down to the stream's end."""
    rows = 256
    w = g.generate(rows, ntx, theta=0.8, read_ratio=0.5, len_min=1, len_max=8)
    print(f"[stash] scheme={scheme} wd={wd} bs={bs} window={window} ntx={ntx}", flush=True)
    with g.Context(scheme, rows=rows, warp_density=wd, block_size=bs, batch_size=1 << 20,
                   persist_window=window) as ctx:
        ctx.seed_table()
        ctx.load_ops(w)
        st = ctx.run("persistent")
        res = ctx.fetch()
    assert st["committed"] == ntx and st["error_flags"] == 0
    exp_t, exp_r, ties = orc.replay(rows, 10, g.SEED, orc.seed_table(g.SEED, rows, 10), w.ops, w.tx_off, res["order"])
    isr = ~g.op_is_write(w.ops)
    assert ties == 0 and np.array_equal(res["table"], exp_t) and np.array_equal(res["reads"][isr], exp_r[isr])


COMB_CHUNK = 256  # accesses per combiner chunk; the carry splits a queue's chunks over 16 waves


@pytest.mark.gpu
@pytest.mark.parametrize("length", [128, COMB_CHUNK, COMB_CHUNK + 1, 16 * COMB_CHUNK, 40 * COMB_CHUNK + 3])
@pytest.mark.parametrize("cols,write_share", [(3, 0.5), (64, 0.02), (10, 0.0)])
def test_combiner_chunks(length, cols, write_share):
    """Two queues of the same length at chunk edges, beside short ones, run by
    combiners: the serial run in transaction-id order."""
    rng = np.random.default_rng(length * 100 + cols)
    rows = 3 + length
    keys = np.stack([np.full(length, 1), np.full(length, 2), 3 + rng.permutation(length)], axis=1)
    ops = g.make_ops(keys.reshape(-1), rng.integers(0, cols, 3 * length), rng.random(3 * length) < write_share)
    w = g.Ops(ops, np.arange(length + 1, dtype=np.uint64) * np.uint64(3))
    print(f"[comb-chunks] length={length} cols={cols} writes={write_share}", flush=True)
    with g.Context("gacco", rows=rows, cols=cols, warp_density=2, block_size=8, batch_size=1 << 20) as ctx:
        ctx.seed_table()
        ctx.load_ops(w)
        st = ctx.run("persistent")
        res = ctx.fetch()
    assert st["committed"] == length and st["combined"] == 2 * length
    t2, r2 = orc.replay_txid(rows, cols, g.SEED, orc.seed_table(g.SEED, rows, cols), w.ops, w.tx_off)
    isr = ~g.op_is_write(w.ops)
    assert np.array_equal(res["table"], t2) and np.array_equal(res["reads"][isr], r2[isr])


FILTER_MIN = 1 << 20  # ops from which only the accesses of written rows are sorted


@pytest.mark.gpu
@pytest.mark.parametrize("scheme,form", [("gputx", "persistent"), ("gputx", "plain"), ("gacco", "plain")])
@pytest.mark.parametrize("read_ratio,missing", [(0.97, False), (0.97, True), (1.0, False)])
def test_written_rows_filter(scheme, form, read_ratio, missing):
    """Just past the size where only written rows' accesses are sorted, over a
    dense index and over one that lacks keys, and with no write at all: the
    serial replay, and for GPUTx the oracle's ranks."""
    rows, ntx = 262147, FILTER_MIN // 16 + 3
    w = g.generate(rows, ntx, theta=0.3, read_ratio=read_ratio)
    print(f"[filter] scheme={scheme} form={form} reads={read_ratio} missing={missing}", flush=True)
    with g.Context(scheme, rows=rows, warp_density=3, block_size=8, batch_size=1 << 20) as ctx:
        ctx.seed_table()
        if missing:
            keys = np.arange(rows, dtype=np.uint32)
            present = keys[keys % 9 != 4]
            ctx.build_index(present, present)
        ctx.load_ops(w)
        st = ctx.run(form, check=False)
        res = ctx.fetch()
        ranks = ctx.fetch_ranks()[0] if scheme == "gputx" else None
    hit = np.ones(w.nops, dtype=bool) if not missing else g.op_key(w.ops) % 9 != 4
    assert st["committed"] == ntx and st["index_miss"] == int(np.count_nonzero(~hit))
    # the ops that hit, as transactions of their own: what the run must equal
    off = np.concatenate([[0], np.cumsum(hit)])[w.tx_off.astype(np.int64)].astype(np.uint64)
    if missing:
        # written values depend on the op's place in its transaction, so only reads of unwritten cells are compared
        cell = g.op_key(w.ops).astype(np.int64) * 10 + g.op_col(w.ops)
        isw = g.op_is_write(w.ops)
        calm = hit & ~isw & ~np.isin(cell, np.unique(cell[isw & hit]))
        init = orc.seed_table(g.SEED, rows, 10)
        assert np.array_equal(res["reads"][calm], init[cell[calm]])
        touched = np.zeros(rows * 10, dtype=bool)
        touched[cell[isw & hit]] = True
        assert np.array_equal(res["table"][~touched], init[~touched])
        assert not np.any(res["table"][touched] == init[touched])
    else:
        init = orc.seed_table(g.SEED, rows, 10)
        exp_t, exp_r, ties = orc.replay(rows, 10, g.SEED, init, w.ops, w.tx_off, res["order"])
        isr = ~g.op_is_write(w.ops)
        assert ties == 0 and np.array_equal(res["table"], exp_t) and np.array_equal(res["reads"][isr], exp_r[isr])
    if ranks is not None:
        part = g.Ops(w.ops[hit], off)
        assert np.array_equal(ranks, orc.gputx_rank(rows, part.ops, part.tx_off)[0])


@pytest.mark.gpu
@pytest.mark.parametrize("ntx", [1, 2, 63, 64, 65, 200])
@pytest.mark.parametrize("new_order", [True, False])
@pytest.mark.parametrize("form", ["plain", "graph"])
def test_tpcc_queues(ntx, new_order, form):
    """TPC-C queues around a wave's 64 updates (one warehouse), run twice with
    the table carried on, the second time in batches: the oracle's replay."""
    w = g.tpcc_generate(1, ntx, new_order=new_order, seed=ntx)
    cells, _ = g.tpcc_seed_tables(1)
    print(f"[tpcc-queues] ntx={ntx} new_order={new_order} form={form}", flush=True)
    with g.Context("gacco", rows=g.tpcc_rows(1), cols=5, warp_density=4, block_size=4, batch_size=70,
                   tpcc=True) as ctx:
        ctx.load_table(cells)
        ctx.load_ops(w)
        ctx.load_params(w.params)
        for _ in range(2):
            ctx.run(form)
            res = ctx.fetch()
            assert g.tpcc_check(1, cells, res["table"], w, res["order"], res["reads"]) == 0
            exp_t, exp_r = orc.tpcc_replay(g.tpcc_rows(1), cells, w.ops, w.params, w.tx_off, res["order"])[:2]
            assert np.array_equal(res["table"], exp_t) and np.array_equal(res["reads"], exp_r)
            cells = res["table"]
