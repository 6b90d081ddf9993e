"""The grouped matmul that decodes its rows in registers (kernels/moe_cols.h) at the edges of its tiles: experts of 0, 1, 31,
33, 64, 65 and 129 columns, rows of one tile less, exactly and more, one super-block of K, an odd and an even number of
them; GGUF rows and packed planes, one bank and two, gathered rows, a gated activation; against the oracle in f64."""
import numpy as np
import pytest

import oracle
from conftest import nmse
from jitllm_amd import quant, synth

pytestmark = pytest.mark.gpu
FILL = np.float32(4e30)
COUNTS = [1, 0, 31, 33, 64, 65, 129, 0]


@pytest.mark.parametrize("t,layout", [(quant.Q4_K, "rows"), (quant.Q4_K, "one"), (quant.Q4_K, "sheets"), (quant.Q6_K, "rows")],
                         ids=["q4_k", "q4_k-planes", "q4_k-sheets", "q6_k"])
@pytest.mark.parametrize("nrows,k", [(1, 256), (130, 512), (96, 768), (257, 1024)])
def test_columns_against_decoded_rows(dev, devbuf, t, layout, nrows, k):
    from test_gpu_moe import _pack_bank
    n_expert, ncols = len(COUNTS), sum(COUNTS)
    start = np.concatenate([[0], np.cumsum(COUNTS)]).astype(np.uint32)
    dev.SetActWindow(256)
    sheet = nrows * quant.row_bytes(t, k)
    banks = [np.concatenate([synth.random_weights(t, nrows, k, seed=10 * b + e) for e in range(n_expert)]) for b in range(2)]
    x = np.stack([synth.activations(k, seed=300 + r) * np.float32(1 + r % 3) for r in range(40)])
    u = np.stack([synth.activations(k, seed=500 + r) for r in range(40)])
    src = (np.arange(ncols) * 7 % 40).astype(np.uint32)
    xg = (x / (1 + np.exp(-x.astype(np.float64))) * u).astype(np.float32)
    xd, ud, sd, dstart = devbuf(x), devbuf(u), devbuf(src), devbuf(start)
    hold = [_pack_bank(dev, devbuf, t, b, n_expert, nrows, k, layout) if layout != "rows" else (devbuf(b), None) for b in banks]
    try:
        dev.set_tuning(moe__form=9)
        for gated in (False, True):
            act = xg if gated else x
            o = [devbuf(shape=(ncols * nrows + 8,), dtype=np.float32, fill=FILL) for _ in banks]
            args = (xd.ptr, ud.ptr if gated else None, sd.ptr, dstart.ptr, n_expert, ncols, nrows, k)
            if layout == "rows":
                assert dev.moe_matvec_dev(o[0].ptr, o[1].ptr, t, hold[0][0].ptr, hold[1][0].ptr, *args)
            else:
                assert dev.moe_matvec_packed_dev(o[0].ptr, o[1].ptr, t, hold[0][0], hold[1][0], *args)
            dev.synchronize()
            for b in range(2):
                want = np.zeros((ncols, nrows))
                for e in range(n_expert):
                    cols = slice(start[e], start[e + 1])
                    if COUNTS[e]:
                        want[cols] = oracle.matmul_q8act_f64(t, banks[b][e * sheet:(e + 1) * sheet], act[src[cols]], nrows, k, COUNTS[e], 256)
                got = o[b].get()
                assert np.all(got[ncols * nrows:] == FILL)
                # (the gated activation: an exponential of another machine in front of the quantizer)
                assert nmse(got[:ncols * nrows].reshape(ncols, nrows), want) <= (1e-6 if gated else 1e-10), (gated, b)
    finally:
        dev.set_tuning(moe__form=0)
        dev.SetActWindow(32)


@pytest.mark.parametrize("down", [quant.Q4_K, quant.Q6_K], ids=["q4_k", "q6_k"])
def test_block_with_source_rows_quantized_once(dev, devbuf, down):
    """The routed block, where a source row's record serves all of its columns: the bits of a record a column."""
    rows, k_used, n_expert, n_ffn, n_embd = 75, 3, 6, 512, 768
    rng = np.random.default_rng(5)
    sel = np.stack([rng.permutation(n_expert)[:k_used] for _ in range(rows)]).astype(np.uint32)
    perm = np.argsort(sel.reshape(-1), kind="stable")
    start = np.concatenate([[0], np.cumsum(np.bincount(sel.reshape(-1), minlength=n_expert))]).astype(np.uint32)
    ncols = rows * k_used
    dev.SetActWindow(256)
    bank = lambda t, nrows, k, s: devbuf(np.concatenate([synth.random_weights(t, nrows, k, seed=s + e) for e in range(n_expert)]))
    gate, up, dn = bank(quant.Q4_K, n_ffn, n_embd, 0), bank(quant.Q4_K, n_ffn, n_embd, 50), bank(down, n_embd, n_ffn, 90)
    x = np.stack([synth.activations(n_embd, seed=700 + r) for r in range(rows)])
    wt = np.full((rows, k_used), 1 / k_used, np.float32)
    xd, sd, wd, start_d = devbuf(x), devbuf(sel), devbuf(wt), devbuf(start)
    perm_d, pos_d = devbuf((perm // k_used).astype(np.uint32)), devbuf(np.argsort(perm, kind="stable").astype(np.uint32))
    try:
        dev.set_tuning(moe__form=9)
        r = devbuf(np.zeros((rows, n_embd), np.float32))
        assert dev.moe_ffn_dev(r.ptr, quant.Q4_K, gate.ptr, up.ptr, dn.ptr, xd.ptr, sd.ptr, k_used, wd.ptr, rows, k_used, n_expert, n_ffn,
                               n_embd, down_type=down)
        g, u, y = (devbuf(shape=(ncols, n), dtype=np.float32) for n in (n_ffn, n_ffn, n_embd))
        want = devbuf(np.zeros((rows, n_embd), np.float32))
        assert dev.moe_matvec_dev(g.ptr, u.ptr, quant.Q4_K, gate.ptr, up.ptr, xd.ptr, None, perm_d.ptr, start_d.ptr, n_expert, ncols, n_ffn, n_embd)
        assert dev.moe_matvec_dev(y.ptr, None, down, dn.ptr, None, g.ptr, u.ptr, None, start_d.ptr, n_expert, ncols, n_embd, n_ffn)
        assert dev.moe_combine_dev(want.ptr, y.ptr, wd.ptr, sd.ptr, k_used, pos_d.ptr, rows, k_used, n_embd)
        dev.synchronize()
        assert np.array_equal(r.get().view(np.uint32), want.get().view(np.uint32))
    finally:
        dev.set_tuning(moe__form=0)
        dev.SetActWindow(32)


@pytest.mark.parametrize("t,window", [(quant.Q4_K, 256), (quant.Q6_K, 256), (quant.Q8_0, 32), (quant.Q6_K, 32)], ids=["q4_k", "q6_k", "q8_0", "q6_k-w32"])
@pytest.mark.parametrize("nrows,k", [(1, 256), (17, 512), (300, 768), (2901, 512), (2901, 1024), (2901, 2048), (2100, 4352)])
def test_a_matvec_a_column(dev, devbuf, t, window, nrows, k):
    """A handful of routed columns, a decode matvec each: experts of none, one and several columns (the first and the last
    expert among them), more than 64 experts, one row group and several a workgroup, eight, sixteen and thirty-two lanes a row
    with a last step that is ragged, K past a workgroup's first round of activations; two banks, gathered rows, a gated activation."""
    if nrows * k > 7e6 and t == quant.Q6_K and window == 32:
        pytest.skip("the largest shape runs once a type")
    counts = np.zeros(70 if nrows < 2000 else 5, int)
    counts[[0, 3, -1]] = 2, 3, 1
    n_expert, ncols = len(counts), int(counts.sum())
    start = np.concatenate([[0], np.cumsum(counts)]).astype(np.uint32)
    dev.SetActWindow(window)
    sheet = nrows * quant.row_bytes(t, k)
    banks = [np.concatenate([synth.random_weights(t, nrows, k, seed=20 * b + e) for e in range(n_expert)]) for b in range(2)]
    x, u = (np.stack([synth.activations(k, seed=s + r) for r in range(4)]) for s in (40, 60))
    src = np.array([3, 0, 1, 3, 2, 0], np.uint32)
    xg = (x / (1 + np.exp(-x.astype(np.float64))) * u).astype(np.float32)
    bd, xd, ud, sd, dstart = [devbuf(b) for b in banks], devbuf(x), devbuf(u), devbuf(src), devbuf(start)
    try:
        dev.set_tuning(moe__form=10)   # (the library's own choice has them only for some of these shapes)
        for gated in (False, True):
            o = [devbuf(shape=(ncols * nrows + 8,), dtype=np.float32, fill=FILL) for _ in banks]
            before = dev.launch_count()
            assert dev.moe_matvec_dev(o[0].ptr, o[1].ptr, t, bd[0].ptr, bd[1].ptr, xd.ptr, ud.ptr if gated else None, sd.ptr, dstart.ptr,
                                      n_expert, ncols, nrows, k)
            assert dev.launch_count() - before == 1
            dev.synchronize()
            for b in range(2):
                want = np.zeros((ncols, nrows))
                for e in np.flatnonzero(counts):
                    cols = slice(start[e], start[e + 1])
                    want[cols] = oracle.matmul_q8act_f64(t, banks[b][e * sheet:(e + 1) * sheet], (xg if gated else x)[src[cols]], nrows, k, counts[e], window)
                got = o[b].get()
                assert np.all(got[ncols * nrows:] == FILL)
                assert nmse(got[:ncols * nrows].reshape(ncols, nrows), want) <= (1e-6 if gated else 1e-10), (gated, b)
    finally:
        dev.set_tuning(moe__form=0)
        dev.SetActWindow(32)


@pytest.mark.parametrize("t,down,window,n_expert,k_used,rows,n_ffn,n_embd,pair", [
    (quant.Q4_K, quant.Q6_K, 256, 40, 8, 1, 512, 512, 0),       # fewer slots than two chunks of lanes; one row
    (quant.Q4_K, quant.Q4_K, 256, 9, 3, 3, 1280, 1792, 0),      # ragged chunks, more row groups than workgroups a row
    (quant.Q4_K, quant.Q4_K, 32, 33, 1, 2, 768, 2304, 0),       # one pair a row
    (quant.Q6_K, quant.Q6_K, 32, 20, 2, 5, 512, 512, 0),
    (quant.Q8_0, quant.Q8_0, 32, 20, 16, 2, 256, 256, 0),       # sixteen pairs, the paired form
    (quant.Q8_0, quant.Q8_0, 32, 12, 4, 3, 1024, 768, 2),       # banks that are not on four bytes: the plain form
    (quant.Q8_0, quant.Q6_K, 32, 12, 5, 3, 768, 1024, 0),
    (quant.Q4_K, quant.Q4_K, 256, 6, 4, 24, 768, 512, 0),       # eight lanes a row, several rows a step, the last step ragged
    (quant.Q4_K, quant.Q6_K, 32, 6, 2, 40, 512, 1024, 0),       # sixteen and eight
    (quant.Q4_K, quant.Q4_K, 256, 6, 2, 20, 1024, 2816, 0),     # sixteen lanes of three slots, the last without one for some
    (quant.Q6_K, quant.Q8_0, 32, 6, 2, 20, 768, 2048, 0),       # 32
    (quant.Q4_K, quant.Q4_K, 256, 12, 8, 1, 512, 768, "one"),   # packed planes, the three widths of a run of rows
    (quant.Q4_K, quant.Q4_K, 256, 12, 3, 3, 1280, 1792, "sheets"),
    (quant.Q4_K, quant.Q4_K, 256, 7, 2, 40, 256, 1024, "one"),
    (quant.Q4_K, quant.Q4_K, 256, 7, 4, 16, 768, 512, "sheets"),
], ids=lambda v: str(v))
def test_block_of_pairs(dev, devbuf, t, down, window, n_expert, k_used, rows, n_ffn, n_embd, pair):
    """The routed block without grouping and combine: a selection with a stride of its own, the first and the last expert
    in use, an id no expert has (it adds nothing), the residual added to and nothing behind it touched."""
    from test_gpu_moe import _oracle_block
    rng = np.random.default_rng(7)
    sel = np.full((rows, k_used + 2), 0xFFFFFFFF, np.uint32)
    for r in range(rows):
        sel[r, :k_used] = rng.permutation(n_expert)[:k_used]
    sel[0, 0], sel[-1, k_used - 1] = (0, n_expert - 1) if k_used > 1 or rows > 1 else (0, 0)
    if rows > 2:
        sel[1, 0] = n_expert + 3
    wt = (rng.random((rows, k_used)) / k_used).astype(np.float32)
    bank = lambda ty, nr, k, s: np.concatenate([synth.random_weights(ty, nr, k, seed=s + e) for e in range(n_expert)])
    banks = [bank(t, n_ffn, n_embd, 0), bank(t, n_ffn, n_embd, 100), bank(down, n_embd, n_ffn, 200)]
    x = np.stack([synth.activations(n_embd, seed=900 + r) for r in range(rows)])
    start = rng.standard_normal((rows, n_embd)).astype(np.float32)
    want = start + _oracle_block(t, *banks, x, sel, wt, n_expert, n_ffn, n_embd, window, td=down)
    dev.SetActWindow(window)
    planes = isinstance(pair, str)
    if planes:
        from test_gpu_moe import _pack_bank
        hold = [_pack_bank(dev, devbuf, t, b, n_expert, r, k, pair) for b, (r, k) in zip(banks, [(n_ffn, n_embd)] * 2 + [(n_embd, n_ffn)])]
    else:
        hold = [devbuf(b) for b in banks]
    xd, sd, wd = devbuf(x), devbuf(sel), devbuf(wt)
    try:
        dev.set_tuning(moe__form=11, q8pair=0 if planes else pair)
        resid = devbuf(np.concatenate([start.reshape(-1), np.full(8, FILL)]))
        before = dev.launch_count()
        args = (xd.ptr, sd.ptr, k_used + 2, wd.ptr, rows, k_used, n_expert, n_ffn, n_embd)
        assert dev.moe_ffn_packed_dev(resid.ptr, t, *[b[0] for b in hold], *args) if planes else \
            dev.moe_ffn_dev(resid.ptr, t, *[b.ptr for b in hold], *args, down_type=down)
        dev.synchronize()
        assert dev.launch_count() - before == 2
        got = resid.get()
        assert np.all(got[rows * n_embd:] == FILL)
        # (an exponential of another machine in front of the second quantizer, as for the other forms)
        assert nmse(got[:rows * n_embd].reshape(rows, n_embd), want) <= 1e-6
    finally:
        dev.set_tuning(moe__form=0, q8pair=0)
        dev.SetActWindow(32)


@pytest.mark.parametrize("t,down,window,form", [(quant.Q8_0, quant.Q6_K, 32, 6), (quant.Q8_0, quant.Q8_0, 32, 8), (quant.Q4_K, quant.Q6_K, 32, 7),
                                                (quant.Q6_K, quant.Q6_K, 256, 6)], ids=lambda v: str(v))
@pytest.mark.parametrize("rows", [90, 700])
def test_block_with_work_lists_from_the_grouping(dev, devbuf, t, down, window, form, rows):
    """The tiles of a block from the work lists its grouping made: the bits of the separate calls, whose matvecs make their own;
    experts nobody chose (the last among them), one of most rows, one and several workgroups of pairs."""
    k_used, n_expert, n_ffn, n_embd = 2, 9, 256, 512
    rng = np.random.default_rng(rows)
    sel = np.stack([rng.choice([1, 2, 4, 5, 7], 2, replace=False) for _ in range(rows)]).astype(np.uint32)
    sel[: rows * 2 // 3, 0], sel[: rows * 2 // 3, 1] = 4, 1 + 4 * (np.arange(rows * 2 // 3) % 2)
    perm = np.argsort(sel.reshape(-1), kind="stable")
    start = np.concatenate([[0], np.cumsum(np.bincount(sel.reshape(-1), minlength=n_expert))]).astype(np.uint32)
    ncols = rows * k_used
    dev.SetActWindow(window)
    bank = lambda ty, nrows, k, s: devbuf(np.concatenate([synth.random_weights(ty, nrows, k, seed=s + e) for e in range(n_expert)]))
    gate, up, dn = bank(t, n_ffn, n_embd, 0), bank(t, n_ffn, n_embd, 50), bank(down, n_embd, n_ffn, 90)
    x = np.stack([synth.activations(n_embd, seed=700 + r) for r in range(rows)])
    wt = rng.random((rows, k_used)).astype(np.float32)
    xd, sd, wd, start_d = devbuf(x), devbuf(sel), devbuf(wt), devbuf(start)
    perm_d, pos_d = devbuf((perm // k_used).astype(np.uint32)), devbuf(np.argsort(perm, kind="stable").astype(np.uint32))
    try:
        dev.set_tuning(moe__form=form)
        r = devbuf(np.zeros((rows, n_embd), np.float32))
        g, u, y = (devbuf(shape=(ncols, n), dtype=np.float32) for n in (n_ffn, n_ffn, n_embd))
        want = devbuf(np.zeros((rows, n_embd), np.float32))
        before = dev.launch_count()
        assert dev.moe_matvec_dev(g.ptr, u.ptr, t, gate.ptr, up.ptr, xd.ptr, None, perm_d.ptr, start_d.ptr, n_expert, ncols, n_ffn, n_embd)
        assert dev.moe_matvec_dev(y.ptr, None, down, dn.ptr, None, g.ptr, u.ptr, None, start_d.ptr, n_expert, ncols, n_embd, n_ffn)
        separate = dev.launch_count() - before + 2
        assert dev.moe_combine_dev(want.ptr, y.ptr, wd.ptr, sd.ptr, k_used, pos_d.ptr, rows, k_used, n_embd)
        for _ in range(2):
            r.put(np.zeros((rows, n_embd), np.float32))
            before = dev.launch_count()
            assert dev.moe_ffn_dev(r.ptr, t, gate.ptr, up.ptr, dn.ptr, xd.ptr, sd.ptr, k_used, wd.ptr, rows, k_used, n_expert, n_ffn,
                                   n_embd, down_type=down)
            assert dev.launch_count() - before == separate - 2   # two work lists less
            dev.synchronize()
            assert np.array_equal(r.get().view(np.uint32), want.get().view(np.uint32))
    finally:
        dev.set_tuning(moe__form=0)
        dev.SetActWindow(32)


@pytest.mark.parametrize("t,down,window,rows,n_ffn,n_embd,packed", [
    (quant.Q4_K, quant.Q6_K, 256, 2, 1280, 768, False), (quant.Q6_K, quant.Q6_K, 32, 3, 512, 1024, False),
    (quant.Q8_0, quant.Q8_0, 32, 4, 448, 320, False), (quant.Q4_K, quant.Q4_K, 256, 4, 768, 512, True),
    (quant.Q4_K, quant.Q4_K, 256, 2, 2304, 256, True)], ids=lambda v: str(v))
def test_dense_block_of_a_few_rows(dev, devbuf, t, down, window, rows, n_ffn, n_embd, packed):
    """A dense block's two to four rows in two launches: one expert, no selection; the residual added to and nothing behind it."""
    from test_gpu_moe import _oracle_block, _pack_bank
    w = [synth.random_weights(t, n_ffn, n_embd, seed=1), synth.random_weights(t, n_ffn, n_embd, seed=2), synth.random_weights(down, n_embd, n_ffn, seed=3)]
    x = np.stack([synth.activations(n_embd, seed=900 + r) for r in range(rows)])
    start = np.stack([synth.activations(n_embd, seed=30 + r) for r in range(rows)])
    sel, wt = np.zeros((rows, 2), np.uint32), np.full((rows, 1), 0.75, np.float32)
    want = start + _oracle_block(t, *w, x, sel, wt, 1, n_ffn, n_embd, window, td=down)
    dev.SetActWindow(window)
    xd, sd, wd = devbuf(x), devbuf(sel), devbuf(wt)
    try:
        resid = devbuf(np.concatenate([start.reshape(-1), np.full(8, FILL)]))
        args = (xd.ptr, sd.ptr, 2, wd.ptr, rows, 1, 1, n_ffn, n_embd)
        before = dev.launch_count()
        if packed:
            hold = [_pack_bank(dev, devbuf, t, b, 1, r, k, "one") for b, (r, k) in zip(w, [(n_ffn, n_embd)] * 2 + [(n_embd, n_ffn)])]
            before = dev.launch_count()
            assert dev.moe_ffn_packed_dev(resid.ptr, t, *[b[0] for b in hold], *args)
        else:
            hold = [devbuf(b) for b in w]
            if t == quant.Q8_0:   # (a mixture takes K in 256s: the dense block by its handle, weight one)
                want = start + _oracle_block(t, *w, x, sel, np.ones_like(wt), 1, n_ffn, n_embd, window, td=down)
                from jitllm_amd import _lib
                assert dev.PrepLayer(0, _lib.LAYER_DENSE, t, n_embd, n_ffn, *w)
                before = dev.launch_count()
                assert dev.layer_ffn_dev(0, xd.ptr, resid.ptr, rows)
            else:
                assert dev.moe_ffn_dev(resid.ptr, t, *[b.ptr for b in hold], *args, down_type=down)
        dev.synchronize()
        assert dev.launch_count() - before == 2
        got = resid.get()
        assert np.all(got[rows * n_embd:] == FILL)
        assert nmse(got[:rows * n_embd].reshape(rows, n_embd), want) <= 1e-6
    finally:
        dev.ReleaseLayers(0, 1)
        dev.SetActWindow(32)


@pytest.mark.parametrize("k_used,n_embd", [(1, 4), (2, 1020), (8, 1024), (9, 1028), (16, 2052)])
def test_combine_bits(dev, devbuf, k_used, n_embd):
    """The weighted sum at the edges of its groups of eight experts and of its workgroups of 1024 columns: one f32 product and
    one f32 addition an expert, ascending ids, ids that are equal in slot order (bit for bit)."""
    rows = 3
    rng = np.random.default_rng(k_used)
    sel = rng.permuted(np.tile(np.arange(20, dtype=np.uint32), (rows, 1)), axis=1)[:, :k_used + 2].copy()
    sel[1, :k_used] = 7
    wt = rng.random((rows, k_used), dtype=np.float32)
    pos = rng.permutation(rows * k_used).astype(np.uint32)
    y = rng.standard_normal((rows * k_used, n_embd)).astype(np.float32)
    resid = rng.standard_normal((rows, n_embd)).astype(np.float32)
    want = resid.copy()
    for r in range(rows):
        for s in np.argsort(sel[r, :k_used], kind="stable"):
            want[r] = want[r] + wt[r, s] * y[pos[r * k_used + s]]
    rd, yd, wd, sd, pd = devbuf(resid), devbuf(y), devbuf(wt), devbuf(sel), devbuf(pos)
    assert dev.moe_combine_dev(rd.ptr, yd.ptr, wd.ptr, sd.ptr, k_used + 2, pd.ptr, rows, k_used, n_embd)
    dev.synchronize()
    assert np.array_equal(rd.get().view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("t,down,window,forms", [
    (quant.Q4_K, quant.Q4_K, 256, ((0, 0), (1, 0), (2, 0), (3, 1), (3, 2), (3, 3), (4, 0), (5, 0), (9, 0), (10, 0), (11, 0))),
    (quant.Q4_K, quant.Q6_K, 256, ((0, 0), (5, 0), (9, 0), (10, 0), (11, 0))), (quant.Q8_0, quant.Q8_0, 32, ((0, 0), (1, 0), (5, 0), (6, 0), (10, 0), (11, 0))),
    (quant.Q4_K, "one", 256, ((0, 0), (1, 0), (3, 1), (4, 0), (5, 0), (9, 0), (11, 0)))], ids=["q4_k", "q4_k-q6_k", "q8_0", "planes"])
@pytest.mark.parametrize("rows", [2, 40, 600])
def test_ids_that_no_expert_has(dev, devbuf, t, down, window, forms, rows):
    """Pairs whose id no expert has add nothing, in every form of the block, with one workgroup of pairs and with several: the
    grouping leaves them out, so the columns behind the last expert's have no source row and a pair no column.  The last
    expert is nobody's and holds an infinite scale, which must reach no row."""
    from test_gpu_moe import _oracle_block, _pack_bank
    n_expert, k_used, n_ffn, n_embd, period = 5, 3, 512, 256, 8
    planes = isinstance(down, str)
    td = t if planes else down
    rng = np.random.default_rng(11)
    some = np.stack([rng.permutation(n_expert - 1)[:k_used] for _ in range(period)]).astype(np.uint32)
    some[0, 1], some[1, 0], some[3, 2], some[4], some[6, 0] = 0xFFFFFFFF, n_expert, 70000, n_expert + 1, 0x80000000
    wts = (rng.random((period, k_used)) / k_used).astype(np.float32)
    xs = np.stack([synth.activations(n_embd, seed=900 + r) for r in range(period)])
    bank = lambda ty, nr, k, s: np.concatenate([synth.random_weights(ty, nr, k, seed=s + e) for e in range(n_expert)])
    banks = [bank(t, n_ffn, n_embd, 0), bank(t, n_ffn, n_embd, 100), bank(td, n_embd, n_ffn, 200)]
    want = _oracle_block(t, *banks, xs, some, wts, n_expert, n_ffn, n_embd, window, td=td)
    last = banks[2][(n_expert - 1) * (len(banks[2]) // n_expert):].reshape(-1, quant.BLOCK[td][1])
    d = {quant.Q4_K: 0, quant.Q6_K: 208, quant.Q8_0: 0}[td]
    last[:, d], last[:, d + 1] = 0x00, 0x7C
    at = np.arange(rows) % period
    dev.SetActWindow(window)
    hold = [_pack_bank(dev, devbuf, t, b, n_expert, r, k, "one") for b, (r, k) in zip(banks, [(n_ffn, n_embd)] * 2 + [(n_embd, n_ffn)])] if planes else \
        [devbuf(b) for b in banks]
    xd, sd, wd = devbuf(xs[at]), devbuf(some[at]), devbuf(wts[at])
    try:
        for form, g16 in forms:
            if form in (10, 11) and rows > 40:
                continue
            dev.set_tuning(moe__form=form, moe__group16=g16)
            resid = devbuf(np.concatenate([np.zeros(rows * n_embd, np.float32), np.full(8, FILL)]))
            args = (xd.ptr, sd.ptr, k_used, wd.ptr, rows, k_used, n_expert, n_ffn, n_embd)
            assert dev.moe_ffn_packed_dev(resid.ptr, t, *[b[0] for b in hold], *args) if planes else \
                dev.moe_ffn_dev(resid.ptr, t, *[b.ptr for b in hold], *args, down_type=down)
            dev.synchronize()
            got = resid.get()
            assert np.all(got[rows * n_embd:] == FILL)
            # (an exponential of another machine in front of the second quantizer, as for the other tests of a block)
            assert nmse(got[:rows * n_embd].reshape(rows, n_embd), want[at]) <= 1e-6, (form, g16)
    finally:
        dev.set_tuning(moe__form=0, moe__group16=0)
        dev.SetActWindow(32)


@pytest.mark.parametrize("t,window,nrows,k,counts,launches", [
    (quant.Q6_K, 256, 2048, 4096, [9, 7], 2), (quant.Q8_0, 32, 2048, 4096, [9, 7], 2), (quant.Q4_K, 32, 4096, 4096, [9, 7], 2),
    (quant.Q6_K, 256, 1024, 1024, [1, 2, 1, 1], 1), (quant.Q8_0, 32, 4096, 2048, [1] * 8, 1)],
    ids=lambda v: str(v))
def test_columns_that_share_a_large_sheet(dev, devbuf, t, window, nrows, k, counts, launches):
    """Columns that share sheets of some megabytes are not given a decode matvec each, which would read a sheet again for every
    one of them (two launches); small sheets and columns of their own are (one)."""
    n_expert, ncols = len(counts), sum(counts)
    start = np.concatenate([[0], np.cumsum(counts)]).astype(np.uint32)
    sheet = nrows * quant.row_bytes(t, k)
    banks = [np.concatenate([synth.random_weights(t, nrows, k, seed=20 * b + e) for e in range(n_expert)]) for b in range(2)]
    x = np.stack([synth.activations(k, seed=40 + r) for r in range(ncols)])
    bd, xd, sd = [devbuf(b) for b in banks], devbuf(x), devbuf(start)
    dev.SetActWindow(window)
    try:
        o = [devbuf(shape=(ncols, nrows), dtype=np.float32, fill=FILL) for _ in banks]
        before = dev.launch_count()
        assert dev.moe_matvec_dev(o[0].ptr, o[1].ptr, t, bd[0].ptr, bd[1].ptr, xd.ptr, None, None, sd.ptr, n_expert, ncols, nrows, k)
        made = dev.launch_count() - before
        dev.synchronize()
        assert made == launches
        e = n_expert - 1
        for b in range(2):
            want = oracle.matmul_q8act_f64(t, banks[b][e * sheet:], x[start[e]:], nrows, k, counts[e], window)
            assert nmse(o[b].get()[start[e]:], want) <= 1e-10
    finally:
        dev.SetActWindow(32)


def test_pairs_that_share_large_sheets_are_grouped(dev, devbuf):
    """16 experts, top-4: six rows' pairs, which share sheets of 7.8 MB, are grouped; two rows' hardly share any and are not.
    (Blocks of zeros: the residual stays.)"""
    n_expert, k_used, n_ffn, n_embd = 16, 4, 2048, 3584
    bank = devbuf(np.zeros(n_expert * n_ffn * quant.row_bytes(quant.Q8_0, n_embd), np.uint8))
    for rows, pairs_alone in ((6, False), (2, True)):
        sel = np.stack([np.random.default_rng(r).permutation(n_expert)[:k_used] for r in range(rows)]).astype(np.uint32)
        start = np.stack([synth.activations(n_embd, seed=30 + r) for r in range(rows)])
        xd, sd, wd, resid = devbuf(start), devbuf(sel), devbuf(np.full((rows, k_used), 0.25, np.float32)), devbuf(start)
        before = dev.launch_count()
        assert dev.moe_ffn_dev(resid.ptr, quant.Q8_0, bank.ptr, bank.ptr, bank.ptr, xd.ptr, sd.ptr, k_used, wd.ptr, rows, k_used, n_expert, n_ffn, n_embd)
        assert (dev.launch_count() - before == 2) == pairs_alone
        dev.synchronize()
        assert np.array_equal(resid.get(), start)
