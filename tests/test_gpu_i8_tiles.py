"""The int8 tile kernels (kernels/gemm_i8.h), dense and per expert, at the edges of their tiles: rows and tokens one
short of, at and one past a tile, K of an odd number of stages, K splits, every shape; against the oracle in f64."""
import time

import numpy as np
import pytest

import oracle
from conftest import nmse
from jitllm_amd import quant, synth
from jitllm_amd.device import Packed

pytestmark = pytest.mark.gpu
FILL = np.float32(4e30)
KINDS = [(quant.Q8_0, 32), (quant.Q4_K, 32), (quant.Q6_K, 32), (quant.Q6_K, 256)]


@pytest.mark.parametrize("t,window", KINDS, ids=["q8_0", "q4_k", "q6_k", "q6_k-w256"])
@pytest.mark.parametrize("nrows,k,ntok", [(1, 256, 65), (63, 512, 127), (129, 768, 129), (200, 256, 300), (130, 1280, 66)])
def test_dense_tiles(dev, devbuf, t, window, nrows, k, ntok):
    if t == quant.Q8_0 and k == 768:
        k = 640   # five stages of 128
    dev.SetActWindow(window)
    w = synth.random_weights(t, nrows, k, seed=nrows + k)
    x = np.stack([synth.activations(k, seed=900 + i) * np.float32(1 + i % 3) for i in range(ntok)])
    want = oracle.matmul_q8act_f64(t, w, x, nrows, k, ntok, window)
    wd, xd = devbuf(w), devbuf(x)
    try:
        for shape in (0, 1, 2) if t == quant.Q8_0 else (0, 2):
            for split in (0, 1, 2, 5):
                dev.set_tuning(gemm__i8=shape, gemm__split=split)
                o = devbuf(shape=(ntok * nrows + 8,), dtype=np.float32, fill=FILL)
                assert dev.matmul_dev(o.ptr, t, wd.ptr, xd.ptr, nrows, k, ntok)
                dev.synchronize()
                got = o.get()
                assert np.all(got[ntok * nrows:] == FILL)
                assert nmse(got[:ntok * nrows].reshape(ntok, nrows), want) <= 1e-10, (shape, split)
    finally:
        dev.set_tuning(gemm__i8=0, gemm__split=0)
        dev.SetActWindow(32)


@pytest.mark.parametrize("t,window", KINDS, ids=["q8_0", "q4_k", "q6_k", "q6_k-w256"])
@pytest.mark.parametrize("nrows,k", [(130, 512), (256, 256)])
def test_tiles_per_expert(dev, devbuf, t, window, nrows, k):
    """Experts of 0, 1, 31, 64, 65 and 129 columns, two banks, gathered rows, a gated activation; the few-token kernel
    and every tile."""
    counts = [1, 0, 31, 64, 65, 129, 0]
    n_expert, ncols = len(counts), sum(counts)
    start = np.concatenate([[0], np.cumsum(counts)]).astype(np.uint32)
    dev.SetActWindow(window)
    sheet = nrows * quant.row_bytes(t, k)
    banks = [np.concatenate([synth.random_weights(t, nrows, k, seed=10 * b + e) for e in range(n_expert)]) for b in range(2)]
    x = np.stack([synth.activations(k, seed=300 + r) for r in range(40)])
    src = (np.arange(ncols) * 7 % 40).astype(np.uint32)
    u = np.stack([synth.activations(k, seed=500 + r) for r in range(40)])
    xg = (x / (1 + np.exp(-x.astype(np.float64))) * u).astype(np.float32)
    bd, xd, ud, sd, dstart = [devbuf(b) for b in banks], devbuf(x), devbuf(u), devbuf(src), devbuf(start)
    try:
        for gated in (False, True):
            act = xg if gated else x
            want = [np.zeros((ncols, nrows)) for _ in banks]
            for b in range(2):
                for e in range(n_expert):
                    cols = slice(start[e], start[e + 1])
                    if counts[e]:
                        want[b][cols] = oracle.matmul_q8act_f64(t, banks[b][e * sheet:(e + 1) * sheet], act[src[cols]], nrows, k, counts[e], window)
            # (8: Q8_0's tiles of 128 x 128; 7: Q6_K's of 64 columns, window 32)
            for form in (0, 5, 6) + ((8,) if t == quant.Q8_0 else (7,) if t == quant.Q6_K and window == 32 else ()):
                dev.set_tuning(moe__form=form)
                o = [devbuf(shape=(ncols * nrows + 8,), dtype=np.float32, fill=FILL) for _ in banks]
                assert dev.moe_matvec_dev(o[0].ptr, o[1].ptr, t, bd[0].ptr, bd[1].ptr, xd.ptr, ud.ptr if gated else None, sd.ptr, dstart.ptr,
                                          n_expert, ncols, nrows, k)
                dev.synchronize()
                for b in range(2):
                    got = o[b].get()
                    assert np.all(got[ncols * nrows:] == FILL)
                    # (the gated activation: an exponential of another machine in front of the quantizer)
                    assert nmse(got[:ncols * nrows].reshape(ncols, nrows), want[b]) <= (1e-6 if gated else 1e-10), (gated, form, b)
    finally:
        dev.set_tuning(moe__form=0)
        dev.SetActWindow(32)


@pytest.mark.parametrize("nrows,k,ntok", [(1, 256, 256), (65, 640, 255), (191, 128, 513), (300, 1280, 257)])
def test_tiles_of_64_rows_behind_those_of_128(dev, devbuf, nrows, k, ntok):
    """Q8_0, 256 tokens: none, some and all of the rows in tiles of 64 rows (two threads a block of weights); a row whose scale
    is infinite among them.  Every value is the tile of 128 rows' bit for bit."""
    dev.SetActWindow(32)
    w = synth.random_weights(quant.Q8_0, nrows, k, seed=nrows + k)
    w.reshape(nrows, -1)[-1, 34:36] = (0x00, 0x7C)   # an infinite scale in the last row's second block
    x = np.stack([synth.activations(k, seed=900 + i) * np.float32(1 + i % 3) for i in range(ntok)])
    wd, xd = devbuf(w), devbuf(x)
    want = oracle.matmul_q8act_f64(quant.Q8_0, w, x, nrows, k, ntok, 32)
    try:
        ref = None
        for tall in [1] + [2 + n for n in range((nrows + 127) // 128 + 1)]:
            dev.set_tuning(gemm__i8=3, gemm__split=1, gemm__tall=tall)
            o = devbuf(shape=(ntok * nrows + 8,), dtype=np.float32, fill=FILL)
            assert dev.matmul_dev(o.ptr, quant.Q8_0, wd.ptr, xd.ptr, nrows, k, ntok)
            dev.synchronize()
            got = o.get()
            assert np.all(got[ntok * nrows:] == FILL)
            got = got[:ntok * nrows].reshape(ntok, nrows)
            ref = got if ref is None else ref
            assert np.array_equal(got.view(np.uint32), ref.view(np.uint32)), tall
        if nrows > 1:
            assert nmse(ref[:, :-1], want[:, :-1]) <= 1e-10
        assert np.all(np.isinf(ref[:, -1]) | np.isnan(ref[:, -1]))
    finally:
        dev.set_tuning(gemm__i8=0, gemm__split=0, gemm__tall=0)


@pytest.mark.parametrize("nrows,k,ntok", [(1, 128, 257), (127, 640, 255), (129, 512, 513), (300, 1280, 256)])
def test_tiles_of_256_tokens(dev, devbuf, nrows, k, ntok):
    """Q8_0, 256 tokens x 128 rows on eight wavefronts: one token past a tile and one short of it, a wavefront and more without a
    token of theirs, rows that end inside a tile, one stage of K; K slices."""
    dev.SetActWindow(32)
    w = synth.random_weights(quant.Q8_0, nrows, k, seed=nrows + k)
    x = np.stack([synth.activations(k, seed=900 + i) * np.float32(1 + i % 3) for i in range(ntok)])
    want = oracle.matmul_q8act_f64(quant.Q8_0, w, x, nrows, k, ntok, 32)
    wd, xd = devbuf(w), devbuf(x)
    try:
        for split in (1, 3):
            dev.set_tuning(gemm__i8=3, gemm__split=split)
            o = devbuf(shape=(ntok * nrows + 8,), dtype=np.float32, fill=FILL)
            assert dev.matmul_dev(o.ptr, quant.Q8_0, wd.ptr, xd.ptr, nrows, k, ntok)
            dev.synchronize()
            got = o.get()
            assert np.all(got[ntok * nrows:] == FILL)
            assert nmse(got[:ntok * nrows].reshape(ntok, nrows), want) <= 1e-10, split
    finally:
        dev.set_tuning(gemm__i8=0, gemm__split=0)


@pytest.mark.parametrize("t", [quant.Q8_0, quant.Q4_K], ids=["q8_0", "q4_k"])
@pytest.mark.parametrize("ntok", [1, 3, 40, 300])
def test_scales_that_are_no_numbers(dev, devbuf, t, ntok):
    """A block whose scale is infinite makes its row infinite with the scale's sign, two of opposite sign or a NaN make it NaN, in every kernel (matvec, few tokens, tiles, K slices, tiles per expert); the other rows as ever."""
    nrows, k, window = 131, 768, 32
    dev.SetActWindow(window)
    w = synth.random_weights(t, nrows, k, seed=3)
    # (weights, scales and activations above zero: a block's products have one sign)
    x = np.abs(np.stack([synth.activations(k, seed=900 + i) for i in range(ntok)])) + np.float32(0.1)
    b = w.reshape(nrows, -1, quant.BLOCK[t][1])
    if t == quant.Q4_K:
        b[:, :, 4:16] |= 1      # every sub-block's scale at least one
        b[:, :, 8:12] &= 0x3F   # (minimums: six bits)
    else:
        b[:, :, 2:] = b[:, :, 2:] & 0x7F | 1
    inf, ninf, nan = (0x00, 0x7C), (0x00, 0xFC), (0x00, 0x7E)
    b[5, 0, :2], b[64, 1, :2], b[127, 2, :2], b[130, 1, :2] = inf, ninf, nan, inf
    b[100, 0, :2], b[100, 2, :2] = inf, ninf
    want = oracle.matmul_q8act_f64(t, w, x, nrows, k, ntok, window)
    want[:, [5, 64, 100, 127, 130]] = np.inf, -np.inf, np.nan, np.nan, np.inf   # (the oracle forms Q8_0 with a bias: NaN there)
    wd, xd = devbuf(w), devbuf(x)
    start = devbuf(np.array([0, 0, ntok], np.uint32))
    bank = devbuf(np.concatenate([w, w]))

    def check(o, what):
        dev.synchronize()
        got = o.get()[:ntok * nrows].reshape(ntok, nrows)
        assert np.array_equal(np.isnan(got), np.isnan(want)), what
        assert np.array_equal(np.isposinf(got), np.isposinf(want)) and np.array_equal(np.isneginf(got), np.isneginf(want)), what
        ok = np.isfinite(want)
        assert nmse(got[ok], want[ok]) <= 1e-10, what
    try:
        with np.errstate(invalid="ignore"):
            for few, shape, split in ((0, 0, 0), (1, 0, 0), (2, 0, 0), (2, 0, 2), (2, 1, 0), (2, 2, 3), (2, 3, 0)):
                if shape in (1, 3) and t != quant.Q8_0:
                    continue
                dev.set_tuning(gemm__few=few, gemm__i8=shape, gemm__split=split)
                o = devbuf(shape=(ntok * nrows + 8,), dtype=np.float32, fill=FILL)
                assert dev.matmul_dev(o.ptr, t, wd.ptr, xd.ptr, nrows, k, ntok)
                check(o, (few, shape, split))
            for form in (0, 5, 6, 8) if t == quant.Q8_0 else (0, 5, 6):
                dev.set_tuning(gemm__few=0, gemm__i8=0, gemm__split=0, moe__form=form)
                o = devbuf(shape=(ntok * nrows + 8,), dtype=np.float32, fill=FILL)
                assert dev.moe_matvec_dev(o.ptr, None, t, bank.ptr, None, xd.ptr, None, None, start.ptr, 2, ntok, nrows, k)
                check(o, form)
    finally:
        dev.set_tuning(gemm__few=0, gemm__i8=0, gemm__split=0, moe__form=0)
        dev.SetActWindow(32)


@pytest.mark.parametrize("planes", [False, True], ids=["rows", "planes"])
@pytest.mark.parametrize("ntok", [12, 40, 300])   # (fewer may be the matvec's, which sums four sub-scales first: row 77 is infinite there)
def test_q6_scales_that_are_no_numbers(dev, devbuf, planes, ntok):
    """Q6_K, window 32, where the row's scale meets sums of blocks: a row whose scale is infinite in a super-block has the infinities and NaN of its blocks' products one by one, in the few-token kernel, the tiles and K slices; the other rows as ever."""
    nrows, k, window, t = 131, 1536, 32, quant.Q6_K
    dev.SetActWindow(window)
    w = synth.random_weights(t, nrows, k, seed=4)
    x = np.abs(np.stack([synth.activations(k, seed=950 + i) for i in range(ntok)])) + np.float32(0.1)
    b = w.reshape(nrows, -1, 210)
    b[:, :, :128] |= 0x11                                   # every weight 33 .. 47 less 32, every sub-scale 1 .. 127: a block's products have one sign
    b[:, :, 128:192] = 0xAA
    b[:, :, 192:208] = b[:, :, 192:208] & 0x7F | 1
    b[:, :, 209] &= 0x7F
    inf, ninf, nan = (0x00, 0x7C), (0x00, 0xFC), (0x00, 0x7E)
    b[5, 0, 208:], b[64, 5, 208:], b[127, 2, 208:], b[130, 1, 208:] = inf, ninf, nan, inf
    b[100, 0, 208:], b[100, 4, 208:] = inf, ninf
    b[77, 3, 208:] = inf
    b[77, 3, 192:194] = 0xFF                                # (one block's products below zero, the sum of the super-block's above)
    want = oracle.matmul_q8act_f64(t, w, x, nrows, k, ntok, window)
    want[:, [5, 64, 77, 100, 127, 130]] = np.inf, -np.inf, np.nan, np.nan, np.nan, np.inf
    wd, xd = devbuf(w), devbuf(x)
    mat = wd.ptr
    if planes:
        bufs = [devbuf(shape=(n,), dtype=np.uint32) for n in quant.packed_words(t, nrows, k)]
        assert dev.pack_weights_dev(t, wd.ptr, nrows, k, *[a.ptr for a in bufs])
        mat = Packed(*[a.ptr for a in bufs], 0, nrows)
    try:
        for few, split in ((0, 0), (1, 0), (2, 0), (2, 2), (2, 3)):
            dev.set_tuning(gemm__few=few, gemm__split=split)
            o = devbuf(shape=(ntok * nrows + 8,), dtype=np.float32, fill=FILL)
            assert (dev.matmul_packed_dev if planes else dev.matmul_dev)(o.ptr, t, mat, xd.ptr, nrows, k, ntok)
            dev.synchronize()
            got = o.get()
            assert np.all(got[ntok * nrows:] == FILL)
            got = got[:ntok * nrows].reshape(ntok, nrows)
            assert np.array_equal(np.isnan(got), np.isnan(want)), (few, split)
            assert np.array_equal(np.isposinf(got), np.isposinf(want)) and np.array_equal(np.isneginf(got), np.isneginf(want)), (few, split)
            ok = np.isfinite(want)
            assert nmse(got[ok], want[ok]) <= 1e-10, (few, split)
    finally:
        dev.set_tuning(gemm__few=0, gemm__split=0)
        dev.SetActWindow(32)


@pytest.mark.parametrize("ntok,few", [(12, 0), (200, 2)], ids=["few", "tiles"])
@pytest.mark.parametrize("t", [quant.Q8_0, quant.Q4_K, quant.Q6_K], ids=["q8_0", "q4_k", "q6_k"])
def test_an_activation_that_is_no_number(dev, devbuf, t, ntok, few):
    """Window 32, one activation infinite or NaN, in the first and the last token: that token's sums are NaN, the others' bits are those
    without it, and the call takes about as long (three times allowed; summed again row by row it was 6 to 130 times).  One that is
    finite but large enough for sums without the row's scale to pass the largest f32: the oracle's values."""
    nrows, k = 2048, 2048
    dev.SetActWindow(32)
    w = synth.quantized_weights(t, nrows, k, seed=31)
    x = np.stack([synth.activations(k, seed=970 + i) for i in range(ntok)])
    wd, o = devbuf(w), devbuf(shape=(ntok, nrows), dtype=np.float32)

    def call(xd):
        assert dev.matmul_dev(o.ptr, t, wd.ptr, xd.ptr, nrows, k, ntok)

    def us(xd):
        best = 1e30
        for _ in range(5):
            dev.synchronize()
            t0 = time.perf_counter()
            for _ in range(20):
                call(xd)
            dev.synchronize()
            best = min(best, (time.perf_counter() - t0) / 20 * 1e6)
        return best

    dev.set_tuning(gemm__few=few)
    try:
        clean = devbuf(x)
        call(clean)
        dev.synchronize()
        ref, base = o.get(), us(clean)
        for tok in (0, ntok - 1):
            for v in (np.inf, np.nan, 3e36):
                y = x.copy()
                y[tok, 77] = v
                yd = devbuf(y)
                call(yd)
                dev.synchronize()
                got = o.get()
                others = np.arange(ntok) != tok
                assert np.array_equal(got[others].view(np.uint32), ref[others].view(np.uint32))
                if np.isfinite(v):
                    want = oracle.matmul_q8act_f64(t, w, y[tok:tok + 1], nrows, k, 1, 32)
                    assert np.isfinite(got[tok]).all() and nmse(got[tok].astype(np.float64) * 1e-20, want[0] * 1e-20) <= 1e-10
                else:
                    assert np.isnan(got[tok]).all()
                    assert us(yd) <= 3 * base, (tok, v)
    finally:
        dev.set_tuning(gemm__few=0)


@pytest.mark.parametrize("t,avg,form", [(quant.Q8_0, 36, 5), (quant.Q8_0, 46, 6), (quant.Q4_K, 40, 5), (quant.Q4_K, 55, 5), (quant.Q6_K, 36, 5), (quant.Q6_K, 55, 7)])
def test_banks_at_forty_to_fifty_six_columns(dev, devbuf, t, avg, form):
    """What a grouped matmul takes by itself between the few-token kernel and the large tiles, window 32: the forced form's values bit for bit, the few-token kernel's also with its columns in fours of tiles, and the oracle's."""
    n_expert, nrows, k = 128, 160, 256
    ncols = n_expert * avg
    dev.SetActWindow(32)
    w = synth.random_weights(t, nrows, k, seed=21)
    x = np.stack([synth.activations(k, seed=400 + i) for i in range(61)])
    src = (np.arange(ncols) * 7 % 61).astype(np.uint32)
    cuts = np.arange(n_expert + 1, dtype=np.int64) * avg
    cuts[1:-1] += np.random.default_rng(5).integers(-avg // 2, avg // 2, n_expert - 1)   # (up to two averages an expert)
    want = oracle.matmul_q8act_f64(t, w, x, nrows, k, 61, 32)[src]
    bank, xd, sd, cd = devbuf(np.tile(w, n_expert)), devbuf(x), devbuf(src), devbuf(cuts.astype(np.uint32))
    try:
        got = []
        for f, nt in ((0, 0), (form, 4 if form == 5 else 0)):
            dev.set_tuning(moe__form=f, few__nt=nt)
            o = [devbuf(shape=(ncols * nrows + 8,), dtype=np.float32, fill=FILL) for _ in range(2)]
            assert dev.moe_matvec_dev(o[0].ptr, o[1].ptr, t, bank.ptr, bank.ptr, xd.ptr, None, sd.ptr, cd.ptr, n_expert, ncols, nrows, k)
            dev.synchronize()
            got.append([a.get() for a in o])
        for a, b in zip(*got):
            assert np.all(a[ncols * nrows:] == FILL) and np.array_equal(a, b)
            assert nmse(a[:ncols * nrows].reshape(ncols, nrows), want) <= 1e-10
    finally:
        dev.set_tuning(moe__form=0, few__nt=0)
        dev.SetActWindow(32)
