"""The int8 few-token matmul (up to 64 tokens) and the planes-to-rows kernels at the sizes where they can go
wrong: one token and every edge of a token tile, rows that end inside a row tile, K of one super-block, K that
ends inside a unit of 256 (Q8_0), more super-blocks than wavefronts, a row range of a larger plane set.  Bar:
NMSE <= 1e-10 against the f64 evaluation of the same int8 activations."""
import numpy as np
import pytest

import oracle
from conftest import nmse
from jitllm_amd import quant, synth
from jitllm_amd.device import Packed

pytestmark = pytest.mark.gpu

SHAPES = [(1, 16, 256), (3, 37, 1280), (16, 100, 2816), (17, 130, 1024), (33, 48, 512), (64, 200, 2304), (5, 33, 160),
          (20, 50, 320), (7, 64, 832)]
# (token tiles, row tiles): the built-in choice and every compiled pair
TILES = [(0, 0), (1, 1), (1, 2), (2, 1), (3, 1), (3, 2), (4, 1), (4, 2), (1, 4), (2, 2), (2, 4)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("window", [32, 256])
@pytest.mark.parametrize("t", [quant.Q8_0, quant.Q4_K, quant.Q6_K], ids=["q8_0", "q4_k", "q6_k"])
def test_few_tokens_rows_and_planes(dev, devbuf, t, window, shape):
    ntok, nrows, k = shape
    if k % quant.block_elems(t):
        pytest.skip("K is not a whole number of this type's blocks")
    dev.SetActWindow(window)
    w = synth.random_weights(t, nrows, k, seed=ntok)
    x = np.stack([synth.activations(k, seed=100 + i) * np.float32(1 + i % 7) for i in range(ntok)])
    x[ntok // 2, :32] = 0
    want = oracle.matmul_q8act_f64(t, w, x, nrows, k, ntok, window)
    wd, xd = devbuf(w), devbuf(x)
    planes = [devbuf(np.zeros(max(n, 4), np.uint32)) for n in quant.packed_words(t, nrows, k)]
    assert dev.pack_weights_dev(t, wd.ptr, nrows, k, *[p.ptr for p in planes])
    r0, part = 3, nrows - 7
    try:
        for nt, rt in TILES:
            dev.set_tuning(gemm__few=1, few__nt=nt, few__rt=rt)
            calls = [(True, 0, nrows), (True, r0, part)]
            if nt < 4 and rt < 4 and (nt, rt) != (2, 2) or nt == 4:
                calls.append((False, 0, nrows))
            for packed, lo, n in calls:
                out = devbuf(np.full(ntok * n + 8, 3e30, np.float32))
                if packed:
                    assert dev.matmul_packed_dev(out.ptr, t, Packed(*[p.ptr for p in planes], lo, nrows), xd.ptr, n, k, ntok)
                else:
                    assert dev.matmul_dev(out.ptr, t, wd.ptr, xd.ptr, n, k, ntok)
                dev.synchronize()
                got = out.get()
                assert np.all(got[ntok * n:] == np.float32(3e30)), "wrote past the output"
                e = nmse(got[:ntok * n].reshape(ntok, n), want[:, lo:lo + n])
                assert e <= 1e-10, (nt, rt, packed, lo, e)
    finally:
        dev.set_tuning(gemm__few=0, few__nt=0, few__rt=0)
        dev.SetActWindow(32)


@pytest.mark.parametrize("rows", [1, 2])
@pytest.mark.parametrize("waves", [1, 3, 4, 8])
def test_few_tokens_three_tiles_dealt_over_wavefronts(dev, devbuf, waves, rows):
    """K of eleven super-blocks over fewer wavefronts than that, the last round part empty; 33, 47 and 48 tokens."""
    t, nrows, k = quant.Q4_K, 70, 2816
    w = synth.random_weights(t, nrows, k, seed=3)
    x = np.stack([synth.activations(k, seed=i) for i in range(48)])
    want = oracle.matmul_q8act_f64(t, w, x, nrows, k, 48, 32)
    wd, xd = devbuf(w), devbuf(x)
    try:
        dev.set_tuning(few__waves=waves, few__rt=rows)
        for ntok in (33, 47, 48):
            out = devbuf(np.full(ntok * nrows + 8, 3e30, np.float32))
            assert dev.matmul_dev(out.ptr, t, wd.ptr, xd.ptr, nrows, k, ntok)
            dev.synchronize()
            got = out.get()
            assert np.all(got[ntok * nrows:] == np.float32(3e30))
            assert nmse(got[:ntok * nrows].reshape(ntok, nrows), want[:ntok]) <= 1e-10
    finally:
        dev.set_tuning(few__waves=0, few__rt=0)


@pytest.mark.parametrize("t,nrows,k", [(quant.Q8_0, 65, 32), (quant.Q8_0, 130, 544), (quant.Q4_K, 63, 256), (quant.Q6_K, 129, 768),
                                       (quant.MXFP4, 67, 96), (quant.MXFP4, 200, 800)])
def test_planes_to_rows_round_trip(dev, devbuf, t, nrows, k):
    src = synth.random_weights(t, nrows, k, seed=k)
    wd = devbuf(src)
    planes = [devbuf(np.zeros(max(n, 4), np.uint32)) for n in quant.packed_words(t, nrows, k)]
    assert dev.pack_weights_dev(t, wd.ptr, nrows, k, *[p.ptr for p in planes])
    rb = quant.row_bytes(t, k)
    for lo, n in ((0, nrows), (1, nrows - 2), (nrows - 1, 1)):
        dst = devbuf(np.full(n * rb + 32, 0xEE, np.uint8))
        assert dev.unpack_weights_dev(t, Packed(*[p.ptr for p in planes], lo, nrows), n, k, dst.ptr)
        dev.synchronize()
        got = dst.get()
        assert np.array_equal(got[:n * rb], src[lo * rb:(lo + n) * rb]) and np.all(got[n * rb:] == 0xEE)


@pytest.mark.parametrize("ntok,nrows,k", [(65, 200, 256), (97, 77, 2304), (130, 16, 1024), (200, 1030, 1152)], ids=lambda v: str(v))
@pytest.mark.parametrize("window", [32, 256])
@pytest.mark.parametrize("t", [quant.Q8_0, quant.Q4_K, quant.Q6_K], ids=["q8_0", "q4_k", "q6_k"])
def test_more_than_one_group_of_tokens(dev, devbuf, t, window, ntok, nrows, k):
    """Groups of tokens on workgroups of their own: token tiles the groups do not divide (a last tile that belongs to the next
    group is not stored twice), one token in the last, the library's own choice; rows and planes."""
    if k % quant.block_elems(t) or (t == quant.Q8_0 and window == 256):
        pytest.skip("K is not a whole number of this type's blocks")
    dev.SetActWindow(window)
    w = synth.random_weights(t, nrows, k, seed=ntok)
    x = np.stack([synth.activations(k, seed=100 + i) * np.float32(1 + i % 7) for i in range(ntok)])
    want = oracle.matmul_q8act_f64(t, w, x, nrows, k, ntok, window)
    wd, xd = devbuf(w), devbuf(x)
    planes = [devbuf(np.zeros(max(n, 4), np.uint32)) for n in quant.packed_words(t, nrows, k)]
    assert dev.pack_weights_dev(t, wd.ptr, nrows, k, *[p.ptr for p in planes])
    try:
        for nt in (0, 1, 2, 3, 4):
            dev.set_tuning(gemm__few=1 if nt else 0, few__nt=nt)
            for packed in (False, True):
                out = devbuf(np.full(ntok * nrows + 8, 3e30, np.float32))
                if packed:
                    assert dev.matmul_packed_dev(out.ptr, t, Packed(*[p.ptr for p in planes], 0, nrows), xd.ptr, nrows, k, ntok)
                else:
                    assert dev.matmul_dev(out.ptr, t, wd.ptr, xd.ptr, nrows, k, ntok)
                dev.synchronize()
                got = out.get()
                assert np.all(got[ntok * nrows:] == np.float32(3e30)), "wrote past the output"
                assert nmse(got[:ntok * nrows].reshape(ntok, nrows), want) <= 1e-10, (nt, packed)
    finally:
        dev.set_tuning(gemm__few=0, few__nt=0)
        dev.SetActWindow(32)


@pytest.mark.parametrize("ntok,nrows,k", [(2, 16, 256), (2, 700, 2048), (3, 4100, 1024), (8, 1030, 4352), (16, 37, 1280)], ids=lambda v: str(v))
@pytest.mark.parametrize("t", [quant.Q8_0, quant.Q4_K, quant.Q6_K], ids=["q8_0", "q4_k", "q6_k"])
def test_a_few_tokens_as_matvecs_in_one_launch(dev, devbuf, t, ntok, nrows, k):
    """One launch, and the values of the decode matvec token by token, over rows and planes; a plane set's row range."""
    dev.SetActWindow(32)
    w = synth.random_weights(t, nrows, k, seed=ntok)
    x = np.stack([synth.activations(k, seed=100 + i) * np.float32(1 + i % 7) for i in range(ntok)])
    want = oracle.matmul_q8act_f64(t, w, x, nrows, k, ntok, 32)
    wd, xd = devbuf(w), devbuf(x)
    planes = [devbuf(np.zeros(max(n, 4), np.uint32)) for n in quant.packed_words(t, nrows, k)]
    assert dev.pack_weights_dev(t, wd.ptr, nrows, k, *[p.ptr for p in planes])
    lo, part = 3, nrows - 5
    try:
        dev.set_tuning(gemm__few=3)
        for packed, r0, n in ((False, 0, nrows), (True, 0, nrows), (True, lo, part)):
            out = devbuf(np.full(ntok * n + 8, 3e30, np.float32))
            before = dev.launch_count()
            if packed:
                assert dev.matmul_packed_dev(out.ptr, t, Packed(*[p.ptr for p in planes], r0, nrows), xd.ptr, n, k, ntok)
            else:
                assert dev.matmul_dev(out.ptr, t, wd.ptr, xd.ptr, n, k, ntok)
            assert dev.launch_count() == before + 1
            dev.synchronize()
            got = out.get()
            assert np.all(got[ntok * n:] == np.float32(3e30)), "wrote past the output"
            assert nmse(got[:ntok * n].reshape(ntok, n), want[:, r0:r0 + n]) <= 1e-10, (packed, r0)
    finally:
        dev.set_tuning(gemm__few=0)


# A rounding of a sum whose mantissa is spread evenly over its logarithm: 2^-46 / 12 of [1, 2)'s mean square 1.5 / ln 2.
ROUNDING = 2.0 ** -46 / 12 / (1.5 / np.log(2))


@pytest.mark.parametrize("t", [quant.Q4_K, quant.Q6_K], ids=["q4_k", "q6_k"])
def test_few_tokens_round_once_a_super_block(dev, devbuf, t):
    """The k-quant window, 56 super-blocks over eight wavefronts: no more roundings than one scaling a super-block, a chain of
    seven and a tree of eight make, counted in a result's size -- d P (Q4_K: d P - dmin M, whose second product is 2.7 of it
    for weights spread as N(0, s)), four for the chain's sums that grow to an eighth, one a level.  Half as many again for what
    the count leaves out; scaled by halves and added one after the other it was 13 (Q6_K) and 19."""
    nrows, k, ntok = 256, 14336, 70
    units = 1 + 4 + 3 + (2.7 if t == quant.Q4_K else 0)
    w = synth.quantized_weights(t, nrows, k, seed=5)
    x = np.stack([synth.activations(k, seed=300 + i) for i in range(ntok)])
    wd, xd = devbuf(w), devbuf(x)
    dev.SetActWindow(256)
    try:
        want = oracle.matmul_q8act_f64(t, w, x, nrows, k, ntok, 256)
        dev.set_tuning(gemm__few=1, few__waves=8)
        out = devbuf(shape=(ntok, nrows), dtype=np.float32)
        assert dev.matmul_dev(out.ptr, t, wd.ptr, xd.ptr, nrows, k, ntok)
        dev.synchronize()
        assert nmse(out.get(), want) <= 1.5 * units * ROUNDING
    finally:
        dev.set_tuning(gemm__few=0, few__waves=0)
        dev.SetActWindow(32)


@pytest.mark.parametrize("t", [quant.Q4_K, quant.Q6_K], ids=["q4_k", "q6_k"])
def test_tokens_side_by_side_round_no_more_than_the_few_token_kernel(dev, devbuf, t):
    """The k-quant window, decode matvecs of eight tokens and of routed columns at K = 2048: roundings counted as above -- Q6_K two
    products a super-block and three levels of a tree of eight; Q4_K d P - dmin M and half of two products a slot and the five
    levels of 32 slots.  (Every run of Q6_K scaled for itself made 8.5, both products of Q4_K rounded 13.4.)"""
    nrows, k, ntok = 1500, 2048, 8
    units = 2 + 3 if t == quant.Q6_K else 2.7 + 1 + 1 + 5
    w = synth.quantized_weights(t, nrows, k, seed=6)
    x = np.stack([synth.activations(k, seed=300 + i) for i in range(ntok)])
    start = np.array([0, ntok], np.uint32)
    wd, xd, sd = devbuf(w), devbuf(x), devbuf(start)
    planes = [devbuf(np.zeros(max(n, 4), np.uint32)) for n in quant.packed_words(t, nrows, k)]
    assert dev.pack_weights_dev(t, wd.ptr, nrows, k, *[p.ptr for p in planes])
    dev.SetActWindow(256)
    try:
        want = oracle.matmul_q8act_f64(t, w, x, nrows, k, ntok, 256)
        dev.set_tuning(gemm__few=3, moe__form=10)
        for form in ("rows", "columns") + (("planes",) if t == quant.Q4_K else ()):
            out = devbuf(shape=(ntok, nrows), dtype=np.float32)
            before = dev.launch_count()
            if form == "rows":
                assert dev.matmul_dev(out.ptr, t, wd.ptr, xd.ptr, nrows, k, ntok)
            elif form == "planes":
                assert dev.matmul_packed_dev(out.ptr, t, Packed(*[p.ptr for p in planes], 0, nrows), xd.ptr, nrows, k, ntok)
            else:
                assert dev.moe_matvec_dev(out.ptr, None, t, wd.ptr, None, xd.ptr, None, None, sd.ptr, 1, ntok, nrows, k)
            assert dev.launch_count() == before + 1
            dev.synchronize()
            assert nmse(out.get(), want) <= 1.5 * units * ROUNDING, form
    finally:
        dev.set_tuning(gemm__few=0, moe__form=0)
        dev.SetActWindow(32)


@pytest.mark.parametrize("t,ntok", [(quant.Q6_K, 2), (quant.Q8_0, 3)], ids=["q6_k", "q8_0"])
def test_short_rows_over_planes_keep_their_kernels(dev, devbuf, t, ntok):
    """Under K = 1024, two tokens of Q6_K are the decode matvec's bits token by token and three of Q8_0 the few-token kernel's: side
    by side in one launch they round more."""
    nrows, k = 8192, 512
    w = synth.quantized_weights(t, nrows, k, seed=7)
    x = np.stack([synth.activations(k, seed=300 + i) for i in range(ntok)])
    wd, xd = devbuf(w), devbuf(x)
    planes = [devbuf(np.zeros(max(n, 4), np.uint32)) for n in quant.packed_words(t, nrows, k)]
    assert dev.pack_weights_dev(t, wd.ptr, nrows, k, *[p.ptr for p in planes])
    p = Packed(*[p.ptr for p in planes], 0, nrows)
    out, want = (devbuf(shape=(ntok, nrows), dtype=np.float32) for _ in range(2))
    assert dev.matmul_packed_dev(out.ptr, t, p, xd.ptr, nrows, k, ntok)
    try:
        if t == quant.Q6_K:
            for i in range(ntok):
                assert dev.matvec_packed_dev(want.ptr + i * nrows * 4, t, p, xd.ptr + i * k * 4, nrows, k)
        else:
            dev.set_tuning(gemm__few=1)
            assert dev.matmul_packed_dev(want.ptr, t, p, xd.ptr, nrows, k, ntok)
        dev.synchronize()
        assert np.array_equal(out.get().view(np.uint32), want.get().view(np.uint32))
    finally:
        dev.set_tuning(gemm__few=0)
