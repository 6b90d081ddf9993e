"""A dense block by handle for several rows (no norm in front): few rows, the edge of the few-token form, a prompt;
rows and planes, one type and two.  Bar: the oracle's matvecs chained, rel-L2 2e-3 of the block's contribution
(a 32-bit sum on a rounding boundary moves one value of the gated activation by one step in 127)."""
import numpy as np
import pytest

import oracle
from conftest import rel_l2
from jitllm_amd import _lib, quant, synth

pytestmark = pytest.mark.gpu


def _planes(t, w, nrows, k):
    qs, d, sc = oracle.pack_weights(t, w, nrows, k)
    return qs, d, (sc if sc is not None and sc.size else None)


@pytest.mark.parametrize("n", [2, 33, 64, 65])
@pytest.mark.parametrize("packed", [False, True], ids=["rows", "planes"])
@pytest.mark.parametrize("t,down_t", [(quant.Q4_K, quant.Q6_K), (quant.Q8_0, quant.Q8_0)], ids=["q4_k_q6_k", "q8_0"])
def test_dense_block_rows(dev, devbuf, t, down_t, packed, n):
    E, F = 512, 768
    window = quant.act_window([t, down_t])
    dev.SetActWindow(window)
    gate, up = (synth.quantized_weights(t, F, E, seed=s) for s in (1, 2))
    down = synth.quantized_weights(down_t, E, F, seed=3)
    h = np.stack([synth.activations(E, seed=20 + i) for i in range(n)])
    resid0 = np.stack([synth.activations(E, seed=90 + i) for i in range(n)])
    mats = [(t, gate, F, E), (t, up, F, E), (down_t, down, E, F)]
    ops = [_planes(*m) for m in mats] if packed else [gate, up, down]
    assert dev.PrepLayer(0, _lib.LAYER_DENSE, t, E, F, *ops, down_type=down_t)
    try:
        hd = devbuf(h)
        for _ in range(2):
            got = devbuf(resid0)
            assert dev.layer_ffn_dev(0, hd.ptr, got.ptr, n)
            dev.synchronize()
        g = oracle.matmul_q8act_f64(t, gate, h, F, E, n, window).astype(np.float32)
        u = oracle.matmul_q8act_f64(t, up, h, F, E, n, window).astype(np.float32)
        act = (g / (1 + np.exp(-g.astype(np.float64))) * u.astype(np.float64)).astype(np.float32)
        want = oracle.matmul_q8act_f64(down_t, down, act, E, F, n, window)
        assert rel_l2(got.get() - resid0, want) <= 2e-3
    finally:
        dev.ReleaseLayers(0, 1)
        dev.SetActWindow(32)


@pytest.mark.parametrize("n", [2, 65])
@pytest.mark.parametrize("packed", [False, True], ids=["rows", "planes"])
def test_dense_block_rows_off_their_alignment(dev, devbuf, packed, n):
    """Rows whose vectors of four floats do not begin on 16 bytes are declined; a residual that does not is served
    row by row, with the values of an aligned one; rows the decode kernels decline for their length are declined."""
    E, F, t = 256, 512, quant.Q8_0
    dev.SetActWindow(32)
    mats = [(t, synth.quantized_weights(t, r, k, seed=r + k), r, k) for r, k in ((F, E), (F, E), (E, F))]
    ops = [_planes(*m) for m in mats] if packed else [m[1] for m in mats]
    h = np.stack([synth.activations(E, seed=20 + i) for i in range(n)])
    r0 = np.stack([synth.activations(E, seed=90 + i) for i in range(n)])
    hd, hoff = devbuf(h), devbuf(np.concatenate([[0], h.ravel()]).astype(np.float32))
    roff = devbuf(np.concatenate([[0], r0.ravel(), [7]]).astype(np.float32))
    assert dev.PrepLayer(0, _lib.LAYER_DENSE, t, E, F, *ops)
    try:
        want = devbuf(r0)
        assert not dev.layer_ffn_dev(0, hoff.ptr + 4, want.ptr, n)
        for i in range(n):
            assert dev.layer_ffn_dev(0, hd.ptr + 4 * E * i, want.ptr + 4 * E * i, 1)
        assert dev.layer_ffn_dev(0, hd.ptr, roff.ptr + 4, n)
        dev.synchronize()
        got = roff.get()
        assert got[0] == 0 and got[-1] == 7
        assert np.array_equal(got[1:-1].view(np.uint32), want.get().ravel().view(np.uint32))
        if not packed:
            long = 131072
            assert dev.PrepLayer(0, _lib.LAYER_DENSE, t, E, long, *[np.zeros(E * long // 32 * 34, np.uint8)] * 3)
            assert not dev.layer_ffn_dev(0, hd.ptr, want.ptr, 1) and not dev.layer_ffn_dev(0, hd.ptr, want.ptr, n)
    finally:
        dev.ReleaseLayers(0, 1)
