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
