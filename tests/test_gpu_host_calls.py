"""Calls over host memory: the order in which results are handed over, operands and results too large for pinned
memory, the pinned buffer's growth, contexts in threads of their own.  Results are compared bit for bit with the
device-pointer forms, which other tests hold to the oracle."""
import numpy as np
import pytest

import oracle
from jitllm_amd import quant, synth
from jitllm_amd.device import Device, MVGroup, Packed

pytestmark = pytest.mark.gpu


def _bits(a):
    return np.ascontiguousarray(a).view(np.uint32)


def _packed(t, w, rows, k):
    qs, d, sc = oracle.pack_weights(t, w, rows, k)
    return Packed(qs, d, sc if sc is not None and sc.size else None, 0, rows)


def test_group_results_the_residual_last(dev):
    """A residual that is also the first matrix's output keeps the sum, and so does one that is another's."""
    k, rows, t = 1024, 256, quant.Q4_K
    dev.SetActWindow(256)
    ps = [_packed(t, synth.quantized_weights(t, rows, k, seed=s), rows, k) for s in (1, 2)]
    x, r0 = synth.activations(k, seed=3), synth.activations(rows, seed=4)
    call = lambda outs, resid: dev.MatVecPackedGroup(MVGroup(outs, [t, t], ps, [rows, rows], x, k, Resid=resid, Alpha=0.5))
    try:
        outs, want = [np.zeros(rows, np.float32) for _ in range(2)], r0.copy()
        assert call(outs, want) and not np.array_equal(want, outs[0])
        for i in range(2):
            shared, other = r0.copy(), np.zeros(rows, np.float32)
            assert call([shared, other] if i == 0 else [other, shared], shared)
            assert np.array_equal(_bits(shared), _bits(want)), i
            assert np.array_equal(_bits(other), _bits(outs[1 - i])), i
    finally:
        dev.SetActWindow(32)
