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
        for p in ps:
            dev.ForgetPacked(p)
        dev.SetActWindow(32)


def _sizes():
    # (kind, rows, k, tokens): operands, results or neither above a mebibyte each, the first call of a context small
    return [("rows", 300, 512, 1), ("rows", 40, 4096, 65), ("rows", 4100, 512, 65), ("planes", 4100, 512, 70),
            ("planes", 300, 512, 3), ("rows", 1030, 1024, 256), ("rows", 300, 512, 1)]


def test_host_calls_small_growing_and_past_the_pinned_limit(dev, devbuf):
    """A context of its own, so that its pinned buffer is seen to grow from the first call on; calls whose operands,
    results or both pass 1 MiB are copied.  Poison behind every result."""
    t, window = quant.Q8_0, 32
    dev.SetActWindow(window)
    keep = []   # (weights are resident by their address)
    with Device(device=0, act_window=window) as d:
        for kind, rows, k, ntok in _sizes():
            w = synth.quantized_weights(t, rows, k, seed=rows + k)
            x = np.stack([synth.activations(k, seed=i) for i in range(ntok)])
            got = np.full(ntok * rows + 16, np.float32(5e30))
            xd, want = devbuf(x), devbuf(shape=(ntok, rows), dtype=np.float32, fill=0)
            if kind == "rows":
                keep.append(w)
                assert d.MatMul(got, t, w, x, rows, k, ntok)
                wd = devbuf(w)
                assert dev.matmul_dev(want.ptr, t, wd.ptr, xd.ptr, rows, k, ntok) if ntok > 1 else dev.matvec_dev(want.ptr, t, wd.ptr, xd.ptr, rows, k)
            else:
                p = _packed(t, w, rows, k)
                keep.append(p)
                assert d.MatMulPacked(got, t, p, x, rows, k, ntok)
                qd, dd = devbuf(p.qs), devbuf(p.d)
                assert dev.matmul_packed_dev(want.ptr, t, Packed(qd.ptr, dd.ptr, None, 0, rows), xd.ptr, rows, k, ntok)
            dev.synchronize()
            assert np.all(got[ntok * rows:] == np.float32(5e30)), (kind, rows, k, ntok)
            assert np.array_equal(_bits(got[:ntok * rows]), _bits(want.get()).ravel()), (kind, rows, k, ntok)


def test_two_contexts_in_two_threads(dev):
    """Host calls of two contexts, a thread each, at the same time: pinned, growing and copied ones, each result its
    own context's."""
    import threading
    t, window = quant.Q8_0, 32
    work = [[(rows + 8 * j, k, ntok, synth.quantized_weights(t, rows + 8 * j, k, seed=rows + j),
              np.stack([synth.activations(k, seed=100 * j + i) for i in range(ntok)])) for _, rows, k, ntok in _sizes()] for j in range(2)]

    def run(d, items, out):
        for rows, k, ntok, w, x in items:
            o = np.zeros(ntok * rows, np.float32)
            assert d.MatMul(o, t, w, x, rows, k, ntok)
            out.append(o)

    with Device(device=0, act_window=window) as a, Device(device=0, act_window=window) as b:
        want = [[], []]
        for d, items, out in zip((a, b), work, want):
            run(d, items, out)
        got = [[], []]
        threads = [threading.Thread(target=lambda d=d, items=items, out=out: [run(d, items, out) for _ in range(5)])
                   for d, items, out in zip((a, b), work, got)]
        for th in threads:
            th.start()
        for th in threads:
            th.join(60)
        assert not any(th.is_alive() for th in threads)
        for w, g in zip(want, got):
            assert len(g) == 5 * len(w)
            for i, o in enumerate(g):
                assert np.array_equal(_bits(o), _bits(w[i % len(w)])), i
