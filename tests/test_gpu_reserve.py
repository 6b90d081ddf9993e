"""jl_reserve: calls within what it was asked for allocate nothing, whatever their type and rows, and their values are
those of a context that grows its workspaces as it goes (up to the order of the f32 sums)."""
import numpy as np
import pytest

from conftest import nmse
from jitllm_amd import quant, synth
from jitllm_amd.device import Device
from jitllm_amd.hipmem import mem_info

pytestmark = pytest.mark.gpu

# (MXFP4 512 x 2880 x 2880: its fastest form turns the rows into planes; most others are cut along K)
SHAPES = [(quant.MXFP4, 32, 300, 5760, 2880), (quant.MXFP4, 32, 512, 2880, 2880), (quant.MXFP4, 32, 200, 640, 3072),
          (quant.MXFP4, 32, 40, 2880, 2880), (quant.Q8_0, 32, 300, 512, 3072), (quant.Q8_0, 32, 500, 4096, 2944),
          (quant.Q8_0, 32, 2, 512, 2048), (quant.Q4_K, 32, 130, 512, 3072), (quant.Q6_K, 32, 130, 512, 3072),
          (quant.Q6_K, 256, 130, 512, 3072), (quant.Q4_K, 256, 512, 4096, 2048), (quant.Q4_K, 256, 100, 512, 3072),
          (quant.Q4_K, 256, 20, 512, 3072)]


def _operands(devbuf, t, ntok, nrows, k):
    w = synth.random_weights(t, nrows, k, seed=nrows + ntok)
    x = np.stack([synth.activations(k, seed=i) for i in range(ntok)])
    if t == quant.MXFP4:
        x = (np.ascontiguousarray(x).view(np.uint32) >> 16).astype(np.uint16)
    return devbuf(w), devbuf(x), [devbuf(np.full(ntok * nrows + 8, 3e30, np.float32)) for _ in range(2)]


def _run(d, o, t, window, wd, xd, nrows, k, ntok):
    d.SetActWindow(window)
    if t == quant.MXFP4:
        assert d.matmul_mxfp4_bf16_dev(o.ptr, wd.ptr, xd.ptr, nrows, k, ntok)
    else:
        assert d.matmul_dev(o.ptr, t, wd.ptr, xd.ptr, nrows, k, ntok)
    d.synchronize()
    got = o.get()
    assert np.all(got[ntok * nrows:] == np.float32(3e30))
    return got[:ntok * nrows]


def test_reserved_calls_allocate_nothing(dev, devbuf):
    with Device(device=0, act_window=32) as grows, Device(device=0, act_window=32) as held:
        # (a kernel with spilled registers takes memory of the runtime's on a stream's first launch of it)
        wd, xd, (a, b) = _operands(devbuf, quant.MXFP4, 70, 200, 256)
        for form in (3, 4):
            held.set_tuning(mxfp4__planes=form)
            _run(held, a, quant.MXFP4, 32, wd, xd, 200, 256, 70)
        held.set_tuning(mxfp4__planes=0)
        held.Reserve(512, 3072)
        for t, window, ntok, nrows, k in SHAPES:
            wd, xd, (a, b) = _operands(devbuf, t, ntok, nrows, k)
            want = _run(grows, a, t, window, wd, xd, nrows, k, ntok)
            free, _ = mem_info()
            got = _run(held, b, t, window, wd, xd, nrows, k, ntok)
            assert mem_info()[0] == free, (quant.NAMES[t], window, ntok, nrows, k)
            assert nmse(got, want) <= 1e-11, (quant.NAMES[t], window, ntok, nrows, k)
            for buf in (wd, xd, a, b):
                buf.free()
        # the room one shape's fastest form takes: the launches of a context that grows, and still nothing allocated
        t, window, ntok, nrows, k = SHAPES[1]
        wd, xd, (a, b) = _operands(devbuf, t, ntok, nrows, k)
        want = _run(grows, a, t, window, wd, xd, nrows, k, ntok)
        assert held.reserve_shape(t, nrows, k, ntok)
        free, _ = mem_info()
        got = _run(held, b, t, window, wd, xd, nrows, k, ntok)
        assert mem_info()[0] == free
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
