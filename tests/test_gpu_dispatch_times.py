"""What a rule takes by itself is about as fast as the best of the forms it could have taken, where a rule once was not: device time of
calls queued behind a wait, the fastest of several windows of either in turn.  The limits are half of what the wrong pick cost, several
times what two measurements of one launch differ."""
import itertools

import numpy as np
import pytest

from jitllm_amd import quant, synth
from jitllm_amd.hipmem import Gate, timed_windows

pytestmark = pytest.mark.gpu


def us(dev, calls, steps=30):
    """calls: name -> (tuning, call).  us a call of each, the fastest of fifteen windows, in turn."""
    best = {n: 1e30 for n in calls}
    for _ in range(3):
        for n, (tuning, call) in calls.items():
            dev.set_tuning(**tuning)
            try:
                for _ in range(3):
                    assert call()
                dev.synchronize()
                _, per = timed_windows(lambda i: call(), steps, dev.stream, 5, Gate(dev))
                best[n] = min(best[n], min(per) * 1e3)
            finally:
                dev.set_tuning(**{k: 0 for k in tuning})
    return best


def random_bank(devbuf, t, sheets, nrows, k):
    """A bank of equal sheets (what the kernels read has no part in their time)."""
    return devbuf(np.tile(synth.random_weights(t, nrows, k, seed=3), sheets))


class Columns:
    """A grouped matmul of `counts` columns an expert over n banks."""

    def __init__(self, dev, devbuf, t, counts, nrows, k, nmat):
        self.dev, self.n, ncols = dev, len(counts), int(np.sum(counts))
        self.banks = [random_bank(devbuf, t, len(counts), nrows, k) for _ in range(nmat)]
        self.x, self.src = devbuf(np.stack([synth.activations(k, seed=i) for i in range(64)])), devbuf((np.arange(ncols) % 64).astype(np.uint32))
        self.start = devbuf(np.concatenate([[0], np.cumsum(counts)]).astype(np.uint32))
        self.out = [devbuf(shape=(ncols, nrows), dtype=np.float32) for _ in range(nmat)]
        second = (self.out[1].ptr, self.banks[1].ptr) if nmat == 2 else (None, None)
        self.args = (self.out[0].ptr, second[0], t, self.banks[0].ptr, second[1], self.x.ptr, None, self.src.ptr, self.start.ptr, len(counts), ncols, nrows, k)

    def __call__(self):
        return self.dev.moe_matvec_dev(*self.args)


def test_experts_without_columns(dev, devbuf):
    """Q4_K columns against decoded rows: eight of 128 experts with all of the columns against all with 32 each, 1.4 times; with every
    other workgroup bringing rows for nothing it was 1.9."""
    dev.SetActWindow(256)
    try:
        even, few = np.full(128, 32), np.zeros(128, int)
        few[5::16] = 512
        form = dict(moe__form=9)
        t = us(dev, {n: (form, Columns(dev, devbuf, quant.Q4_K, c, 2048, 768, 1)) for n, c in (("even", even), ("few", few))})
        assert t["few"] <= 1.65 * t["even"], t
    finally:
        dev.SetActWindow(32)


@pytest.mark.parametrize("t,window,n_expert,nrows,k,nmat,avg", [
    (quant.Q8_0, 32, 8, 512, 1024, 1, 44), (quant.Q4_K, 32, 4, 2048, 2048, 1, 44), (quant.Q6_K, 32, 2, 1024, 4096, 2, 44),
    (quant.Q6_K, 256, 8, 512, 1024, 1, 44), (quant.Q8_0, 32, 128, 768, 2048, 2, 36)], ids=lambda v: str(v))
def test_token_tiles_of_a_group(dev, devbuf, t, window, n_expert, nrows, k, nmat, avg):
    """Banks of few experts and a large one at more than 32 columns an expert: the token tiles a workgroup of the few-token kernel takes."""
    dev.SetActWindow(window)
    try:
        counts = np.full(n_expert, avg)
        counts[::2] += 7
        counts[1::2] -= 7
        call = Columns(dev, devbuf, t, counts, nrows, k, nmat)
        forms = {"auto": ({}, call)} | {nt: (dict(moe__form=5, few__nt=nt), call) for nt in (2, 3, 4)}
        got = us(dev, forms)
        assert got["auto"] <= 1.1 * min(got[nt] for nt in (2, 3, 4)), got
    finally:
        dev.SetActWindow(32)


@pytest.mark.parametrize("wdt,n_expert,k,ntok,rows", [("f16", 256, 7168, 16, 1), ("f32", 384, 7168, 2048, 8), ("f32", 128, 2048, 2048, 8)])
def test_order_of_the_router_s_grid(dev, devbuf, wdt, n_expert, k, ntok, rows):
    """Token groups or rows of the router side by side (tuning 16 / 32 + rows a workgroup): one where an L2 does not hold the router, a
    large router with few tokens, and a small one with many."""
    w = np.random.default_rng(1).standard_normal((n_expert, k)).astype(np.float16 if wdt == "f16" else np.float32)
    x = np.random.default_rng(2).standard_normal((ntok, k)).astype(np.float32)
    wd, xd, ld = [devbuf(w) for _ in range(3)], [devbuf(x) for _ in range(3)], devbuf(shape=(ntok, n_expert), dtype=np.float32)
    turn = itertools.count()   # (copies in turn, past what an L2 still holds)

    def call():
        i = next(turn) % 3
        return dev.moe_logits_dev(ld.ptr, 1 if wdt == "f16" else 0, wd[i].ptr, xd[i].ptr, n_expert, k, ntok)

    got = us(dev, {"auto": ({}, call), "tokens": (dict(moe__logits=16 + rows), call), "rows": (dict(moe__logits=32 + rows), call)})
    assert got["auto"] <= 1.08 * min(got["tokens"], got["rows"]), got


@pytest.mark.parametrize("nrows,k,ntok,gains", [(11009, 512, 1535, False), (14336, 1024, 2048, True)])
def test_tail_of_64_rows_by_itself(dev, devbuf, nrows, k, ntok, gains):
    """Q8_0: where the rows of a last round go to tiles of 64 rows, which gives the bits of the tiles of 128 rows and is faster, and where
    it must not take the call from another tile."""
    dev.SetActWindow(32)
    w, x = random_bank(devbuf, quant.Q8_0, 1, nrows, k), devbuf(np.random.default_rng(1).standard_normal((ntok, k)).astype(np.float32))
    o = devbuf(shape=(ntok, nrows), dtype=np.float32)

    def call():
        return dev.matmul_dev(o.ptr, quant.Q8_0, w.ptr, x.ptr, nrows, k, ntok)

    got = us(dev, {"auto": ({}, call), "flat": (dict(gemm__tall=1), call)}, 20)
    assert got["auto"] <= (0.98 if gains else 1.05) * got["flat"], got
    values = []
    for tall in (0, 1):
        dev.set_tuning(gemm__tall=tall)
        assert call()
        dev.synchronize()
        dev.set_tuning(gemm__tall=0)
        values.append(o.get())
    assert np.array_equal(values[0].view(np.uint32), values[1].view(np.uint32))


def mxfp4_planes(devbuf, nrows, k, ntok):
    from jitllm_amd.device import Packed
    rng = np.random.default_rng(1)
    nq, nd, _ = quant.packed_words(quant.MXFP4, nrows, k)
    qs = devbuf(rng.integers(0, 1 << 32, nq, dtype=np.uint32))
    d = devbuf(np.full(nd, 0x78787878, np.uint32))
    x = devbuf((rng.standard_normal((ntok, k)).astype(np.float32).view(np.uint32) >> 16).astype(np.uint16))
    return qs, d, x, devbuf(shape=(ntok, nrows), dtype=np.float32), Packed(qs.ptr, d.ptr, None, 0, nrows)


@pytest.mark.parametrize("nrows,k", [(201088, 2880), (8448, 8192), (1024, 5760)], ids=str)
def test_mxfp4_planes_two_tokens(dev, devbuf, nrows, k):
    """The plane matvec where its rounds are the shorter ones, else the one-launch form: a tall matrix, one whose matvec leaves half of
    the CUs idle, a small one of long rows."""
    qs, d, x, o, p = mxfp4_planes(devbuf, nrows, k, 2)

    def call():
        return dev.matmul_mxfp4_packed_bf16_dev(o.ptr, p, x.ptr, nrows, k, 2)

    got = us(dev, {"auto": ({}, call), "matvec": (dict(mxfp4__one=1), call), "one": (dict(mxfp4__one=11), call), "one of 32 rows": (dict(mxfp4__one=12), call)}, 20)
    assert got["auto"] <= 1.07 * min(got.values()), got


@pytest.mark.parametrize("packed,nrows,k,ntok", [(True, 2880, 2880, 64), (True, 5760, 5760, 16), (False, 2880, 2880, 16), (False, 2880, 2880, 128)])
def test_mxfp4_one_launch_by_itself(dev, devbuf, packed, nrows, k, ntok):
    """A few tokens take the form without a prep launch, whichever of its widths, unasked."""
    qs, d, x, o, p = mxfp4_planes(devbuf, nrows, k, ntok)
    w = None if packed else devbuf(synth.random_weights(quant.MXFP4, nrows, k, seed=1))
    n0 = dev.launch_count()
    assert dev.matmul_mxfp4_packed_bf16_dev(o.ptr, p, x.ptr, nrows, k, ntok) if packed else dev.matmul_mxfp4_bf16_dev(o.ptr, w.ptr, x.ptr, nrows, k, ntok)
    dev.synchronize()
    assert dev.launch_count() - n0 == 1


@pytest.mark.parametrize("kernel,waves", [("jl_few_q6k_planes_t4r1", 4), ("jl_few_q6k_planes_t4r2", 3)])
def test_wavefronts_a_simd_holds(dev, kernel, waves):
    """Kernels a register or seven past a step of the register file: it holds 512 a lane, and a workgroup of eight wavefronts takes two on
    each SIMD, so that one wavefront fewer can be half of a CU's workgroups."""
    import ctypes as C

    from jitllm_amd import _lib
    from jitllm_amd.hipmem import check, hip
    module, function, regs = C.c_void_p(), C.c_void_p(), C.c_int()
    check(hip().hipModuleLoad(C.byref(module), _lib.CODE_OBJECT_PATH.encode()), "hipModuleLoad")
    try:
        check(hip().hipModuleGetFunction(C.byref(function), module, kernel.encode()), kernel)
        check(hip().hipFuncGetAttribute(C.byref(regs), 4, function), kernel)   # HIP_FUNC_ATTRIBUTE_NUM_REGS
    finally:
        check(hip().hipModuleUnload(module), "hipModuleUnload")
    assert 512 // (-(-regs.value // 8) * 8) >= waves, regs.value
